// The RCCD / RCCSD residual of a small system: the same terms as cc.hip and ccsd.hip, in three to five
// launches instead of 30 to 90.
//
// At ov of a few hundred and below every product is a few microseconds of latency whatever its size, so
// the number of launches sets the iteration's time (RCCSD of water, o=5 v=2: 90 launches, 260 us of kernels of
// 2 to 4 us each for 2e4 flop; 8 launches and 48 us in this form.  o=5 v=19: RCCD 121 -> 53 us, RCCSD
// 344 -> 72 us).  Here the residual is a list of outputs, each the sum of contractions over
// tensors read where they lie (no amplitude layouts, no permuted copies), and outputs that do not
// depend on each other share a launch:
//   RCCD    pack T+-, [Fae, Fmi, W', WJ, WE, pp-ladders], [Y, X, sums], [H]
//   RCCSD   tau arrays and pack, [Fae, Fmi, Fme, W', Z, WJ, WE, ...], [Fb, Fj, Y, X], [H, R1]
// The descriptors are built once per stage from the buffers that the stage's work set owns.
#include "cc.h"

#include <algorithm>
#include <cstring>
#include <string>

namespace jues {

// C[m0,m1;n0,n1] = sum of terms + sum of points + beta (sum of nd blocks of D, each dstep after the other), over
// output dims d[4] with strides c[4] (D: e[4]).  Of the terms' concatenated 16-deep k-slabs it takes s0 .. s1: a long
// contraction of few tiles is cut into partial outputs, which the output that reads them as D adds up.
template <typename T>
struct SmallOut {
  T* C;
  double* C64;  // if set, the result goes here in FP64 instead
  const T* D;
  T beta;
  int d[4], c[4], e[4];
  int tiles_m, tiles_n, tile0;  // 16 x 16 tiles; the first one's place in the launch
  int t0, t1, p0, p1;           // its terms and points
  int s0, s1, nd, dstep;
};
// alpha sum_k A[m,k] B[k,n]: A indexed by (m0,m1) and up to three contraction digits, B by (n0,n1) and those
template <typename T>
struct SmallTerm {
  const T *A, *B;
  T alpha;
  int K, k0, k1;  // contraction length and its first two digits' dimensions
  int a[2], b[2], ka[3], kb[3];
};
// alpha sum_k A[x,k] B[x,k] with either operand indexed by any of the four output indices: the terms whose
// operands do not separate into rows and columns of the output, all of them a contraction over one occupied or
// virtual index
template <typename T>
struct SmallPoint {
  const T *A, *B;
  T alpha;
  int K, ka, kb;
  int a[4], b[4];
};

namespace {

typedef double dvec4 __attribute__((ext_vector_type(4)));
typedef float fvec4 __attribute__((ext_vector_type(4)));
template <typename T> struct Mma;
template <> struct Mma<double> {
  typedef dvec4 acc;
  __device__ static inline int row(int lane, int r) { return (lane >> 4) + 4 * r; }
  __device__ static inline acc op(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
};
template <> struct Mma<float> {
  typedef fvec4 acc;
  __device__ static inline int row(int lane, int r) { return 4 * (lane >> 4) + r; }
  __device__ static inline acc op(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

constexpr int SW = 8;  // wavefronts per workgroup

// One workgroup per 16 x 16 tile of an output.  Its eight wavefronts share the contraction: the 16-deep k-slabs of
// all terms are dealt to them in turn, each wavefront reading its fragments from memory through the terms'
// strides (lane l: row or column l % 16, k = 4 (l / 16) + u at MFMA step u), and the partial tiles are added in a
// fixed order through LDS.  beta D and the points are added by the thread that stores an element.
// Bound by memory latency: a wavefront has two slabs' loads in flight and at most a few slabs to do (long
// contractions are cut), so a launch takes 5 to 10 us up to ov = 200.  32 x 32 tiles measured slower below ov = 400.
template <typename T>
__global__ __launch_bounds__(64 * SW) void small_contract_kernel(const SmallOut<T>* __restrict__ outs, int nouts,
                                                                 const SmallTerm<T>* __restrict__ terms,
                                                                 const SmallPoint<T>* __restrict__ points) {
  __shared__ T red[SW][256];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int x = 0;
  while (x + 1 < nouts && (int)blockIdx.x >= outs[x + 1].tile0) ++x;
  const SmallOut<T>& O = outs[x];
  const int tile = (int)blockIdx.x - O.tile0, tm = tile % O.tiles_m, tn = tile / O.tiles_m;
  const int M = O.d[0] * O.d[1], N = O.d[2] * O.d[3];
  const int fr = lane & 15, fk = lane >> 4;
  const int m = min(16 * tm + fr, M - 1), n = min(16 * tn + fr, N - 1);
  const int m0 = m % O.d[0], m1 = m / O.d[0], n0 = n % O.d[2], n1 = n / O.d[2];
  typename Mma<T>::acc acc{0, 0, 0, 0};
  int turn = wave, base = 0;  // slabs until this wavefront's next one; the terms' slabs so far
  for (int q = O.t0; q < O.t1; ++q) {
    const SmallTerm<T>& t = terms[q];
    const int slabs = (t.K + 15) / 16, lo = max(0, O.s0 - base), hi = min(slabs, O.s1 - base);
    base += slabs;
    if (hi <= lo) continue;
    const T* A = t.A + m0 * t.a[0] + m1 * t.a[1];
    const T* B = t.B + n0 * t.b[0] + n1 * t.b[1];
    auto load = [&](int s, T (&ra)[4], T (&rb)[4]) {
      const int k = 16 * s + 4 * fk;
      unsigned d0 = (unsigned)k % (unsigned)t.k0, r = (unsigned)k / (unsigned)t.k0;
      unsigned d1 = r % (unsigned)t.k1, d2 = r / (unsigned)t.k1;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool in = k + u < t.K;
        const int oa = in ? (int)(d0 * t.ka[0] + d1 * t.ka[1] + d2 * t.ka[2]) : 0;
        const int ob = in ? (int)(d0 * t.kb[0] + d1 * t.kb[1] + d2 * t.kb[2]) : 0;
        const T va = A[oa], vb = B[ob];
        ra[u] = in ? t.alpha * va : T(0);
        rb[u] = in ? vb : T(0);
        if (++d0 == (unsigned)t.k0) {
          d0 = 0;
          if (++d1 == (unsigned)t.k1) { d1 = 0; ++d2; }
        }
      }
    };
    auto mma = [&](const T (&ra)[4], const T (&rb)[4]) {
#pragma unroll
      for (int u = 0; u < 4; ++u) acc = Mma<T>::op(rb[u], ra[u], acc);
    };
    int s = lo + turn;
    for (; s + SW < hi; s += 2 * SW) {
      T ra[2][4], rb[2][4];
      load(s, ra[0], rb[0]);
      load(s + SW, ra[1], rb[1]);
      mma(ra[0], rb[0]);
      mma(ra[1], rb[1]);
    }
    for (; s < hi; s += SW) {
      T ra[4], rb[4];
      load(s, ra, rb);
      mma(ra, rb);
    }
    turn = s - hi;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][16 * Mma<T>::row(lane, r) + fr] = acc[r];
  __syncthreads();
  const int em = 16 * tm + tid % 16, en = 16 * tn + tid / 16;
  if (tid >= 256 || em >= M || en >= N) return;
  const int i[4] = {em % O.d[0], em / O.d[0], en % O.d[2], en / O.d[2]};
  double val = (double)red[0][tid];  // (the sums of partial results are in FP64 and rounded once)
#pragma unroll
  for (int w = 1; w < SW; ++w) val += (double)red[w][tid];
  for (int q = O.p0; q < O.p1; ++q) {
    const SmallPoint<T>& p = points[q];
    const T* A = p.A + i[0] * p.a[0] + i[1] * p.a[1] + i[2] * p.a[2] + i[3] * p.a[3];
    const T* B = p.B + i[0] * p.b[0] + i[1] * p.b[1] + i[2] * p.b[2] + i[3] * p.b[3];
    T s = 0;
#pragma unroll 8
    for (int k = 0; k < p.K; ++k) s += A[k * p.ka] * B[k * p.kb];
    val += (double)(p.alpha * s);
  }
  if (O.D) {
    const T* D = O.D + i[0] * O.e[0] + i[1] * O.e[1] + i[2] * O.e[2] + i[3] * O.e[3];
    double s = 0;
    for (int q = 0; q < O.nd; ++q) s += (double)D[(long)q * O.dstep];
    val += (double)O.beta * s;
  }
  const int at = i[0] * O.c[0] + i[1] * O.c[1] + i[2] * O.c[2] + i[3] * O.c[3];
  if (O.C64) O.C64[at] = val;
  else O.C[at] = (T)val;
}

// What the contractions read of the amplitudes, in the compute type: t2 and t1 themselves (FP32 only), with t1 also
// tau = t2 + t1 t1, tau' = t2 + t1 t1 / 2 and xi = t2 + 2 t1 t1, and the packed pairs of tau (of t2 without
// t1) for the pp-ladder.  Null outputs are skipped.
template <typename T>
struct SmallPrep {
  const double *t2, *t1;
  int o, v;
  T *t2c, *t1c, *tau, *taup, *xi, *Tp, *Tm;
  PairTables P;
};
template <typename T>
__global__ __launch_bounds__(256) void small_prep_kernel(SmallPrep<T> S) {
  const int o = S.o, v = S.v;
  const long oo = (long)o * o, n2 = oo * v * v, n1 = (long)o * v;
  const long np = S.Tp ? S.P.npo * S.P.npv : 0, nm = S.Tm ? S.P.nmo * S.P.nmv : 0;
  const long total = n2 + np + nm + (S.t1c ? n1 : 0);
  for (long x = blockIdx.x * 256L + threadIdx.x; x < total; x += (long)gridDim.x * 256L) {
    if (x < n2) {
      const double t = S.t2[x];
      if (S.t2c) S.t2c[x] = (T)t;
      if (S.tau) {
        const int ij = (int)(x % oo), ab = (int)(x / oo);
        const double tt = S.t1[ij % o + (long)o * (ab % v)] * S.t1[ij / o + (long)o * (ab / v)];
        S.tau[x] = (T)(t + tt);
        S.taup[x] = (T)(t + 0.5 * tt);
        S.xi[x] = (T)(t + 2.0 * tt);
      }
    } else if (x < n2 + np + nm) {
      const bool plus = x < n2 + np;
      const long y = x - n2 - (plus ? 0 : np), nr = plus ? S.P.npo : S.P.nmo;
      const int2 ij = plus ? S.P.o_le[y % nr] : S.P.o_lt[y % nr], ef = plus ? S.P.v_le[y / nr] : S.P.v_lt[y / nr];
      const long base = ij.x + (long)o * ij.y;
      double a = S.t2[base + oo * (ef.x + (long)v * ef.y)], b = S.t2[base + oo * (ef.y + (long)v * ef.x)];
      if (S.t1) {
        a += S.t1[ij.x + (long)o * ef.x] * S.t1[ij.y + (long)o * ef.y];
        b += S.t1[ij.x + (long)o * ef.y] * S.t1[ij.y + (long)o * ef.x];
      }
      if (plus) S.Tp[y] = (T)(ef.x == ef.y ? a : a + b);
      else S.Tm[y] = (T)(a - b);
    } else {
      const long y = x - n2 - np - nm;
      S.t1c[y] = (T)S.t1[y];
    }
  }
}

// A tensor and its index letters, first fastest: i..n occupied, a..f virtual, P (p) rows (columns) of an
// explicit dimension
struct Ten {
  const void* p;
  const char* idx;
};

template <typename T>
class Builder {
 public:
  Builder(int o, int v) : o_(o), v_(v) {}
  // explicit dimensions of the letters w, x, y, z (packed pairs)
  void dim(char c, long d) { extra_[c - 'w'] = d; }
  // a new output C[idx] whose tile rows are the letters m and columns the letters n (at most two each)
  void out(const void* C, const char* idx, const char* m, const char* n, const void* D = nullptr,
           const char* didx = nullptr, double beta = 0.0, double* C64 = nullptr, int nd = 1, long dstep = 0) {
    SmallOut<T> x{};
    x.C = static_cast<T*>(const_cast<void*>(C));
    x.C64 = C64;
    x.D = static_cast<const T*>(D);
    x.beta = (T)beta;
    x.nd = nd;
    x.dstep = (int)dstep;
    x.s0 = 0;
    x.s1 = 1 << 30;
    std::memset(l_, 0, sizeof(l_));
    for (int q = 0; q < 2; ++q) {
      if ((int)std::strlen(m) > q) l_[q] = m[q];
      if ((int)std::strlen(n) > q) l_[2 + q] = n[q];
    }
    for (int q = 0; q < 4; ++q) {
      x.d[q] = l_[q] ? (int)size(l_[q]) : 1;
      x.c[q] = l_[q] ? stride(idx, l_[q]) : 0;
      x.e[q] = D && l_[q] ? stride(didx, l_[q]) : 0;
    }
    x.tiles_m = (x.d[0] * x.d[1] + 15) / 16;
    x.tiles_n = (x.d[2] * x.d[3] + 15) / 16;
    x.t0 = x.t1 = (int)terms.size();
    x.p0 = x.p1 = (int)points.size();
    outs.push_back(x);
  }
  // the current output += alpha A B; the letters that the output has not are summed over
  void add(double alpha, Ten A, Ten B) {
    auto has = [](const char* s, char c) { return c && std::strchr(s, c) != nullptr; };
    auto of_rows = [&](const char* s) {  // no column letter of the output
      return !has(s, l_[2]) && !has(s, l_[3]);
    };
    auto of_cols = [&](const char* s) { return !has(s, l_[0]) && !has(s, l_[1]); };
    std::string k;
    for (const char* c = A.idx; *c; ++c)
      if (std::memchr(l_, *c, 4) == nullptr) {
        JUES_REQUIRE(has(B.idx, *c), "small contraction: unsupported index");
        k += *c;
      }
    if (!(of_rows(A.idx) && of_cols(B.idx)) && of_rows(B.idx) && of_cols(A.idx)) std::swap(A, B);
    if (of_rows(A.idx) && of_cols(B.idx)) {
      JUES_REQUIRE(k.size() <= 3 && !k.empty(), "small contraction: too many summed indices");
      std::sort(k.begin(), k.end(), [&](char p, char q) { return stride(A.idx, p) < stride(A.idx, q); });
      SmallTerm<T> t{};
      t.A = static_cast<const T*>(A.p);
      t.B = static_cast<const T*>(B.p);
      t.alpha = (T)alpha;
      t.K = 1;
      t.k0 = t.k1 = 1;
      for (size_t q = 0; q < k.size(); ++q) {
        t.K *= (int)size(k[q]);
        t.ka[q] = stride(A.idx, k[q]);
        t.kb[q] = stride(B.idx, k[q]);
      }
      t.k0 = (int)size(k[0]);
      if (k.size() > 1) t.k1 = (int)size(k[1]);
      for (int q = 0; q < 2; ++q) {
        t.a[q] = l_[q] ? stride(A.idx, l_[q]) : 0;
        t.b[q] = l_[2 + q] ? stride(B.idx, l_[2 + q]) : 0;
      }
      terms.push_back(t);
      outs.back().t1 = (int)terms.size();
      return;
    }
    JUES_REQUIRE(k.size() == 1, "small contraction: operands do not separate");
    SmallPoint<T> p{};
    p.A = static_cast<const T*>(A.p);
    p.B = static_cast<const T*>(B.p);
    p.alpha = (T)alpha;
    p.K = (int)size(k[0]);
    p.ka = stride(A.idx, k[0]);
    p.kb = stride(B.idx, k[0]);
    for (int q = 0; q < 4; ++q) {
      p.a[q] = l_[q] ? stride(A.idx, l_[q]) : 0;
      p.b[q] = l_[q] ? stride(B.idx, l_[q]) : 0;
    }
    points.push_back(p);
    outs.back().p1 = (int)points.size();
  }
  // The current output, of a long contraction and few tiles, in partial outputs of at most four slabs per
  // wavefront; returns how many, each `step` elements after the other from its C (at most `most`)
  int cut(long step, int most) {
    SmallOut<T> x = outs.back();
    int slabs = 0;
    for (int q = x.t0; q < x.t1; ++q) slabs += (terms[q].K + 15) / 16;
    const int parts = std::max(1, std::min(most, (slabs + 4 * SW - 1) / (4 * SW)));
    const int each = (slabs + parts - 1) / parts;
    outs.pop_back();
    for (int q = 0; q < parts; ++q) {
      SmallOut<T> y = x;
      y.C = x.C + q * step;
      y.s0 = q * each;
      y.s1 = (q + 1) * each;
      if (q > 0) {
        y.D = nullptr;
        y.p0 = y.p1;
      }
      outs.push_back(y);
    }
    return parts;
  }
  // the outputs since the last call make one launch
  void launch() {
    int tiles = 0;
    for (size_t q = first_; q < outs.size(); ++q) {
      outs[q].tile0 = tiles;
      tiles += outs[q].tiles_m * outs[q].tiles_n;
    }
    groups.push_back({first_, (int)outs.size() - first_, tiles});
    first_ = (int)outs.size();
  }
  std::vector<SmallOut<T>> outs;
  std::vector<SmallTerm<T>> terms;
  std::vector<SmallPoint<T>> points;
  std::vector<SmallGroup> groups;

 private:
  long size(char c) const {
    if (c >= 'w') return extra_[c - 'w'];
    return c >= 'i' && c <= 'n' ? o_ : v_;
  }
  // elements between neighbours in the letter c (0 without it); the kernel's offsets have 32 bits
  int stride(const char* idx, char c) const {
    long s = 1, at = 0;
    for (; *idx; ++idx) {
      if (*idx == c) at = s;
      s *= size(*idx);
    }
    JUES_REQUIRE(s < (1L << 31), "small contraction: tensor too large");
    return (int)at;
  }
  int o_, v_, first_ = 0;
  long extra_[4] = {1, 1, 1, 1};
  char l_[4];
};

}  // namespace

// The outputs of the residual.  Names and terms are those of rccd_contractions (cc.hip) and
// rccsd_contractions (ccsd.hip), except that the Fock-like terms enter H directly
// (H += t.Fb^T - Fj^T.t, whose transposes S = H + H^T supplies) and the hole-hole ladder is
// unpacked: X = W' tau / 2, of which the update kernel adds X[ijab] + X[jiba].
template <typename T>
void SmallPlan<T>::build(jues_ctx* ctx, CCState& S) {
  const int o = S.o, v = S.v;
  const long ov = (long)o * v, N2 = ov * ov, oo = (long)o * o, vv = (long)v * v;
  CCInts<T>& I = ints<T>(S);
  CCWork<T>& W = work<T>(S);
  const PairTables& P = S.P;
  const bool cc2 = S.method == 1, mrccsd = S.opts.ccsd_eqs == JUES_CCSD_MRCCSD;
  const bool stored = !S.ladder_recompute;
  const void *t2 = S.t.p, *t1 = S.t.as<double>() + N2;
  if (sizeof(T) == 4) {
    t2 = bufp_t<T>(W.Tov, N2);
    t1 = bufp_t<T>(W.t1, ov);
  }
  const void* tau = cc2 ? bufp_t<T>(W.Tpp, N2) : t2;    // t2 + t1 t1
  const void* taup = cc2 ? bufp_t<T>(W.Upp, N2) : t2;   // t2 + t1 t1 / 2
  const void* xi = cc2 ? bufp_t<T>(W.Ttov, N2) : t2;    // t2 + 2 t1 t1
  T *WJ = bufp_t<T>(W.WJ, N2), *WE = bufp_t<T>(W.WE, N2), *H = bufp_t<T>(W.H, N2), *Y = bufp_t<T>(W.Y, N2),
    *X = bufp_t<T>(W.X2, N2), *Wp = bufp_t<T>(W.Wp, oo * oo);
  // Fae, Fmi and the T1 residual: partial outputs, summed in the second and third launch
  constexpr int PARTS = 16;
  T *Fae = bufp_t<T>(W.Fae, (PARTS + 1) * vv), *Fmi = bufp_t<T>(W.Fmi, (PARTS + 1) * oo);
  bufp_t<T>(W.Tp, P.npo * P.npv);
  bufp_t<T>(W.Tm, std::max(1L, P.nmo * P.nmv));
  bufp_t<T>(W.Lp, P.npo * P.npv);
  bufp_t<T>(W.Lm, std::max(1L, P.nmo * P.nmv));
  T *Fme = nullptr, *n1 = nullptr, *Z = nullptr, *Qa = nullptr, *Qb = nullptr;
  if (cc2) {
    Fme = bufp_t<T>(W.Fme, ov);
    n1 = bufp_t<T>(W.n1, (PARTS + 2) * ov);
    Z = bufp_t<T>(W.Z, oo * ov);
    Qa = bufp_t<T>(W.Q, 2 * oo * ov);
    Qb = Qa + oo * ov;
  }
  Builder<T> b(o, v);
  auto t = [&](const char* idx) { return Ten{t2, idx}; };
  auto tp = [&](const char* idx) { return Ten{taup, idx}; };
  auto x = [&](const char* idx) { return Ten{xi, idx}; };
  auto s1 = [&](const char* idx) { return Ten{t1, idx}; };
  auto K = [&](const char* idx) { return Ten{I.Kov.p, idx}; };
  auto J = [&](const char* idx) { return Ten{I.Jov.p, idx}; };
  auto G3 = [&](const char* idx) { return Ten{I.ooov_c.p, idx}; };   // (ij|ka)
  auto G1 = [&](const char* idx) { return Ten{I.ovvv_c.p, idx}; };   // (ia|bc)
  auto pp_ladder = [&](const DevBuf& L, const DevBuf& Tx, const DevBuf& V, long no, long nv) {
    b.dim('w', no);
    b.dim('x', nv);
    b.dim('y', nv);
    b.out(L.p, "wx", "w", "x");
    b.add(1.0, {Tx.p, "wy"}, {V.p, "yx"});
  };

  // ---- from the amplitudes alone
  b.out(Fae, "ae", "a", "e");
  b.add(-2.0, tp("mnaf"), K("menf"));
  b.add(1.0, tp("nmaf"), K("menf"));
  int nfae = b.cut(vv, PARTS);
  b.out(Fmi, "mi", "m", "i");
  b.add(2.0, K("menf"), tp("inef"));
  b.add(-1.0, K("menf"), tp("nief"));
  int nfmi = b.cut(oo, PARTS), nn1 = 0;
  if (cc2) {
    // their terms linear in t1, as vectors over the pair
    b.out(Fae + vv * nfae++, "ae", "ae", "");
    b.add(2.0, G1("mfae"), s1("mf"));
    b.add(-1.0, G1(mrccsd ? "maef" : "meaf"), s1("mf"));
    b.out(Fmi + oo * nfmi++, "mi", "mi", "");
    b.add(2.0, G3("mine"), s1("ne"));
    b.add(-1.0, G3("nime"), s1("ne"));
    b.out(n1, "ia", "i", "a");
    b.add(-2.0, G3("mine"), t("nmea"));
    b.add(1.0, G3("nime"), t("nmea"));
    b.add(2.0, t("imef"), G1("mfae"));
    b.add(-1.0, t("imef"), G1("meaf"));
    nn1 = b.cut(ov, PARTS);
    b.out(n1 + ov * nn1++, "ia", "ia", "");
    b.add(2.0, K("iame"), s1("me"));
    b.add(-1.0, J("maie"), s1("me"));
  }
  b.out(Wp, "mnij", "mn", "ij", I.oooo.p, "mnij", 1.0);
  b.add(1.0, K("menf"), {tau, "ijef"});
  if (cc2) {
    b.add(1.0, s1("je"), G3("mine"));
    b.add(1.0, s1("ie"), G3("njme"));
  }
  // K (U - 2 tt^x)/2 - Kx T/2 with U - 2 tt^x = 2 t2[kjcb] - xi[kjbc]
  b.out(WJ, "mejb", "me", "jb", I.Kov.p, "mejb", 1.0);
  b.add(1.0, K("mekc"), t("kjcb"));
  b.add(-0.5, K("mekc"), x("kjbc"));
  b.add(-0.5, K("mcke"), t("kjcb"));
  if (cc2) {
    b.add(1.0, s1("jf"), G1("mebf"));
    b.add(-1.0, s1("nb"), G3("njme"));
  }
  b.out(WE, "mejb", "me", "jb", I.Jov.p, "mejb", -1.0);
  b.add(0.5, K("mcke"), x("kjbc"));
  if (cc2) {
    b.add(-1.0, s1("jf"), G1("mfbe"));
    b.add(1.0, s1("nb"), G3("mjne"));
  }
  if (stored) {
    pp_ladder(W.Lp, W.Tp, I.Vp, P.npo, P.npv);
    if (P.nmo > 0 && P.nmv > 0) pp_ladder(W.Lm, W.Tm, I.Vm, P.nmo, P.nmv);
  }
  if (cc2) {
    b.out(Fme, "me", "me", "");
    b.add(2.0, K("menf"), s1("nf"));
    b.add(-1.0, K("mfne"), s1("nf"));
    b.out(Z, "ijma", "ij", "ma");
    b.add(1.0, {tau, "ijef"}, G1("mfae"));
    b.out(Qa, "imjb", "im", "jb");
    b.add(1.0, s1("ie"), K("jbme"));
    b.out(Qb, "imaj", "im", "aj");
    b.add(1.0, s1("ie"), J("maje"));
  }
  b.launch();

  // ---- from the intermediates
  T *Fa = bufp_t<T>(W.FmiT, 2 * (oo + vv)), *Fi = Fa + vv, *Fb = Fa, *Fj = Fi;
  b.out(Fa, "be", "b", "e", Fae, "be", 1.0, nullptr, nfae, vv);
  b.out(Fi, "mj", "m", "j", Fmi, "mj", 1.0, nullptr, nfmi, oo);
  if (cc2) {
    Fb = Fi + oo;
    Fj = Fb + vv;
    b.out(Fb, "be", "b", "e", Fae, "be", 1.0, nullptr, nfae, vv);
    b.add(-0.5, s1("mb"), {Fme, "me"});
    b.out(Fj, "mj", "m", "j", Fmi, "mj", 1.0, nullptr, nfmi, oo);
    b.add(0.5, {Fme, "me"}, s1("je"));
    b.out(n1 + ov * nn1++, "ia", "ia", "");
    b.add(2.0, t("imae"), {Fme, "me"});
    b.add(-1.0, t("miae"), {Fme, "me"});
  }
  b.out(X, "ijab", "ij", "ab");
  b.add(0.5, {Wp, "mnij"}, {tau, "mnab"});
  if (cc2) b.add(-1.0, s1("mb"), {Z, "ijma"});
  b.out(Y, "iajb", "ia", "jb");
  b.add(1.0, t("ikca"), {WE, "kcjb"});
  b.launch();
  b.out(H, "iajb", "ia", "jb");
  b.add(1.0, t("ikac"), {WE, "kcjb"});
  b.add(2.0, t("ikac"), {WJ, "kcjb"});
  b.add(-1.0, t("kiac"), {WJ, "kcjb"});
  b.add(1.0, t("ijac"), {Fb, "bc"});
  b.add(-1.0, t("ikab"), {Fj, "kj"});
  if (cc2) {
    b.add(-1.0, s1("ma"), {Qa, "imjb"});
    b.add(-1.0, s1("mb"), {Qb, "imaj"});
    b.add(1.0, s1("ie"), G1("jbae"));
    b.add(-1.0, s1("ma"), G3("mijb"));
    b.out(nullptr, "ia", "i", "a", n1, "ia", 1.0, S.R1.as<double>(), nn1, ov);
    b.add(1.0, s1("ie"), {Fa, "ae"});
    b.add(-1.0, {Fi, "mi"}, s1("ma"));
  }
  b.launch();

  groups = b.groups;
  const size_t no = b.outs.size() * sizeof(SmallOut<T>), nt = b.terms.size() * sizeof(SmallTerm<T>),
               np = b.points.size() * sizeof(SmallPoint<T>);
  term_at = (no + 15) / 16 * 16;
  point_at = (term_at + nt + 15) / 16 * 16;
  std::vector<char> h(point_at + np);
  std::memcpy(h.data(), b.outs.data(), no);
  std::memcpy(h.data() + term_at, b.terms.data(), nt);
  if (np) std::memcpy(h.data() + point_at, b.points.data(), np);
  desc.alloc(h.size());
  h2d(ctx, desc.p, h.data(), h.size());
}

template <typename T>
void small_contractions(jues_ctx* ctx, CCState& S) {
  const int o = S.o, v = S.v;
  const long N2 = (long)o * o * v * v;
  CCWork<T>& W = work<T>(S);
  const bool cc2 = S.method == 1;
  const double *t2 = S.t.as<double>(), *t1 = cc2 ? t2 + N2 : nullptr;
  if constexpr (sizeof(T) == 4) {
    CCInts<float>& b = *S.i32;
    if (!S.ladder_recompute && !b.Vp.p) {  // made by the stage's first ladder
      bufp_t<float>(b.Vp, S.i64->Vp.bytes / sizeof(double));
      bufp_t<float>(b.Vm, S.i64->Vm.bytes / sizeof(double));
      convert<double, float>(ctx, S.i64->Vp.as<double>(), b.Vp.as<float>(), (long)(S.i64->Vp.bytes / sizeof(double)));
      convert<double, float>(ctx, S.i64->Vm.as<double>(), b.Vm.as<float>(), (long)(S.i64->Vm.bytes / sizeof(double)));
    }
  }
  if (!W.small) {  // (kept only when it is whole: building it allocates)
    std::unique_ptr<SmallPlan<T>> p(new SmallPlan<T>());
    p->build(ctx, S);
    W.small = std::move(p);
  }
  const SmallPlan<T>& plan = *W.small;
  const PairTables& P = S.P;
  SmallPrep<T> A{};
  A.t2 = t2;
  A.t1 = t1;
  A.o = o;
  A.v = v;
  A.P = P;
  if (sizeof(T) == 4) {
    A.t2c = W.Tov.template as<T>();
    if (cc2) A.t1c = W.t1.template as<T>();
  }
  if (cc2) {
    A.tau = W.Tpp.template as<T>();
    A.taup = W.Upp.template as<T>();
    A.xi = W.Ttov.template as<T>();
  }
  if (S.ladder_recompute) {
    ladder_mm<T>(ctx, S, t2, W.Tp.template as<T>(), W.Tm.template as<T>(), W.Lp.template as<T>(),
                 W.Lm.template as<T>(), t1);
  } else {
    A.Tp = W.Tp.template as<T>();
    if (P.nmo > 0 && P.nmv > 0) A.Tm = W.Tm.template as<T>();
  }
  KTimer k(ctx, "cc_small", 0.0, 0.0);
  const long n = N2 + P.npo * P.npv + P.nmo * P.nmv + (long)o * v;
  if (A.t2c || A.tau || A.Tp)
    hipLaunchKernelGGL((small_prep_kernel<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, A);
  const char* d = plan.desc.template as<char>();
  for (const SmallGroup& g : plan.groups) {
    const auto* outs = reinterpret_cast<const SmallOut<T>*>(d) + g.first;
    const auto* terms = reinterpret_cast<const SmallTerm<T>*>(d + plan.term_at);
    const auto* points = reinterpret_cast<const SmallPoint<T>*>(d + plan.point_at);
    hipLaunchKernelGGL((small_contract_kernel<T>), dim3((unsigned)g.tiles), dim3(64 * SW), 0, ctx->stream, outs,
                       g.count, terms, points);
  }
  JUES_HIP(hipGetLastError());
  W.out_H = W.H.template as<T>();
  W.out_Y = W.Y.template as<T>();
  W.out_X = W.X2.template as<T>();
}

template struct SmallPlan<double>;
template struct SmallPlan<float>;
template void small_contractions<double>(jues_ctx*, CCState&);
template void small_contractions<float>(jues_ctx*, CCState&);

}  // namespace jues
