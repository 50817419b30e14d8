// Bandwidth-bound kernels of the coupled-cluster iteration: symmetric packing of
// the particle-particle ladder, the fused residual-assembly / Jacobi update /
// energy / DIIS-dot kernel, the deterministic partial-sum reduction, the on-device
// bordered DIIS solve and the extrapolation.
#include "cc_kernels.h"

namespace jues {
namespace {

// pair (p<=q) index p + q(q+1)/2 and strict pair (p<q) index p + q(q-1)/2
__device__ inline long tri_le(int p, int q) { return (long)p + (long)q * (q + 1) / 2; }
__device__ inline long tri_lt(int p, int q) { return (long)p + (long)q * (q - 1) / 2; }

// Tp[(i<=j),(e<=f)] = t[ijef] + t[ijfe] (e<f), t[ijee] (e=f)
// Tm[(i<j),(e<f)]   = t[ijef] - t[ijfe]
// With t1 non-null the packed amplitudes are those of tau = t + t1 t1,
// tau[ijef] = t[ijef] + t1[i,e] t1[j,f] (the CCSD ladders), formed on the fly.
// With ROWDIAG the single term is taken on the row diagonal instead: for the hole-hole
// ladder integrals K[kl,cd] = <kl|cd>, KP[(k<=l),(c<=d)] = K[klcd] + K[kldc] (k<l),
// K[kkcd] (k=l) and KM[(k<l),(c<d)] = K[klcd] - K[kldc].
template <typename T, bool ROWDIAG = false>
__global__ __launch_bounds__(256) void pack_t_kernel(const double* __restrict__ t, const double* __restrict__ t1,
                                                     int o, int v,
                                                     const int2* __restrict__ pairs_o_le, const int2* __restrict__ pairs_v_le,
                                                     long npo, long npv, T* __restrict__ Tp,
                                                     const int2* __restrict__ pairs_o_lt, const int2* __restrict__ pairs_v_lt,
                                                     long nmo, long nmv, T* __restrict__ Tm) {
  const long oo = (long)o * o;
  const long tot_p = npo * npv, tot_m = nmo * nmv;
  for (long x = blockIdx.x * 256L + threadIdx.x; x < tot_p + tot_m; x += (long)gridDim.x * 256L) {
    const bool plus = x < tot_p;
    const long y = plus ? x : x - tot_p;
    const long nr = plus ? npo : nmo;
    const long r = y % nr, c = y / nr;
    const int2 ij = plus ? pairs_o_le[r] : pairs_o_lt[r], ef = plus ? pairs_v_le[c] : pairs_v_lt[c];
    const long base = ij.x + (long)o * ij.y;
    double a = t[base + oo * (ef.x + (long)v * ef.y)];
    double b = t[base + oo * (ef.y + (long)v * ef.x)];
    if (t1) {
      a += t1[ij.x + (long)o * ef.x] * t1[ij.y + (long)o * ef.y];
      b += t1[ij.x + (long)o * ef.y] * t1[ij.y + (long)o * ef.x];
    }
    if (plus) Tp[y] = (T)((ROWDIAG ? ij.x == ij.y : ef.x == ef.y) ? a : a + b);
    else Tm[y] = (T)(a - b);
  }
}

// From a chemist slab X[a,e,b,f'] = (ae|bf) (f' = f - f0, f in [f0,f1); a, e of its rows with e < f1, ldx between
// columns) build
// Vp[(e<=f),(a<=b)] = ((ae|bf) + (af|be))/2 and Vm[(e<f),(a<b)] = ((ae|bf) - (af|be))/2,
// using (af|be) = X[b,e,a,f'].
// Row rr of the packed matrix goes to Vp[(rr - rowp0) + ldp * c] (Vm likewise): the full
// matrix with rowp0 = 0, ldp = npv, or a slab holding only this call's rows.
// X is contiguous in a, the packed rows in e: a workgroup takes 16 a, 16 b >= a and 16 e of one f through LDS, where
// X[a,e,b] and X[b,e,a] give both of V+ and V-, so that every run read or written is 16 elements and X is read once.
// At 190 virtual orbitals the elements one by one, strided, took 21 ms at 0.75 TB/s, 3.6 this way.
template <typename T>
__global__ __launch_bounds__(256) void pack_v_kernel(const T* __restrict__ X, long ldx, int v, int f0,
                                                     T* __restrict__ Vp, long rowp0, long ldp, T* __restrict__ Vm,
                                                     long rowm0, long ldm) {
  constexpr int TS = 16, LD = TS + 1;
  __shared__ T P[TS * TS * LD], Q[TS * TS * LD];  // P[(b 16 + e) LD + a] = X[a,e,b], Q[(a 16 + e) LD + b] = X[b,e,a]
  const int f = f0 + (int)blockIdx.z, e0 = (int)blockIdx.y * TS;
  if (e0 > f) return;
  int tb = (int)((sqrtf(8.0f * blockIdx.x + 1.0f) - 1.0f) / 2.0f);
  while (tb * (tb + 1) / 2 > (int)blockIdx.x) --tb;
  while ((tb + 1) * (tb + 2) / 2 <= (int)blockIdx.x) ++tb;
  const int b0 = tb * TS, a0 = ((int)blockIdx.x - tb * (tb + 1) / 2) * TS;
  const int lo = threadIdx.x & 15, hi = threadIdx.x >> 4;
  const T* Xf = X + ldx * ((long)v * blockIdx.z);
  const int e = min(e0 + hi, f);
  T x[TS];
#pragma unroll
  for (int k = 0; k < TS; ++k) x[k] = Xf[min(a0 + lo, v - 1) + (long)v * e + ldx * min(b0 + k, v - 1)];
#pragma unroll
  for (int k = 0; k < TS; ++k) P[(k * TS + hi) * LD + lo] = x[k];
  if (a0 != b0) {
#pragma unroll
    for (int k = 0; k < TS; ++k) x[k] = Xf[min(b0 + lo, v - 1) + (long)v * e + ldx * min(a0 + k, v - 1)];
#pragma unroll
    for (int k = 0; k < TS; ++k) Q[(k * TS + hi) * LD + lo] = x[k];
  }
  __syncthreads();
  const T* q = a0 != b0 ? Q : P;
  const int ee = e0 + lo, a = a0 + hi;
  const long rp = (long)f * (f + 1) / 2 + ee - rowp0, rm = (long)f * (f - 1) / 2 + ee - rowm0;
  if (ee > f) return;
#pragma unroll
  for (int k = 0; k < TS; ++k) {
    const int b = b0 + k;
    if (b >= v || a > b) continue;
    const double s = (double)P[(k * TS + lo) * LD + hi], t = (double)q[(hi * TS + lo) * LD + k];
    Vp[rp + ldp * (a + (long)b * (b + 1) / 2)] = (T)(0.5 * (s + t));
    if (ee < f && a < b) Vm[rm + ldm * (a + (long)b * (b - 1) / 2)] = (T)(0.5 * (s - t));
  }
}

// G+-[(e,f),(a,m)] = ((mf|ae) +- (me|af))/2 from X[f,m,a,e] = (mf|ae): as pack_v_kernel, but X is contiguous in f and
// the column (a,m) is no pair.  A workgroup takes 16 e, 16 f >= e and 8 columns: X[f,e] goes through LDS, X[e,f] is
// read as it is written.  Bound by memory.
template <typename T>
__global__ __launch_bounds__(256) void pack_z_kernel(const T* __restrict__ X, int v, int cnt, long npv,
                                                     T* __restrict__ Gp, long nmv, T* __restrict__ Gm) {
  constexpr int TS = 16, LD = TS + 1, NC = 8;
  __shared__ T P[NC][TS * LD];
  int tf = (int)((sqrtf(8.0f * blockIdx.x + 1.0f) - 1.0f) / 2.0f);
  while (tf * (tf + 1) / 2 > (int)blockIdx.x) --tf;
  while ((tf + 1) * (tf + 2) / 2 <= (int)blockIdx.x) ++tf;
  const int f0 = tf * TS, e0 = ((int)blockIdx.x - tf * (tf + 1) / 2) * TS;
  const int lo = threadIdx.x & 15, hi = threadIdx.x >> 4;
  const long nr = (long)v * cnt, c0 = (long)blockIdx.y * NC;
  const auto at = [&](int f, int e, long c) {
    const int a = (int)(c % v), m = (int)(c / v);
    return X[min(f, v - 1) + (long)v * m + nr * (a + (long)v * min(e, v - 1))];
  };
  T x[NC], y[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) x[k] = at(f0 + lo, e0 + hi, min(c0 + k, nr - 1));
#pragma unroll
  for (int k = 0; k < NC; ++k) y[k] = e0 == f0 ? x[k] : at(e0 + lo, f0 + hi, min(c0 + k, nr - 1));
#pragma unroll
  for (int k = 0; k < NC; ++k) P[k][hi * LD + lo] = x[k];
  __syncthreads();
  const int e = e0 + lo, f = f0 + hi;
  if (f >= v || e > f) return;
  const long rp = (long)f * (f + 1) / 2 + e, rm = (long)f * (f - 1) / 2 + e;
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const long c = c0 + k;
    if (c >= nr) return;
    const double s = (double)P[k][lo * LD + hi], t = (double)y[k];
    Gp[rp + npv * c] = (T)(0.5 * (s + t));
    if (e < f) Gm[rm + nmv * c] = (T)(0.5 * (s - t));
  }
}

template <typename T>
__global__ __launch_bounds__(256) void unpack_z_kernel(const T* __restrict__ Zp, const T* __restrict__ Zm, int o,
                                                       long npo, long nmo, long total, T* __restrict__ Z) {
  const int oo = o * o;
  for (long x = blockIdx.x * 256L + threadIdx.x; x < total; x += (long)gridDim.x * 256L) {
    const long c = x / oo;
    const int ij = (int)(x - c * oo), i = ij % o, j = ij / o, p = min(i, j), q = max(i, j);
    T z = Zp[tri_le(p, q) + npo * c];
    if (Zm && i != j) {
      const T w = Zm[tri_lt(p, q) + nmo * c];
      z += i < j ? w : -w;
    }
    Z[x] = z;
  }
}

// W[m,n,i,j] (o^4, holding <mn|ij> plus any T1 terms) on packed pairs, transposed:
// WPT[(i<=j),(k<=l)] = W[klij] + W[lkij] (k<l), W[kkij] (k=l);  WMT[(i<j),(k<l)] = W[klij] - W[lkij]
template <typename T>
__global__ __launch_bounds__(256) void pack_whh_kernel(const T* __restrict__ W, int o, const int2* __restrict__ o_le,
                                                       long npo, T* __restrict__ WPT, const int2* __restrict__ o_lt,
                                                       long nmo, T* __restrict__ WMT) {
  const long oo = (long)o * o;
  const long tot_p = npo * npo, tot_m = nmo * nmo;
  for (long x = blockIdx.x * 256L + threadIdx.x; x < tot_p + tot_m; x += (long)gridDim.x * 256L) {
    const bool plus = x < tot_p;
    const long y = plus ? x : x - tot_p, n = plus ? npo : nmo;
    const long r = y % n, c = y / n;
    const int2 ij = plus ? o_le[r] : o_lt[r], kl = plus ? o_le[c] : o_lt[c];
    const long col = oo * (ij.x + (long)o * ij.y);
    const double a = (double)W[kl.x + (long)o * kl.y + col];
    const double b = (double)W[kl.y + (long)o * kl.x + col];
    if (plus) WPT[y] = (T)(kl.x == kl.y ? a : a + b);
    else WMT[y] = (T)(a - b);
  }
}

// Tq = Tp with its (a,a) columns doubled (exact)
template <typename T>
__global__ __launch_bounds__(256) void pair_diag2_kernel(const T* __restrict__ Tp, long npo, long npv,
                                                         const int2* __restrict__ v_le, T* __restrict__ Tq) {
  for (long x = blockIdx.x * 256L + threadIdx.x; x < npo * npv; x += (long)gridDim.x * 256L) {
    const int2 ab = v_le[x / npo];
    const T t = Tp[x];
    Tq[x] = ab.x == ab.y ? t + t : t;
  }
}

// WE[(k,c),(j,b)] += s (delta_kj Fae[b,c] - delta_cb Fmi[k,j]) on the ov layout (row k + o c,
// column j + o b), with Fmi held transposed (FmiT[j,k] = Fmi[k,j]).  Threads x < o v^2 take
// the (k,c,b) entries with j = k (and the Fmi part where c = b); the rest take (k, j != k, b)
// with c = b, so every entry has one writer.
template <typename T>
__global__ __launch_bounds__(256) void fock_dress_kernel(T* __restrict__ WE, const T* __restrict__ Fae,
                                                         const T* __restrict__ FmiT, int o, int v, T s) {
  const long ov = (long)o * v, n1 = ov * v, n2 = (long)o * (o - 1) * v;
  for (long x = blockIdx.x * 256L + threadIdx.x; x < n1 + n2; x += (long)gridDim.x * 256L) {
    if (x < n1) {
      const int k = (int)(x % o);
      const long cb = x / o;
      const int c = (int)(cb % v), b = (int)(cb / v);
      T d = Fae[b + (long)v * c];
      if (c == b) d -= FmiT[k + (long)o * k];
      WE[k + (long)o * c + ov * (k + (long)o * b)] += s * d;
    } else {
      const long y = x - n1;
      const int k = (int)(y % o);
      const long jb = y / o;
      const int jj = (int)(jb % (o - 1)), b = (int)(jb / (o - 1));
      const int j = jj < k ? jj : jj + 1;
      WE[k + (long)o * b + ov * (j + (long)o * b)] -= s * FmiT[j + (long)o * k];
    }
  }
}

// Start of the ring intermediates: WE = s X + D/2 and W = K + WE/2 (+ A), D as in fock_dress_kernel (X may be WE).
// One pass at the copy rate in place of a copy, a scaled copy and the two dressings.
template <typename T>
__global__ __launch_bounds__(256) void ring_start_kernel(const T* __restrict__ K, T s, const T* X,
                                                         const T* __restrict__ Fae, const T* __restrict__ FmiT, int o,
                                                         int v, T* WE, T* __restrict__ W, const T* __restrict__ A) {
  const int ov = o * v;
  for (int jb = blockIdx.x; jb < ov; jb += gridDim.x) {
    const int j = jb % o, b = jb / o;
    for (int kc = threadIdx.x; kc < ov; kc += 256) {
      const int k = kc % o, c = kc / o;
      const long x = kc + (long)ov * jb;
      T w = s * X[x];
      if (k == j) w += T(0.5) * Fae[b + (long)v * c];
      if (c == b) w -= T(0.5) * FmiT[j + (long)o * k];
      WE[x] = w;
      W[x] = A ? K[x] + T(0.5) * w + A[x] : K[x] + T(0.5) * w;
    }
  }
}

// The RCCD residual's amplitude layouts from t2 (FP64, [i,j,a,b]) in one pass:
// Tpp = t, Upp = 2t - t^(ij) ([i,j,a,b]); Uov[i,a,j,b] = U[ijab];
// Ttov[i,b,j,a] = t[ijab] (that is t[i,j,b,a] at [i,a,j,b]).  Threads run i fastest, so
// every write is a contiguous run of o; the exchanged read t[jiab] stays in one o x o slab.
template <typename T>
__global__ __launch_bounds__(256) void rccd_layouts_kernel(const double* __restrict__ t, int o, int v,
                                                           T* __restrict__ Tpp, T* __restrict__ Upp,
                                                           T* __restrict__ Ttov, T* __restrict__ Uov) {
  const long oo = (long)o * o, ov = (long)o * v, n = oo * v * v;
  for (long x = blockIdx.x * 256L + threadIdx.x; x < n; x += (long)gridDim.x * 256L) {
    const long ij = x % oo, ab = x / oo;
    const int i = (int)(ij % o), j = (int)(ij / o);
    const int a = (int)(ab % v), b = (int)(ab / v);
    const double tv = t[x];
    const double u = 2.0 * tv - t[j + (long)o * i + oo * ab];
    if (Tpp) Tpp[x] = (T)tv;
    if (Upp) Upp[x] = (T)u;
    const long y = i + (long)o * a + ov * (j + (long)o * b);
    Uov[y] = (T)u;
    Ttov[i + (long)o * b + ov * (j + (long)o * a)] = (T)tv;
  }
}

// The same layouts with the o x o slab t[:,:,a,b] of one (a,b) pair staged in LDS (rows padded to
// o + 1), so that the exchanged read t[j,i,a,b] comes from LDS and every global read is
// contiguous.  Dynamic LDS: o (o + 1) doubles.
template <typename T>
__global__ __launch_bounds__(256) void rccd_layouts_slab_kernel(const double* __restrict__ t, int o, int v,
                                                                T* __restrict__ Tpp, T* __restrict__ Upp,
                                                                T* __restrict__ Ttov, T* __restrict__ Uov) {
  extern __shared__ double slab[];  // slab[i + (o + 1) j] = t[i,j,a,b]
  const int oo = o * o, ld = o + 1;
  const long ov = (long)o * v, vv = (long)v * v;
  for (long ab = blockIdx.x; ab < vv; ab += gridDim.x) {
    const int a = (int)(ab % v), b = (int)(ab / v);
    const double* src = t + ab * oo;
    __syncthreads();  // the previous pair's readers are done with the slab
    for (int q = threadIdx.x; q < oo; q += 256) slab[q % o + ld * (q / o)] = src[q];
    __syncthreads();
    for (int q = threadIdx.x; q < oo; q += 256) {
      const int i = q % o, j = q / o;
      const double tv = slab[i + ld * j];
      const double u = 2.0 * tv - slab[j + ld * i];
      if (Tpp) Tpp[ab * oo + q] = (T)tv;
      if (Upp) Upp[ab * oo + q] = (T)u;
      const long y = i + (long)o * a + ov * (j + (long)o * b);
      Uov[y] = (T)u;
      Ttov[i + (long)o * b + ov * (j + (long)o * a)] = (T)tv;
    }
  }
}

__device__ inline double block_sum256(double v, double* sh) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// One block per (a,b): assemble R[ijab] = K[ijab] + S[ia,jb] + L+ + L- (both ladders) + X[ijab] + X[jiba] (extra),
// t_new = R/D, e = t_new - t_old; write t_new and e into the DIIS slot; block
// partial sums of E = sum Lener*t_new, e.e and e.e_k for the stored errors.
template <typename TR>
__global__ __launch_bounds__(256) void t2_update_kernel(UpdateArgs<TR> A) {
  __shared__ double sh[4];
  const int o = A.o, v = A.v;
  const int ab = blockIdx.x;
  const int a = ab % v, b = ab / v;
  const long oo = (long)o * o, ov = (long)o * v;
  const double dab = -A.eps[o + a] - A.eps[o + b];
  const int sab = a < b ? 1 : (a > b ? -1 : 0);
  const long qp = a <= b ? (long)a + (long)b * (b + 1) / 2 : (long)b + (long)a * (a + 1) / 2;
  const long qm = a < b ? (long)a + (long)b * (b - 1) / 2 : (long)b + (long)a * (a - 1) / 2;
  double sE = 0.0, sEE = 0.0;
  double sd[MAX_DIIS];
#pragma unroll
  for (int k = 0; k < MAX_DIIS; ++k) sd[k] = 0.0;
  // fused symmetrisation: the transposed terms H[jb,ia] + Y[ja,ib] run along j in memory, so
  // they are read as contiguous j-runs into an LDS slab[j + (o + 1) i] and taken from there
  extern __shared__ __attribute__((aligned(16))) unsigned char dyn_lds[];
  TR* slab = reinterpret_cast<TR*>(dyn_lds);
  const int ld = o + 1;
  // (each of Y's two o x o blocks serves an exchanged and a direct term)
  const TR yd = (TR)A.y_direct;
  if (A.H) {
    for (int q = threadIdx.x; q < (int)oo; q += 256) {
      const int j = q % o, i = q / o;
      const long ba = (long)j + (long)o * b + ov * ((long)i + (long)o * a);
      slab[j + ld * i] = A.H[ba] + A.Y[(long)j + (long)o * a + ov * ((long)i + (long)o * b)] + yd * A.Y[ba];
    }
    __syncthreads();
  }
  for (int ij = threadIdx.x; ij < (int)oo; ij += 256) {
    const int i = ij % o, j = ij / o;
    const long x = (long)ij + oo * ab;
    double R = A.Kpp[x];
    if (A.S) R += (double)A.S[(long)i + (long)o * a + ov * ((long)j + (long)o * b)];
    if (A.H) {
      const long iajb = (long)i + (long)o * a + ov * ((long)j + (long)o * b);
      R += (double)A.H[iajb] + (double)A.Y[(long)i + (long)o * b + ov * ((long)j + (long)o * a)] +
           A.y_direct * (double)A.Y[iajb] + (double)slab[j + ld * i];
    }
    if (A.Lp) {
      const long pp = i <= j ? (long)i + (long)j * (j + 1) / 2 : (long)j + (long)i * (i + 1) / 2;
      R += (double)A.Lp[pp + A.npo * qp];
      const int sij = i < j ? 1 : (i > j ? -1 : 0);
      if (sij != 0 && sab != 0) {
        const long pm = i < j ? (long)i + (long)j * (j - 1) / 2 : (long)j + (long)i * (i - 1) / 2;
        R += (double)(sij * sab) * (double)A.Lm[pm + A.nmo * qm];
      }
    }
    if (A.extra) R += (double)A.extra[x] + (double)A.extra[j + (long)o * i + oo * (b + (long)v * a)];
    if (A.R_out) A.R_out[x] = R;
    const double tn = A.lambda * R / (A.eps[i] + A.eps[j] + dab);
    const double e = tn - A.t_old[x];
    A.t_new[x] = tn;
    A.e_new[x] = e;
    const double tt = A.t1n ? A.t1n[i + (long)o * a] * A.t1n[j + (long)o * b] : 0.0;
    sE += A.lambda * A.Lener[x] * (tn + tt);
    sEE += e * e;
#pragma unroll
    for (int k = 0; k < MAX_DIIS; ++k)
      if (k < A.nold) sd[k] += e * A.e_old[k][x];
  }
  const long PB = A.part_stride;
  double r = block_sum256(sE, sh);
  if (threadIdx.x == 0) A.part[0 * PB + A.part_off + blockIdx.x] = r;
  r = block_sum256(sEE, sh);
  if (threadIdx.x == 0) A.part[1 * PB + A.part_off + blockIdx.x] = r;
  for (int k = 0; k < A.nold; ++k) {
    r = block_sum256(sd[k], sh);
    if (threadIdx.x == 0) A.part[(2 + k) * PB + A.part_off + blockIdx.x] = r;
  }
}

// T1 part of the update: t1_new = R1/D_ia, error and partials (RCCSD).
__global__ __launch_bounds__(256) void t1_update_kernel(T1UpdateArgs A) {
  __shared__ double sh[4];
  const long n1 = (long)A.o * A.v;
  double sE = 0.0, sEE = 0.0, sd[MAX_DIIS];
#pragma unroll
  for (int k = 0; k < MAX_DIIS; ++k) sd[k] = 0.0;
  for (long x = blockIdx.x * 256L + threadIdx.x; x < n1; x += (long)gridDim.x * 256L) {
    const int i = (int)(x % A.o), a = (int)(x / A.o);
    const double tn = A.lambda * A.R1[x] / (A.eps[i] - A.eps[A.o + a]);
    const double e = tn - A.t_old[x];
    A.t_new[x] = tn;
    A.e_new[x] = e;
    sE += A.Lener1 ? A.Lener1[x] * tn : 0.0;
    sEE += e * e;
#pragma unroll
    for (int k = 0; k < MAX_DIIS; ++k)
      if (k < A.nold) sd[k] += e * A.e_old[k][x];
  }
  const long PB = A.part_stride;
  double r = block_sum256(sE, sh);
  if (threadIdx.x == 0) A.part[0 * PB + A.part_off + blockIdx.x] = r;
  r = block_sum256(sEE, sh);
  if (threadIdx.x == 0) A.part[1 * PB + A.part_off + blockIdx.x] = r;
  for (int k = 0; k < A.nold; ++k) {
    r = block_sum256(sd[k], sh);
    if (threadIdx.x == 0) A.part[(2 + k) * PB + A.part_off + blockIdx.x] = r;
  }
}

// Fixed-order sums of nq partial arrays; out[q] = sum_b part[q*PB + b].
__global__ __launch_bounds__(256) void reduce_rows_kernel(const double* __restrict__ part, long PB, long count,
                                                          double* __restrict__ out) {
  __shared__ double sh[256];
  const int q = blockIdx.x;
  double s = 0.0;
  for (long b = threadIdx.x; b < count; b += 256) s += part[q * PB + b];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[q] = sh[0];
}

// Store the new B row/column and solve the bordered Pulay system (mRCCD.jl:185-198)
// in FP64 with partial pivoting.  small layout: [0]=E, [1]=ee, [2..2+nold)=dots,
// B at SMALL_B (MAX_DIIS^2, by slot), coefficients at SMALL_C (MAX_DIIS, by order).
// One wavefront with the augmented matrix (at most 9 x 10) in LDS: the elements of an elimination step are
// independent, so they are updated together.  (One thread on arrays that the compiler put in scratch memory
// took 24 us at five vectors and 37 us behind a larger solve, of an iteration of 150 us at n = 24.)
// With `part` the sums small[0 .. 2 + nold) are formed here first, each over PB partial sums by one
// wavefront in a fixed order: one launch less where there are few of them.
__global__ __launch_bounds__(256) void diis_solve_kernel(double* small, DiisOrder ord, const double* __restrict__ part,
                                                         long PB) {
  constexpr int NMAX = MAX_DIIS + 1;
  __shared__ double M[NMAX][NMAX + 1];  // column N: the right-hand side, then the solution
  __shared__ double B[MAX_DIIS][MAX_DIIS];
  __shared__ double sums[2 + MAX_DIIS];
  const int t = threadIdx.x;
  for (int q = t >> 6; q < 2 + ord.nold; q += blockDim.x >> 6) {
    double s = 0.0;
    if (part) {
      for (long x = t & 63; x < PB; x += 64) s += part[q * PB + x];
      for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    } else {
      s = small[q];
    }
    if ((t & 63) == 0) {
      sums[q] = s;
      if (part) small[q] = s;
    }
  }
  for (int e = t; e < MAX_DIIS * MAX_DIIS; e += blockDim.x) B[e / MAX_DIIS][e % MAX_DIIS] = small[SMALL_B + e];
  __syncthreads();
  if (t >= 64) return;
  // the rest is the first wavefront's: its lanes' accesses to LDS are in order, so between them only the compiler has to
  // keep that order (a workgroup barrier would have to be reached by the wavefronts that are done, too)
  const auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
  };
  const int s = ord.newest;
  if (t <= ord.nold) {
    const int sk = t < ord.nold ? ord.old_slots[t] : s;
    const double d = t < ord.nold ? sums[2 + t] : sums[1];
    B[s][sk] = B[sk][s] = d;
    small[SMALL_B + s * MAX_DIIS + sk] = small[SMALL_B + sk * MAX_DIIS + s] = d;
  }
  const int m = ord.m, N = m + 1;
  double* c = small + SMALL_C;
  if (m == 1) {
    if (t == 0) { c[0] = 1.0; small[SMALL_FLAG] = 0.0; }
    return;
  }
  wave_sync();
  double mx = t < m * m ? fabs(B[ord.slots[t / m]][ord.slots[t % m]]) : 0.0;  // m * m <= 64
  for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
  if (!(mx > 0.0)) mx = 1.0;
  for (int e = t; e < N * (N + 1); e += 64) {
    const int p = e / (N + 1), q = e % (N + 1);
    double val;
    if (q == N) val = p == m ? -1.0 : 0.0;
    else if (p < m && q < m) val = B[ord.slots[p]][ord.slots[q]] / mx;
    else val = p == m && q == m ? 0.0 : -1.0;
    M[p][q] = val;
  }
  wave_sync();
  bool ok = true;
  for (int k = 0; k < N; ++k) {
    // the first row of the largest |M[p][k]|, p >= k
    double best = t >= k && t < N ? fabs(M[t][k]) : -1.0;
    int piv = t;
    for (int off = 8; off > 0; off >>= 1) {
      const double ob = __shfl_xor(best, off, 64);
      const int op = __shfl_xor(piv, off, 64);
      if (ob > best || (ob == best && op < piv)) { best = ob; piv = op; }
    }
    best = __shfl(best, 0, 64);
    piv = __shfl(piv, 0, 64);
    if (!(best > 1e-300)) { ok = false; break; }
    if (piv != k && t <= N) { const double tmp = M[k][t]; M[k][t] = M[piv][t]; M[piv][t] = tmp; }
    wave_sync();
    // rows below k; column k itself is not read again
    const int rows = N - 1 - k, cols = N - k;
    for (int e = t; e < rows * cols; e += 64) {
      const int p = k + 1 + e / cols, q = k + 1 + e % cols;
      const double f = M[p][k] / M[k][k];
      M[p][q] -= f * M[k][q];
    }
    wave_sync();
  }
  if (ok) {
    for (int k = N - 1; k >= 0; --k) {
      const double xk = M[k][N] / M[k][k];
      wave_sync();
      if (t < k) M[t][N] -= M[t][k] * xk;
      else if (t == k) M[k][N] = xk;
      wave_sync();
    }
    for (int p = 0; p < m; ++p) ok = ok && isfinite(M[p][N]);
  }
  // a singular subspace: take the newest vector (a plain Jacobi step)
  if (t < m) c[t] = ok ? M[t][N] : (t == m - 1 ? 1.0 : 0.0);
  if (t == 0) small[SMALL_FLAG] = ok ? 0.0 : 1.0;
}

// t[x] = sum_k c_k vals[slot_k][x]
__global__ __launch_bounds__(256) void diis_extrap_kernel(const double* __restrict__ vals, long stride, DiisOrder ord,
                                                          const double* __restrict__ small, long n, double* __restrict__ t) {
  double c[MAX_DIIS];
#pragma unroll
  for (int k = 0; k < MAX_DIIS; ++k) c[k] = k < ord.m ? small[SMALL_C + k] : 0.0;
  for (long x = blockIdx.x * 256L + threadIdx.x; x < n; x += (long)gridDim.x * 256L) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < MAX_DIIS; ++k)
      if (k < ord.m) s += c[k] * vals[(long)ord.slots[k] * stride + x];
    t[x] = s;
  }
}

// t[ijab] /= D[ijab]
__global__ __launch_bounds__(256) void divide_d2_kernel(double* __restrict__ t, const double* __restrict__ eps, int o,
                                                        int v, double scale) {
  const long oo = (long)o * o, n = oo * v * v;
  for (long x = blockIdx.x * 256L + threadIdx.x; x < n; x += (long)gridDim.x * 256L) {
    const long ij = x % oo, ab = x / oo;
    const int i = (int)(ij % o), j = (int)(ij / o), a = (int)(ab % v), b = (int)(ab / v);
    t[x] = scale * t[x] / (eps[i] + eps[j] - eps[o + a] - eps[o + b]);
  }
}

int grid256(long n) { return (int)std::max(1L, std::min((n + 255) / 256, 131072L)); }

}  // namespace

template <typename T>
void pack_t(jues_ctx* ctx, const PairTables& P, const double* t, int o, int v, T* Tp, T* Tm, const double* t1) {
  const long tot = P.npo * P.npv + P.nmo * P.nmv;
  KTimer k(ctx, "cc_pack_t", 0.0, (double)tot * (16.0 + sizeof(T)));
  hipLaunchKernelGGL((pack_t_kernel<T>), dim3(grid256(tot)), dim3(256), 0, ctx->stream, t, t1, o, v, P.o_le, P.v_le,
                     P.npo, P.npv, Tp, P.o_lt, P.v_lt, P.nmo, P.nmv, Tm);
  JUES_HIP(hipGetLastError());
}

void pack_khh(jues_ctx* ctx, const PairTables& P, const double* K, int o, int v, double* KP, double* KM) {
  const long tot = P.npo * P.npv + P.nmo * P.nmv;
  KTimer k(ctx, "cc_pack_k", 0.0, (double)tot * 24.0);
  hipLaunchKernelGGL((pack_t_kernel<double, true>), dim3(grid256(tot)), dim3(256), 0, ctx->stream, K, nullptr, o, v,
                     P.o_le, P.v_le, P.npo, P.npv, KP, P.o_lt, P.v_lt, P.nmo, P.nmv, KM);
  JUES_HIP(hipGetLastError());
}

template <typename T>
void pack_whh(jues_ctx* ctx, const PairTables& P, const T* W, int o, T* WPT, T* WMT) {
  const long tot = P.npo * P.npo + P.nmo * P.nmo;
  KTimer k(ctx, "cc_hh_pack", 0.0, (double)tot * 3.0 * sizeof(T));
  hipLaunchKernelGGL((pack_whh_kernel<T>), dim3(grid256(tot)), dim3(256), 0, ctx->stream, W, o, P.o_le, P.npo, WPT,
                     P.o_lt, P.nmo, WMT);
  JUES_HIP(hipGetLastError());
}

template <typename T>
void pair_diag2(jues_ctx* ctx, const PairTables& P, const T* Tp, T* Tq) {
  const long tot = P.npo * P.npv;
  KTimer k(ctx, "cc_hh_pack", 0.0, (double)tot * 2.0 * sizeof(T));
  hipLaunchKernelGGL((pair_diag2_kernel<T>), dim3(grid256(tot)), dim3(256), 0, ctx->stream, Tp, P.npo, P.npv, P.v_le,
                     Tq);
  JUES_HIP(hipGetLastError());
}

template <typename T>
void fock_dress(jues_ctx* ctx, T* WE, const T* Fae, const T* FmiT, int o, int v, T s) {
  const long n = (long)o * v * v + (long)o * (o - 1) * v;
  KTimer k(ctx, "cc_fock", 0.0, (double)n * 3.0 * sizeof(T));
  hipLaunchKernelGGL((fock_dress_kernel<T>), dim3(grid256(n)), dim3(256), 0, ctx->stream, WE, Fae, FmiT, o, v, s);
  JUES_HIP(hipGetLastError());
}

template <typename T>
void ring_start(jues_ctx* ctx, const T* K, T s, const T* X, const T* Fae, const T* FmiT, int o, int v, T* WE, T* W,
                const T* A) {
  const long n = (long)o * v * o * v;
  KTimer k(ctx, "cc_prep", 0.0, (double)n * (A ? 5.0 : 4.0) * sizeof(T));
  hipLaunchKernelGGL((ring_start_kernel<T>), dim3((unsigned)std::min((long)o * v, 1L << 20)), dim3(256), 0, ctx->stream, K, s, X, Fae, FmiT, o, v,
                     WE, W, A);
  JUES_HIP(hipGetLastError());
}

template <typename T>
void rccd_layouts(jues_ctx* ctx, const double* t, int o, int v, T* Tpp, T* Upp, T* Ttov, T* Uov) {
  const long n = (long)o * o * v * v;
  const size_t slab = (size_t)o * (o + 1) * sizeof(double);
  // t is read once through the LDS slab, twice (direct and exchanged) otherwise
  const double outs = 2.0 + (Tpp ? 1.0 : 0.0) + (Upp ? 1.0 : 0.0);
  KTimer k(ctx, "cc_prep", 0.0, (double)n * ((slab <= 65536 ? 8.0 : 16.0) + outs * sizeof(T)));
  if (slab <= 65536) {
    const long vv = (long)v * v;
    hipLaunchKernelGGL((rccd_layouts_slab_kernel<T>), dim3((unsigned)std::min(vv, 1L << 20)), dim3(256), slab,
                       ctx->stream, t, o, v, Tpp, Upp, Ttov, Uov);
  } else {
    hipLaunchKernelGGL((rccd_layouts_kernel<T>), dim3(grid256(n)), dim3(256), 0, ctx->stream, t, o, v, Tpp, Upp, Ttov,
                       Uov);
  }
  JUES_HIP(hipGetLastError());
}

template <typename T>
void pack_z(jues_ctx* ctx, const PairTables& P, const T* X, int v, int cnt, T* Gp, T* Gm) {
  const int nt = (v + 15) / 16;
  const long nr = (long)v * cnt;
  JUES_REQUIRE(nr <= 8L * 65535, "pack_z: too many columns");
  KTimer k(ctx, "cc_ovvv_gen", 0.0, (double)v * v * nr * 2 * sizeof(T));
  hipLaunchKernelGGL((pack_z_kernel<T>), dim3((unsigned)(nt * (nt + 1) / 2), (unsigned)((nr + 7) / 8)), dim3(256), 0,
                     ctx->stream, X, v, cnt, P.npv, Gp, P.nmv, Gm);
  JUES_HIP(hipGetLastError());
}

template <typename T>
void unpack_z(jues_ctx* ctx, const PairTables& P, const T* Zp, const T* Zm, int o, int v, T* Z) {
  const long n = (long)o * o * o * v;
  KTimer k(ctx, "cc_ovvv_gen", 0.0, (double)n * 2 * sizeof(T));
  hipLaunchKernelGGL((unpack_z_kernel<T>), dim3(grid256(n)), dim3(256), 0, ctx->stream, Zp, Zm, o, P.npo, P.nmo, n, Z);
  JUES_HIP(hipGetLastError());
}

template void pack_z<double>(jues_ctx*, const PairTables&, const double*, int, int, double*, double*);
template void pack_z<float>(jues_ctx*, const PairTables&, const float*, int, int, float*, float*);
template void unpack_z<double>(jues_ctx*, const PairTables&, const double*, const double*, int, int, double*);
template void unpack_z<float>(jues_ctx*, const PairTables&, const float*, const float*, int, int, float*);

template <typename T>
void pack_v(jues_ctx* ctx, const PairTables& P, const T* X, long ldx, int v, int f0, int f1, T* Vp, long rowp0,
            long ldp, T* Vm, long rowm0, long ldm) {
  const double rows = 0.5 * f1 * (f1 + 1) - 0.5 * f0 * (f0 + 1);
  const int nt = (v + 15) / 16;
  KTimer k(ctx, "cc_pack_v", 0.0, rows * ((double)v * v + P.npv + P.nmv) * sizeof(T));
  for (int f = f0; f < f1; f += 32768)
    hipLaunchKernelGGL((pack_v_kernel<T>),
                       dim3((unsigned)(nt * (nt + 1) / 2), (unsigned)((f1 + 15) / 16), (unsigned)std::min(f1 - f, 32768)),
                       dim3(256), 0, ctx->stream, X + ldx * v * (f - f0), ldx, v, f, Vp, rowp0, ldp, Vm, rowm0, ldm);
  JUES_HIP(hipGetLastError());
}

template <typename TR>
void t2_update(jues_ctx* ctx, const UpdateArgs<TR>& A) {
  const long v2 = (long)A.v * A.v;
  const long n2 = (long)A.o * A.o * v2;
  // S (or H and Y, each read twice), Lp, Lm and extra in the residual's compute type
  KTimer k(ctx, "cc_update", 0.0, (double)n2 * (8.0 * (5 + A.nold + (A.R_out ? 1 : 0)) + (A.H ? 7 : 4) * sizeof(TR)));
  size_t lds = 0;
  JUES_REQUIRE(A.H || A.S, "t2_update: no ring terms");
  if (A.H) {
    JUES_REQUIRE(A.Y && !A.S && fused_sym(A.o, sizeof(TR)), "t2_update: fused symmetrisation misconfigured");
    lds = (size_t)A.o * (A.o + 1) * sizeof(TR);
  }
  hipLaunchKernelGGL((t2_update_kernel<TR>), dim3((unsigned)v2), dim3(256), lds, ctx->stream, A);
  JUES_HIP(hipGetLastError());
}

void t1_update(jues_ctx* ctx, const T1UpdateArgs& A, int nblocks) {
  hipLaunchKernelGGL(t1_update_kernel, dim3(nblocks), dim3(256), 0, ctx->stream, A);
  JUES_HIP(hipGetLastError());
}

void reduce_rows(jues_ctx* ctx, const double* part, long PB, long count, int nq, double* out) {
  hipLaunchKernelGGL(reduce_rows_kernel, dim3(nq), dim3(256), 0, ctx->stream, part, PB, count, out);
  JUES_HIP(hipGetLastError());
}

void diis_solve(jues_ctx* ctx, double* small, const DiisOrder& ord, const double* part, long PB) {
  // up to 8192 partial sums take the solve's own workgroup under 2 us; more are spread over a launch of their own
  const bool fused = PB * (2 + ord.nold) <= 8192;
  if (!fused) reduce_rows(ctx, part, PB, PB, 2 + ord.nold, small);
  hipLaunchKernelGGL(diis_solve_kernel, dim3(1), dim3(fused ? 256 : 64), 0, ctx->stream, small, ord,
                     fused ? part : nullptr, PB);
  JUES_HIP(hipGetLastError());
}

void diis_extrap(jues_ctx* ctx, const double* vals, long stride, const DiisOrder& ord, const double* small, long n,
                 double* t) {
  KTimer k(ctx, "cc_diis_extrap", 0.0, (double)n * 8.0 * (ord.m + 1));
  hipLaunchKernelGGL(diis_extrap_kernel, dim3(grid256(n)), dim3(256), 0, ctx->stream, vals, stride, ord, small, n, t);
  JUES_HIP(hipGetLastError());
}

void divide_d2(jues_ctx* ctx, double* t, const double* eps, int o, int v, double scale) {
  const long n = (long)o * o * v * v;
  hipLaunchKernelGGL(divide_d2_kernel, dim3(grid256(n)), dim3(256), 0, ctx->stream, t, eps, o, v, scale);
  JUES_HIP(hipGetLastError());
}

template void fock_dress<double>(jues_ctx*, double*, const double*, const double*, int, int, double);
template void fock_dress<float>(jues_ctx*, float*, const float*, const float*, int, int, float);
template void ring_start<double>(jues_ctx*, const double*, double, const double*, const double*, const double*, int,
                                 int, double*, double*, const double*);
template void ring_start<float>(jues_ctx*, const float*, float, const float*, const float*, const float*, int, int,
                                float*, float*, const float*);
template void rccd_layouts<double>(jues_ctx*, const double*, int, int, double*, double*, double*, double*);
template void rccd_layouts<float>(jues_ctx*, const double*, int, int, float*, float*, float*, float*);
template void pack_whh<double>(jues_ctx*, const PairTables&, const double*, int, double*, double*);
template void pack_whh<float>(jues_ctx*, const PairTables&, const float*, int, float*, float*);
template void pair_diag2<double>(jues_ctx*, const PairTables&, const double*, double*);
template void pair_diag2<float>(jues_ctx*, const PairTables&, const float*, float*);
template void pack_t<double>(jues_ctx*, const PairTables&, const double*, int, int, double*, double*, const double*);
template void pack_t<float>(jues_ctx*, const PairTables&, const double*, int, int, float*, float*, const double*);
template void pack_v<double>(jues_ctx*, const PairTables&, const double*, long, int, int, int, double*, long, long,
                             double*, long, long);
template void pack_v<float>(jues_ctx*, const PairTables&, const float*, long, int, int, int, float*, long, long, float*,
                            long, long);
template void t2_update<double>(jues_ctx*, const UpdateArgs<double>&);
template void t2_update<float>(jues_ctx*, const UpdateArgs<float>&);

}  // namespace jues
