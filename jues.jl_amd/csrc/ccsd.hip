// RCCSD residual on the device (CoupledCluster/mRCCSD.jl:118-241, and the
// RCCSD.jl:187-289 variant of Fae).
//
// The doubles residual keeps the RCCD structure of cc.hip with
//   tau  = t2 + t1 t1    in the hole-hole and particle-particle ladders,
//   tau' = t2 + t1 t1/2  in Fae / Fmi,
//   WJ   = K + K (U - 2 tt^x)/2 - Kx T/2 + T1 terms,
//   WE   = -J + Kx (Tx + 2 tt^x)/2 + T1 terms + D/2, tt^x[ia,jb] = t1[ib] t1[ja],
//   D[kc,jb] = delta_kj Fae[b,c] - delta_cb Fmi[k,j] (the Fock-like terms, as in RCCD),
// Wabef's T1 terms become  -sum_m t1[mb] Z[ij,ma] + (ia<->jb)  with
// Z[ij,ma] = sum_ef tau[ij,ef] (mf|ae); the remaining T1 terms are small
// contractions done by the TTGT engine.  Integral labels below: occupied
// letters i j m n, virtual letters a b e f; ooov_c[i,j,k,a] = (ij|ka),
// ovvv_c[i,a,b,c] = (ia|bc).
//
// With AO factors the o v^3 block (ia|bc) = sum_P Lov[i,a,P] Lvv[b,c,P] is never stored
// (at o=80, v=420 it would be 47 GB in FP64, and each TTGT contraction with it a second
// permuted copy): every term that reads it contracts the factors instead, through the
// small intermediates B1[m,P,e] = Y2[m,e,P] = sum_f t1[m,f] Lvv[e,f,P] and
// Y3[m,j,P] = sum_f Lov[m,f,P] t1[j,f], and Z is built from slabs of (mf|ae) generated
// for a few m at a time (2 o v^3 naux flops per iteration).
#include "cc.h"

#include <algorithm>
#include <cstring>

namespace jues {
namespace {

// The amplitude layouts of the CCSD residual in the compute type, all from one read of t2 and t1:
//   Tpp = tau = t2 + t1 t1, Upp = 2 tau' - tau'^(ij) (tau' = t2 + t1 t1 / 2)          [i,j,a,b]
//   Tov = t2, Ttov[i,a,j,b] = t2[i,j,b,a], Uov = 2 t2 - t2^(ij)                        [i,a,j,b]
//   U2 = Uov - 2 tt^x, Q = Ttov + 2 tt^x with tt^x[i,a,j,b] = t1[i,b] t1[j,a]           [i,a,j,b]
template <typename T>
struct CcsdLayouts {
  int o, v;
  T *Tpp, *Upp, *Tov, *Ttov, *Uov, *U2, *Q;
  // element (i,j,a,b) from t2 = t2[ijab], t2x = t2[jiab]
  __device__ inline void put(const double* __restrict__ t1, int i, int j, int a, int b, double t2, double t2x) const {
    const long oo = (long)o * o, ov = (long)o * v, x = i + (long)o * j + oo * (a + (long)v * b);
    const double tt = t1[i + (long)o * a] * t1[j + (long)o * b], ttx = t1[i + (long)o * b] * t1[j + (long)o * a];
    const long y = i + (long)o * a + ov * (j + (long)o * b), yx = i + (long)o * b + ov * (j + (long)o * a);
    if (Tpp) Tpp[x] = (T)(t2 + tt);  // (the factored route takes the packed tau, and U for T)
    Upp[x] = (T)(2.0 * (t2 + 0.5 * tt) - (t2x + 0.5 * ttx));
    const T u = (T)(2.0 * t2 - t2x);
    if (Tov) Tov[y] = (T)t2;
    Uov[y] = u;
    U2[y] = (T)((double)u - 2.0 * (double)(T)ttx);
    Ttov[yx] = (T)t2;                                  // Ttov[i,b,j,a] = t2[i,j,a,b]
    Q[yx] = (T)((double)(T)t2 + 2.0 * (double)(T)tt);  // tt^x[i,b,j,a] = t1[i,a] t1[j,b]
  }
};

// One workgroup per (a,b) pair, whose o x o slab of t2 is staged in LDS (rows padded to o + 1) so that the
// exchanged read t2[j,i,a,b] comes from LDS: t2 is read once and each of the seven layouts written once, in
// runs of o.  Dynamic LDS: o (o + 1) doubles; without it (o too large) the exchanged element is read from memory.
// Bound by the writes; it replaces five launches that made 14 passes over o^2 v^2 elements between them, and the
// three passes that built U2 and Q later.
template <typename T>
__global__ __launch_bounds__(256) void ccsd_layouts_kernel(const double* __restrict__ t2, const double* __restrict__ t1,
                                                           CcsdLayouts<T> L, int staged) {
  extern __shared__ double slab[];
  const int o = L.o, oo = o * o, ld = o + 1;
  const long vv = (long)L.v * L.v;
  for (long ab = blockIdx.x; ab < vv; ab += gridDim.x) {
    const int a = (int)(ab % L.v), b = (int)(ab / L.v);
    const double* src = t2 + ab * oo;
    if (staged) {
      __syncthreads();  // the previous pair's readers are done with the slab
      for (int q = threadIdx.x; q < oo; q += 256) slab[q % o + ld * (q / o)] = src[q];
      __syncthreads();
    }
    for (int q = threadIdx.x; q < oo; q += 256) {
      const int i = q % o, j = q / o;
      L.put(t1, i, j, a, b, staged ? slab[i + ld * j] : src[q], staged ? slab[j + ld * i] : src[j + (long)o * i]);
    }
  }
}

// n1[i,a] += 2 sum_m KT[i,a,m,m] - sum_m JT[m,a,i,m] (KT o x v x o x o, JT o x v x o x o): takes the place of two products
// of t1 with all of (ia|me) and (mi|ae), and of a permuted copy of the latter, 60 us at ov = 2000
template <typename T>
__global__ __launch_bounds__(256) void singles_trace_kernel(const T* __restrict__ KT, const T* __restrict__ JT, int o,
                                                            int v, T* __restrict__ n1) {
  const int x = blockIdx.x * 256 + threadIdx.x;
  if (x >= o * v) return;
  const long ov = (long)o * v, i = x % o, a = x / o;
  double s = 0.0;
  for (int m = 0; m < o; ++m)
    s += 2.0 * (double)KT[x + ov * m + ov * o * m] - (double)JT[m + o * a + ov * i + ov * o * m];
  n1[x] = (T)((double)n1[x] + s);
}

// per (a,b): sum_ij Lener[i,j,a,b] t1[i,a] t1[j,b]
__global__ __launch_bounds__(256) void energy_t1_kernel(const double* __restrict__ Lener, const double* __restrict__ t1,
                                                        int o, int v, double* __restrict__ part) {
  __shared__ double sh[4];
  const long oo = (long)o * o;
  const int ab = blockIdx.x, a = ab % v, b = ab / v;
  const double* L = Lener + oo * ab;
  double s = 0.0;
  for (long ij = threadIdx.x; ij < oo; ij += 256) {
    const int i = (int)(ij % o), j = (int)(ij / o);
    s += L[ij] * t1[i + (long)o * a] * t1[j + (long)o * b];
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[ab] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

__global__ __launch_bounds__(256) void sum_parts_kernel(const double* __restrict__ part, long count,
                                                        double* __restrict__ out) {
  __shared__ double sh[256];
  double s = 0.0;
  for (long i = threadIdx.x; i < count; i += 256) s += part[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = sh[0];
}

int g256(long n) { return (int)std::max(1L, std::min((n + 255) / 256, 131072L)); }

}  // namespace

void cc_build_ccsd_ints(jues_ctx* ctx, CCState& S) {
  const long N1 = (long)S.o * S.v;
  S.R1.alloc(N1 * sizeof(double));
  (void)ctx;
}

double cc_energy_t1(jues_ctx* ctx, CCState& S) {
  // sum_ijab Lener[ijab] t1[ia] t1[jb], fixed-order partials per (a,b)
  const int o = S.o, v = S.v;
  const long N2 = (long)o * o * v * v, vv = (long)v * v;
  const double* t1 = S.t.as<double>() + N2;
  double* part = static_cast<double*>(scratch(ctx, 7, sizeof(double) * (size_t)(vv + 1)));
  hipLaunchKernelGGL(energy_t1_kernel, dim3((unsigned)vv), dim3(256), 0, ctx->stream, S.Lener.as<double>(), t1, o, v,
                     part);
  hipLaunchKernelGGL(sum_parts_kernel, dim3(1), dim3(256), 0, ctx->stream, part, vv, part + vv);
  JUES_HIP(hipGetLastError());
  double E = 0.0;
  d2h(ctx, &E, part + vv, sizeof(double));
  return E;
}

template <typename T>
void rccsd_contractions(jues_ctx* ctx, CCState& S, const double* t2, const double* t1_64) {
  const int o = S.o, v = S.v;
  const long ov = (long)o * v, N2 = ov * ov, oo = (long)o * o, vv = (long)v * v;
  CCInts<T>& I = ints<T>(S);
  CCWork<T>& W = work<T>(S);
  const std::vector<long> d4 = {o, o, v, v};
  auto TN = [&](const void* p, const char* idx) {
    Tens<T> x;
    x.p = const_cast<T*>(static_cast<const T*>(p));
    x.idx = idx;
    for (const char* c = idx; *c; ++c) x.dims.push_back(std::strchr("ijmn", *c) ? (long)o : (long)v);
    return x;
  };
  const bool fac = S.ovvv_factored;
  T* Tpp = bufp_t<T>(W.Tpp, N2);   // tau
  T* Upp = bufp_t<T>(W.Upp, N2);   // 2 tau' - tau'^(ij)
  T* Tov = fac ? nullptr : bufp_t<T>(W.Tov, N2);   // t2 [i,a,j,b]
  T* Ttov = bufp_t<T>(W.Ttov, N2); // t2[i,j,b,a] at [i,a,j,b]
  T* Uov = bufp_t<T>(W.Uov, N2);   // 2 t2 - t2^x (ov)
  T* Ua = bufp_t<T>(W.Ua, N2);
  // WJ and WE are built after Upp and Ua are last read (Fmi, Fae), Y after Tpp (Z): with
  // factored (ia|bc) they share those buffers
  T* WJ = fac ? Upp : bufp_t<T>(W.WJ, N2);
  T* WE = fac ? Ua : bufp_t<T>(W.WE, N2);
  T* Y = fac ? Tpp : bufp_t<T>(W.Y, N2);
  T* H = bufp_t<T>(W.H, N2);
  T* Wp = bufp_t<T>(W.Wp, oo * oo);
  T* Fae = bufp_t<T>(W.Fae, vv);
  T* Fmi = bufp_t<T>(W.Fmi, oo);
  T* Fme = bufp_t<T>(W.Fme, ov);
  T* t1 = bufp_t<T>(W.t1, ov);
  T* n1 = bufp_t<T>(W.n1, ov);
  T* X2 = bufp_t<T>(W.X2, N2);
  T* U2 = bufp_t<T>(W.U2, N2);
  T* Q = bufp_t<T>(W.Q, std::max(N2, oo * ov));
  T* Z = bufp_t<T>(W.Z, oo * ov);
  T* KT = bufp_t<T>(W.KT, oo * ov);
  T* JT = bufp_t<T>(W.JT, oo * ov);
  T* Tp = bufp_t<T>(W.Tp, S.P.npo * S.P.npv);
  T* Tm = bufp_t<T>(W.Tm, std::max(1L, S.P.nmo * S.P.nmv));
  T* Lp = bufp_t<T>(W.Lp, S.P.npo * S.P.npv);
  T* Lm = bufp_t<T>(W.Lm, std::max(1L, S.P.nmo * S.P.nmv));
  const T one = T(1), zero = T(0), half = T(0.5);
  const bool mrccsd = S.opts.ccsd_eqs == JUES_CCSD_MRCCSD;
  const long naux = ctx->naux;

  // ---- amplitudes in the compute type -------------------------------------------
  convert<double, T>(ctx, t1_64, t1, ov);
  {
    const size_t slab = (size_t)o * (o + 1) * sizeof(double);
    const bool staged = slab <= 65536;
    KTimer k(ctx, "cc_prep", 0.0, (double)N2 * ((staged ? 8.0 : 16.0) + (fac ? 5.0 : 7.0) * sizeof(T)));
    hipLaunchKernelGGL((ccsd_layouts_kernel<T>), dim3((unsigned)std::min(vv, 1L << 20)), dim3(256),
                       staged ? slab : 0, ctx->stream, t2, t1_64,
                       CcsdLayouts<T>{o, v, fac ? nullptr : Tpp, Upp, Tov, Ttov, Uov, U2, Q},
                       staged ? 1 : 0);
    JUES_HIP(hipGetLastError());
  }
  permute<T, T>(ctx, Upp, d4, {2, 0, 1, 3}, Ua, 1.0, 0.0, "cc_prep");

  // factors of (ia|bc) and their contractions with t1
  const T* Lov = fac ? I.Lov.template as<T>() : nullptr;    // [m,e,P]
  const T* LovT = fac ? I.LovT.template as<T>() : nullptr;  // [e,m,P]
  const T* Lovp = fac ? I.Lovp.template as<T>() : nullptr;  // [m,P,e]
  const T* Lvv = fac ? I.Lvv.template as<T>() : nullptr;    // [a,e,P]
  T *B1 = nullptr, *Y2 = nullptr, *Y3 = nullptr;
  if (fac) {
    B1 = bufp_t<T>(W.B1, ov * naux);
    Y2 = bufp_t<T>(W.Y2, ov * naux);
    Y3 = bufp_t<T>(W.Y3, oo * naux);
    // B1[m,P,e] = Y2[m,e,P] = sum_f t1[m,f] Lvv[e,f,P] (batched over P; B1's rows interleave
    // the batches through ldc = o naux), Y3[m,j,P] = sum_f Lov[m,f,P] t1[j,f]
    gemm<T>(ctx, false, true, o, v, v, one, t1, o, 0, Lvv, v, vv, zero, B1, o * naux, o, (int)naux, "cc_ovvv_fac");
    gemm<T>(ctx, false, true, o, v, v, one, t1, o, 0, Lvv, v, vv, zero, Y2, o, ov, (int)naux, "cc_ovvv_fac");
    gemm<T>(ctx, false, true, o, o, v, one, Lov, o, ov, t1, o, 0, zero, Y3, o, oo, (int)naux, "cc_ovvv_fac");
  }

  // ---- Fae, Fmi, Fme --------------------------------------------------------------
  gemm<T>(ctx, false, true, v, v, oo * v, T(-1), Ua, v, 0, I.Ka.template as<T>(), v, 0, zero, Fae, v, 0, 1, "cc_fock");
  gemm<T>(ctx, false, true, o, o, ov * v, one, I.Kpp.template as<T>(), o, 0, Upp, o, 0, zero, Fmi, o, 0, 1, "cc_fock");
  const T* ovvv = I.ovvv_c.template as<T>();
  const T* ooov = I.ooov_c.template as<T>();
  const T* Kov = I.Kov.template as<T>();
  const T* Jov = I.Jov.template as<T>();
  // Fae[a,e] += sum_mf t1[mf] (2(mf|ae) - X),  X = (ma|ef) (mRCCSD.jl:140) or (me|af) (RCCSD.jl:189)
  if (fac) {
    // 2 sum_mf t1[mf] (mf|ae) = 2 sum_P g[P] Lvv[(ae),P] with g[P] = sum_(mf) t1[(mf)] Lov[(mf),P];
    // (ma|ef) term: sum_(mP) Lovp[(mP),a] B1[(mP),e]; (me|af) term: sum_(mP) B1[(mP),a] Lovp[(mP),e]
    T* g = bufp_t<T>(W.gP, naux);
    gemm<T>(ctx, true, false, naux, 1, ov, one, Lov, ov, 0, t1, ov, 0, zero, g, naux, 0, 1, "cc_ovvv_fac");
    gemm<T>(ctx, false, false, vv, 1, naux, T(2), Lvv, vv, 0, g, naux, 0, one, Fae, vv, 0, 1, "cc_ovvv_fac");
    gemm<T>(ctx, true, false, v, v, o * naux, T(-1), mrccsd ? Lovp : B1, o * naux, 0, mrccsd ? B1 : Lovp, o * naux, 0,
            one, Fae, v, 0, 1, "cc_ovvv_fac");
  } else {
    contract<T>(ctx, 2.0, TN(t1, "mf"), TN(ovvv, "mfae"), 1.0, TN(Fae, "ae"), "cc_t1");
    contract<T>(ctx, -1.0, TN(t1, "mf"), TN(ovvv, mrccsd ? "maef" : "meaf"), 1.0, TN(Fae, "ae"), "cc_t1");
  }
  // Fmi[m,i] += sum_ne t1[ne] (2(mi|ne) - (ni|me))
  contract<T>(ctx, 2.0, TN(t1, "ne"), TN(ooov, "mine"), 1.0, TN(Fmi, "mi"), "cc_t1");
  contract<T>(ctx, -1.0, TN(t1, "ne"), TN(ooov, "nime"), 1.0, TN(Fmi, "mi"), "cc_t1");
  // Fme[m,e] = sum_nf t1[nf] (2(me|nf) - (ne|mf)), (ne|mf) = (mf|ne) = Kx[m,e,n,f]: 2 Lx t1
  const T* Kx = I.Ktov.template as<T>();
  contract<T>(ctx, 2.0, TN(t1, "nf"), TN(ring_lx<T>(ctx, S), "menf"), 0.0, TN(Fme, "me"), "cc_t1");

  // ---- off-diagonal Fock terms of a non-canonical reference (AutoRCCSD.jl:76-81,127-132):
  // Fae += f_ae - t1[ma] f_me / 2, Fmi += f_mi + t1[ie] f_me / 2, Fme += f_me
  if (S.fock_on) {
    const T* fOO = I.fOO.template as<T>();
    const T* fVV = I.fVV.template as<T>();
    const T* fOV = I.fOV.template as<T>();
    axpby<T>(ctx, vv, 1.0, fVV, 1.0, Fae);
    contract<T>(ctx, -0.5, TN(t1, "ma"), TN(fOV, "me"), 1.0, TN(Fae, "ae"), "cc_fock_t1");
    axpby<T>(ctx, oo, 1.0, fOO, 1.0, Fmi);
    contract<T>(ctx, 0.5, TN(t1, "ie"), TN(fOV, "me"), 1.0, TN(Fmi, "mi"), "cc_fock_t1");
    axpby<T>(ctx, ov, 1.0, fOV, 1.0, Fme);
  }

  // ---- T1 residual (mRCCSD.jl:202-212) ----------------------------------------------
  contract<T>(ctx, 1.0, TN(t1, "ie"), TN(Fae, "ae"), 0.0, TN(n1, "ia"), "cc_t1");
  contract<T>(ctx, -1.0, TN(t1, "ma"), TN(Fmi, "mi"), 1.0, TN(n1, "ia"), "cc_t1");
  contract<T>(ctx, 1.0, TN(Fme, "me"), TN(Uov, "iame"), 1.0, TN(n1, "ia"), "cc_t1");
  // t1[ie] (jb|me) at [j,b,m,i] and t1[je] (mi|be) at [m,b,i,j], which the ring's T1^2 terms take too; their traces over
  // the two m are the terms 2 t1[me] (ia|me) - t1[me] (mi|ae)
  contract<T>(ctx, 1.0, TN(t1, "ie"), TN(Kov, "jbme"), 0.0, TN(KT, "jbmi"), "cc_t1");
  contract<T>(ctx, 1.0, TN(t1, "je"), TN(Jov, "mbie"), 0.0, TN(JT, "mbij"), "cc_t1");
  {
    KTimer k(ctx, "cc_t1", 0.0, 2.0 * oo * v * sizeof(T));
    hipLaunchKernelGGL((singles_trace_kernel<T>), dim3((unsigned)((ov + 255) / 256)), dim3(256), 0, ctx->stream, KT, JT,
                       o, v, n1);
    JUES_HIP(hipGetLastError());
  }
  // -sum_nme (2 T[ne,ma] - T[me,na]) (mi|ne) = -sum U[ne,ma] (mi|ne)
  contract<T>(ctx, -1.0, TN(Uov, "nema"), TN(ooov, "mine"), 1.0, TN(n1, "ia"), "cc_t1");
  if (fac) {
    // sum_emf (2 T[ie,mf] - T[me,if]) (mf|ae) = sum_(eP) W1[i,(eP)] Lvv[a,(eP)] with
    // W1[(ie),P] = sum_(mf) U[(ie),(mf)] Lov[(mf),P], U = 2 T - T^x: both terms in one (ov)^2 naux product
    T* W1 = bufp_t<T>(W.W1, ov * naux);
    fac_uov_lov<T>(ctx, S, Uov, W1);
    gemm<T>(ctx, false, true, o, v, v * naux, one, W1, o, 0, Lvv, v, 0, one, n1, o, 0, 1, "cc_ovvv_fac");
  } else {
    contract<T>(ctx, 2.0, TN(Tov, "iemf"), TN(ovvv, "mfae"), 1.0, TN(n1, "ia"), "cc_t1");
    contract<T>(ctx, -1.0, TN(Tov, "iemf"), TN(ovvv, "meaf"), 1.0, TN(n1, "ia"), "cc_t1");
  }
  if (S.fock_on) axpby<T>(ctx, ov, 1.0, I.fOV.template as<T>(), 1.0, n1);  // f_ia
  convert<T, double>(ctx, n1, S.R1.as<double>(), ov);

  // ---- Fb = Fae - t1.Fme/2, Fj = Fmi + t1.Fme/2 ------------------------------------
  contract<T>(ctx, -0.5, TN(t1, "mb"), TN(Fme, "me"), 1.0, TN(Fae, "be"), "cc_t1");
  contract<T>(ctx, 0.5, TN(t1, "je"), TN(Fme, "me"), 1.0, TN(Fmi, "mj"), "cc_t1");

  // ---- particle-particle ladder on tau = t2 + t1 t1 (packed on the fly) ----------------
  ladder_mm<T>(ctx, S, t2, Tp, Tm, Lp, Lm, t1_64);
  // ---- hole-hole ladder: W' = oooo + T1 terms + <mn|ef> tau[ij,ef], added into Lp / Lm ----
  JUES_HIP(hipMemcpyAsync(Wp, I.oooo.p, oo * oo * sizeof(T), hipMemcpyDeviceToDevice, ctx->stream));
  contract<T>(ctx, 1.0, TN(t1, "je"), TN(ooov, "mine"), 1.0, TN(Wp, "mnij"), "cc_t1");
  contract<T>(ctx, 1.0, TN(t1, "ie"), TN(ooov, "njme"), 1.0, TN(Wp, "mnij"), "cc_t1");
  hh_mm<T>(ctx, S, Wp, Tp, Tm, Lp, Lm);
  // Wabef's T1 part: X2 = Lz[ijab] = -sum_m t1[mb] Z[ij,ma],  Z = tau . (mf|ae); the update kernel adds
  // Lz[ijab] + Lz[jiba]
  if (fac) {
    // Z[i,j,a,m] on the packed pairs of tau over slabs of m, then Lz[(ija),b] = -sum_m Z[(ija),m] t1[m,b]
    const long per_m = (long)v * vv;
    const long ms = std::max(1L, std::min<long>(o, (2L << 30) / (per_m * (long)sizeof(T))));
    T* Zs = bufp_t<T>(W.Zs, (size_t)(ms * per_m));
    T* Zsp = bufp_t<T>(W.Zsp, (size_t)(ms * per_m));
    T* Zp = bufp_t<T>(W.Zpm, (size_t)(oo * ov));
    T* Zm = Zp + S.P.npo * ov;
    for (int m0 = 0; m0 < o; m0 += (int)ms) {
      const int cnt = (int)std::min<long>(ms, o - m0);
      ovvv_z_slab<T>(ctx, S, m0, cnt, LovT, Lvv, Tp, Tm, Zs, Zsp, Zp, Zm);
    }
    // (without pairs e < f the products leave Zm unwritten)
    unpack_z<T>(ctx, S.P, Zp, S.P.nmv > 0 ? Zm : nullptr, o, v, Z);
    gemm<T>(ctx, false, false, oo * v, v, o, T(-1), Z, oo * v, 0, t1, o, 0, zero, X2, oo * v, 0, 1, "cc_t1");
  } else {
    contract<T>(ctx, 1.0, TN(Tpp, "ijef"), TN(ovvv, "mfae"), 0.0, TN(Z, "ijma"), "cc_ovvv");
    contract<T>(ctx, -1.0, TN(t1, "mb"), TN(Z, "ijma"), 0.0, TN(X2, "ijab"), "cc_t1");
  }

  // ---- ring terms -----------------------------------------------------------------------
  // (as in RCCD, with U2 = 2 T - Q: W = WJ + WE/2 = K - J/2 + (K - Kx/2) U2/2 and the T1 terms of WJ and half of
  // WE's, H = U W + Y/2; every left operand of the ring products is a symmetric (ov) x (ov) matrix)
  permute<T, T>(ctx, Jov, {ov, ov}, {0, 1}, WE, -1.0, 0.0, "cc_prep");
  // WE[me,jb] += sum_n t1[nb] (mj|ne) - sum_f t1[jf] (mf|be).  With factors both are products over [(mj),(be)], the
  // second sum_P Y3[(mj),P] Lvv[(be),P], formed in H (free until the ring products) and permuted into WE at once
  if (fac) {
    fac_y3_lvv<T>(ctx, S, Y3, H);
    gemm<T>(ctx, false, false, oo, v, o, T(-1), ooov, oo, oo * o, t1, o, 0, one, H, oo, oo * v, v, "cc_t1");
    permute<T, T>(ctx, H, d4, {0, 3, 1, 2}, WE, -1.0, 1.0, "cc_ovvv_fac");
  } else {
    contract<T>(ctx, -1.0, TN(t1, "jf"), TN(ovvv, "mfbe"), 1.0, TN(WE, "mejb"), "cc_t1");
    contract<T>(ctx, 1.0, TN(t1, "nb"), TN(ooov, "mjne"), 1.0, TN(WE, "mejb"), "cc_t1", H, N2);
  }
  // Fock-like terms with Fb / Fj, carried by WE as in RCCD: WE += D/2 with
  // D[kc,jb] = delta_kj Fb[b,c] - delta_cb Fj[k,j]
  T* FmiT = bufp_t<T>(W.FmiT, oo);
  permute<T, T>(ctx, Fmi, {o, o}, {1, 0}, FmiT, 1.0, 0.0, "cc_fock");
  // A = sum_f t1[jf] (me|bf) at [me,jb] is one of WJ's T1 terms, and H's term t1[ie] (jb|ae) is its transpose, which
  // S = G + G^T cannot tell from A: formed once, in H
  if (fac) fac_lov_y2<T>(ctx, S, Y2, H);
  else contract<T>(ctx, 1.0, TN(t1, "jf"), TN(ovvv, "mebf"), 0.0, TN(H, "mejb"), "cc_t1");
  ring_start<T>(ctx, Kov, one, WE, Fae, FmiT, o, v, WE, WJ, H);
  // WJ's other T1 term, through Y (free until Tx WE)
  contract<T>(ctx, -1.0, TN(t1, "nb"), TN(ooov, "njme"), 1.0, TN(WJ, "mejb"), "cc_t1", Y, N2);
  ring_mm<T>(ctx, S, half, ring_lx<T>(ctx, S), SP_LX, U2, SP_U2, one, WJ);
  ring_mm<T>(ctx, S, half, Kx, SP_KX, Q, SP_Q, one, WE);
  ring_mm<T>(ctx, S, one, Uov, SP_UOV, WJ, SP_WJ, one, H);
  // exchange ring term t[m,i,b,e] WmBEj[m,a,e,j] = (Tx WE)[ib,ja], and half the direct one
  ring_mm<T>(ctx, S, one, Ttov, SP_TTOV, WE, SP_WE, zero, Y);
  // T1^2 terms -t1[ie] t1[ma] (me|jb) and -t1[ie] t1[mb] (mj|ae), T1-linear term -t1[ma] (mi|jb): with the second
  // transposed (S = G + G^T) all are -t1[ma] Q[mi,jb], Q = (mi|jb) + t1[ie] (me|jb) + t1[je] (mi|be); the
  // product permuted into H goes through U2, free once WJ is built
  JUES_HIP(hipMemcpyAsync(Q, ooov, (size_t)(oo * ov) * sizeof(T), hipMemcpyDeviceToDevice, ctx->stream));
  permute<T, T>(ctx, KT, {o, v, o, o}, {2, 3, 0, 1}, Q, 1.0, 1.0, "cc_t1");
  permute<T, T>(ctx, JT, {o, v, o, o}, {0, 2, 3, 1}, Q, 1.0, 1.0, "cc_t1");
  contract<T>(ctx, -1.0, TN(t1, "ma"), TN(Q, "mijb"), 1.0, TN(H, "iajb"), "cc_t1", U2, N2);
  // S = G + G^T, G = H + Y/2 + Y^x: summed by the update kernel, or here (into WJ) when its LDS slab
  // would not fit
  if (!fused_sym(o, sizeof(T))) {
    axpby<T>(ctx, N2, 0.5, Y, 1.0, H);
    permute<T, T>(ctx, Y, {o, v, o, v}, {0, 3, 2, 1}, H, 1.0, 1.0, "cc_sym");
    JUES_HIP(hipMemcpyAsync(WJ, H, N2 * sizeof(T), hipMemcpyDeviceToDevice, ctx->stream));
    permute<T, T>(ctx, H, {ov, ov}, {1, 0}, WJ, 1.0, 1.0, "cc_sym");
  }
  W.y_direct = 0.5;
  W.out_H = H;
  W.out_Y = Y;
  W.out_S = WJ;
  W.out_X = X2;
}

template void rccsd_contractions<double>(jues_ctx*, CCState&, const double*, const double*);
template void rccsd_contractions<float>(jues_ctx*, CCState&, const double*, const double*);

}  // namespace jues
