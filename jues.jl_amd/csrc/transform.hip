// AO -> MO four-index transformation (Backend/Transformation.jl:39-93) and the
// RMP2 energy reduction (MollerPlesset/RMP2.jl:27-41).
//
// Dense route: four quarter transforms, each one MFMA GEMM (plain or batched)
// over the full AO tensor.  The outer index (mu or sigma) with the smaller target
// dimension is contracted first.  If the inner index next to the other outer one
// has a smaller target than it (lambda for mu first, as d3 = o < d4 = v in
// (ia|jb)), that inner index is contracted second, batched, which makes the
// second quarter 2 n^3 d1 d3 instead of 2 n^3 d1 d4; otherwise the other outer
// index is, and the last two quarters contract nu and lambda in place (the
// smaller of d2, d3 first).  Every order writes the result in [p, q, r, s]
// order from its last GEMM, with no permutation pass.  Factor route:
// (pq|rs) = sum_P (C1^T B_P C2)_pq (C3^T B_P C4)_rs, two batched GEMMs per side
// and one GEMM over P; the n^4 AO tensor is never formed.
#include "jues_internal.h"

#include <algorithm>

namespace jues {

template <>
const double* ao_dense<double>(jues_ctx* ctx) {
  JUES_REQUIRE(ctx->gao.p, "no dense AO integrals set");
  return ctx->gao.as<double>();
}
template <>
const float* ao_dense<float>(jues_ctx* ctx) {
  JUES_REQUIRE(ctx->gao.p, "no dense AO integrals set");
  if (!ctx->gao32.p) {
    const long nn = (long)ctx->n * ctx->n * ctx->n * ctx->n;
    ctx->gao32.alloc(sizeof(float) * nn);
    convert<double, float>(ctx, ctx->gao.as<double>(), ctx->gao32.as<float>(), nn);
  }
  return ctx->gao32.as<float>();
}
template <>
const double* ao_factors<double>(jues_ctx* ctx) {
  JUES_REQUIRE(ctx->Bfac.p, "no AO factors set");
  return ctx->Bfac.as<double>();
}
template <>
const float* ao_factors<float>(jues_ctx* ctx) {
  JUES_REQUIRE(ctx->Bfac.p, "no AO factors set");
  if (!ctx->Bfac32.p) {
    const long nn = (long)ctx->n * ctx->n * ctx->naux;
    ctx->Bfac32.alloc(sizeof(float) * nn);
    convert<double, float>(ctx, ctx->Bfac.as<double>(), ctx->Bfac32.as<float>(), nn);
  }
  return ctx->Bfac32.as<float>();
}

template <typename T>
void mo_factors_dev(jues_ctx* ctx, const T* C1, int d1, const T* C2, int d2, T* L) {
  const long n = ctx->n, naux = ctx->naux;
  T* Y = static_cast<T*>(scratch(ctx, 4, sizeof(T) * (size_t)(n * std::min(d1, d2) * naux)));
  mo_factors_dev<T>(ctx, C1, d1, C2, d2, L, Y);
}

template <typename T>
void mo_factors_dev(jues_ctx* ctx, const T* C1, int d1, const T* C2, int d2, T* L, T* Y) {
  const long n = ctx->n, naux = ctx->naux;
  const T* B = ao_factors<T>(ctx);
  // The smaller of d1, d2 is contracted first: 2 n^2 min(d1,d2) naux + 2 n d1 d2 naux flops.
  if (d1 <= d2) {
    // Y[nu, p, P] = B_P^T C1 ; L[p, q, P] = Y_P^T C2
    gemm<T>(ctx, true, false, n, d1, n, T(1), B, n, n * n, C1, n, 0, T(0), Y, n, n * d1, (int)naux,
            "xform_factor");
    gemm<T>(ctx, true, false, d1, d2, n, T(1), Y, n, n * d1, C2, n, 0, T(0), L, d1, (long)d1 * d2, (int)naux,
            "xform_factor");
  } else {
    // Y[mu, q, P] = B_P C2 ; L[p, q, P] = C1^T Y_P
    gemm<T>(ctx, false, false, n, d2, n, T(1), B, n, n * n, C2, n, 0, T(0), Y, n, n * d2, (int)naux,
            "xform_factor");
    gemm<T>(ctx, true, false, d1, d2, n, T(1), C1, n, 0, Y, n, n * d2, T(0), L, d1, (long)d1 * d2, (int)naux,
            "xform_factor");
  }
}

template <typename T>
void tei_transform_dev(jues_ctx* ctx, const T* C1, int d1, const T* C2, int d2, const T* C3, int d3,
                       const T* C4, int d4, T* out) {
  const long n = ctx->n;
  JUES_REQUIRE(n > 0, "no AO integrals set");
  if (ctx->gao.p) {
    const T* G = ao_dense<T>(ctx);
    const long n2 = n * n, n3 = n2 * n;
    const long d12 = (long)d1 * d2;
    if (d1 <= d4 && d3 < d4) {
      // mu first, then lam (a smaller target than sig's), batched over sig: the second quarter
      // costs 2 n^3 d1 d3 instead of 2 n^3 d1 d4, and each product writes its result in the
      // order the next one reads
      //   X1[p, (nu,lam,sig)] = sum_mu C1[mu, p] g[mu, (nu,lam,sig)]
      //   X2[(p,nu), r, sig]  = sum_lam X1[(p,nu), lam, sig] C3[lam, r]   (batched over sig)
      //   X3[(p,nu,r), s]     = sum_sig X2[(p,nu,r), sig] C4[sig, s]
      //   out[p, q, (r,s)]    = sum_nu X3[p, nu, (r,s)] C2[nu, q]        (batched over (r,s))
      const long pn = (long)d1 * n, pnr = pn * d3;
      T* X1 = static_cast<T*>(scratch(ctx, 0, sizeof(T) * (size_t)(d1 * n3)));
      gemm<T>(ctx, true, false, d1, n3, n, T(1), C1, n, 0, G, n, 0, T(0), X1, d1, 0, 1, "xform_q1");
      T* X2 = static_cast<T*>(scratch(ctx, 1, sizeof(T) * (size_t)(pnr * n)));
      gemm<T>(ctx, false, false, pn, d3, n, T(1), X1, pn, pn * n, C3, n, 0, T(0), X2, pn, pnr, (int)n, "xform_q2");
      T* X3 = static_cast<T*>(scratch(ctx, 2, sizeof(T) * (size_t)(pnr * d4)));
      gemm<T>(ctx, false, false, pnr, d4, n, T(1), X2, pnr, 0, C4, n, 0, T(0), X3, pnr, 0, 1, "xform_q3");
      gemm<T>(ctx, false, false, d1, d2, n, T(1), X3, d1, pn, C2, n, 0, T(0), out, d1, d12, d3 * d4, "xform_q4");
    } else if (d1 > d4 && d2 < d1) {
      // the mirror image: sig first, then nu (a smaller target than mu's), batched over (lam,s)
      //   Y1[(mu,nu,lam), s] = sum_sig g[(mu,nu,lam), sig] C4[sig, s]
      //   Y2[mu, q, (lam,s)] = sum_nu Y1[mu, nu, (lam,s)] C2[nu, q]      (batched over (lam,s))
      //   X3[p, (q,lam,s)]   = sum_mu C1[mu, p] Y2[mu, (q,lam,s)]
      //   out[(p,q), r, s]   = sum_lam X3[(p,q), lam, s] C3[lam, r]      (batched over s)
      T* Y1 = static_cast<T*>(scratch(ctx, 0, sizeof(T) * (size_t)(n3 * d4)));
      gemm<T>(ctx, false, false, n3, d4, n, T(1), G, n3, 0, C4, n, 0, T(0), Y1, n3, 0, 1, "xform_q1");
      T* Y2 = static_cast<T*>(scratch(ctx, 1, sizeof(T) * (size_t)(n * d2 * n * d4)));
      gemm<T>(ctx, false, false, n, d2, n, T(1), Y1, n, n2, C2, n, 0, T(0), Y2, n, n * d2, (int)(n * d4), "xform_q2");
      T* X3 = static_cast<T*>(scratch(ctx, 2, sizeof(T) * (size_t)(d12 * n * d4)));
      gemm<T>(ctx, true, false, d1, d2 * n * d4, n, T(1), C1, n, 0, Y2, n, 0, T(0), X3, d1, 0, 1, "xform_q3");
      gemm<T>(ctx, false, false, d12, d3, n, T(1), X3, d12, d12 * n, C3, n, 0, T(0), out, d12, d12 * d3, d4,
              "xform_q4");
    } else {
      // the two outer indices first (the one with the smaller target first), to X2[p, nu, lam, s]
      T* X2 = static_cast<T*>(scratch(ctx, 1, sizeof(T) * (size_t)(d1 * n2 * d4)));
      if (d1 <= d4) {
        T* X1 = static_cast<T*>(scratch(ctx, 0, sizeof(T) * (size_t)(d1 * n3)));
        gemm<T>(ctx, true, false, d1, n3, n, T(1), C1, n, 0, G, n, 0, T(0), X1, d1, 0, 1, "xform_q1");
        gemm<T>(ctx, false, false, d1 * n2, d4, n, T(1), X1, d1 * n2, 0, C4, n, 0, T(0), X2, d1 * n2, 0, 1,
                "xform_q2");
      } else {
        T* Y1 = static_cast<T*>(scratch(ctx, 0, sizeof(T) * (size_t)(n3 * d4)));
        gemm<T>(ctx, false, false, n3, d4, n, T(1), G, n3, 0, C4, n, 0, T(0), Y1, n3, 0, 1, "xform_q1");
        gemm<T>(ctx, true, false, d1, n2 * d4, n, T(1), C1, n, 0, Y1, n, 0, T(0), X2, d1, 0, 1, "xform_q2");
      }
      // then nu and lam where they lie, as batched products, so that the result is written in
      // [p, q, r, s] order with no permutation pass
      if (d3 <= d2) {
        // X3[(p,nu), r, s] = sum_lam X2[(p,nu), lam, s] C3[lam, r]      (batched over s)
        // out[p, q, (r,s)] = sum_nu X3[p, nu, (r,s)] C2[nu, q]         (batched over (r,s))
        T* X3 = static_cast<T*>(scratch(ctx, 2, sizeof(T) * (size_t)((long)d1 * n * d3 * d4)));
        gemm<T>(ctx, false, false, (long)d1 * n, d3, n, T(1), X2, (long)d1 * n, (long)d1 * n2, C3, n, 0, T(0), X3,
                (long)d1 * n, (long)d1 * n * d3, d4, "xform_q3");
        gemm<T>(ctx, false, false, d1, d2, n, T(1), X3, d1, (long)d1 * n, C2, n, 0, T(0), out, d1, d12, d3 * d4,
                "xform_q4");
      } else {
        // X3[p, q, (lam,s)] = sum_nu X2[p, nu, (lam,s)] C2[nu, q]      (batched over (lam,s))
        // out[(p,q), r, s] = sum_lam X3[(p,q), lam, s] C3[lam, r]      (batched over s)
        T* X3 = static_cast<T*>(scratch(ctx, 2, sizeof(T) * (size_t)(d12 * n * d4)));
        gemm<T>(ctx, false, false, d1, d2, n, T(1), X2, d1, (long)d1 * n, C2, n, 0, T(0), X3, d1, d12,
                (int)(n * d4), "xform_q3");
        gemm<T>(ctx, false, false, d12, d3, n, T(1), X3, d12, d12 * n, C3, n, 0, T(0), out, d12, d12 * d3, d4,
                "xform_q4");
      }
    }
  } else {
    const long naux = ctx->naux;
    JUES_REQUIRE(ctx->Bfac.p, "no AO integrals set");
    T* L = static_cast<T*>(scratch(ctx, 5, sizeof(T) * (size_t)((long)d1 * d2 * naux)));
    mo_factors_dev<T>(ctx, C1, d1, C2, d2, L);
    T* R = L;  // (pq|pq)-shaped blocks such as (ia|jb): both sides are the same factors
    if (C1 != C3 || C2 != C4 || d1 != d3 || d2 != d4) {
      R = static_cast<T*>(scratch(ctx, 6, sizeof(T) * (size_t)((long)d3 * d4 * naux)));
      mo_factors_dev<T>(ctx, C3, d3, C4, d4, R);
    }
    const long m = (long)d1 * d2, nn = (long)d3 * d4;
    gemm<T>(ctx, false, true, m, nn, naux, T(1), L, m, 0, R, nn, 0, T(0), out, m, 0, 1, "xform_factor_gemm");
  }
}

namespace {

// One block per (j,b) column of K[i,a,j,b]; each thread walks (i,a) with stride 256.
template <typename T>
__global__ __launch_bounds__(256) void mp2_energy_kernel(const T* __restrict__ K, const double* __restrict__ eps,
                                                         int o, int v, double* __restrict__ part) {
  __shared__ double sh[4];
  const int ov = o * v;
  const int jb = blockIdx.x;
  const int j = jb % o, b = jb / o;
  const double ejb = eps[j] - eps[o + b];
  const long col = (long)jb * ov;
  double s = 0.0;
  for (int ia = threadIdx.x; ia < ov; ia += 256) {
    const int i = ia % o, a = ia / o;
    const double k = (double)K[col + ia];
    const double kx = (double)K[(long)(i + o * b) + (long)ov * (j + o * a)];  // (ib|ja)
    s += k * (2.0 * k - kx) / (eps[i] - eps[o + a] + ejb);
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[jb] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

__global__ __launch_bounds__(256) void sum_fixed_kernel(const double* __restrict__ part, int count,
                                                        double* __restrict__ out) {
  __shared__ double sh[256];
  double s = 0.0;
  for (int i = threadIdx.x; i < count; i += 256) s += part[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = sh[0];
}

// Energy (and adjoint) from the lower triangle of a symmetric K[(i,a),(j,b)] = (ia|jb).  One workgroup per pair
// a >= b: its o x o block X[i,j] = K[ia,jb] also holds the exchanged integrals, K_ibja = X[j,i], and all of the pair
// (b,a)'s, so it is read once into LDS (rows padded to o + 1) and half of K is read in all.  In the blocks a = b,
// which are symmetric, only i >= j is read.
// GRAD (a wavefront takes columns j, its lanes i) writes both blocks of G in runs of o and, with rpart non-null, the sums over one occupied index of
// w = K (2 K - K_ibja) / D^2: rpart[b + v (i + o a)] = sum_j w[ia,jb], and the same with a and b exchanged.
// Bound by the latency of a pair's loads and by memory: 8640 rows take 132 us (257 as a pass over all of K with the
// exchanged integrals read from memory), with G and the sums 328 (720 with w stored and summed by passes of its own).
template <bool GRAD>
__global__ __launch_bounds__(256) void mp2_lower_kernel(const double* __restrict__ K, const double* __restrict__ eps,
                                                        int o, int v, double* __restrict__ G,
                                                        double* __restrict__ rpart, double* __restrict__ part) {
  extern __shared__ double X[];  // X[i + (o + 1) j], then (GRAD) the wavefronts' sums over j, 4 x o
  __shared__ double sh[4];
  const int ld = o + 1, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // pairs in the order of b, then a, a contiguous range of them on each of the 8 XCDs: neighbours, whose runs of o
  // share cache lines, meet in one L2
  const long np = (long)v * (v + 1) / 2, per = np / 8, more = np % 8, xcd = blockIdx.x % 8;
  const long p = np - 1 - (xcd * per + (xcd < more ? xcd : more) + blockIdx.x / 8);
  int x = (int)((sqrt(8.0 * p + 1.0) - 1.0) / 2.0);
  while ((long)x * (x + 1) / 2 > p) --x;
  while ((long)(x + 1) * (x + 2) / 2 <= p) ++x;
  const int b = v - 1 - x, a = v - 1 - (int)(p - (long)x * (x + 1) / 2);
  const long ov = (long)o * v, blk = (long)o * a + ov * ((long)o * b), mir = (long)o * b + ov * ((long)o * a);
  // eight loads of a thread in flight (158 us at 8640 rows with one at a time)
  for (int q0 = threadIdx.x; q0 < o * o; q0 += 2048) {
    double x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int q = min(q0 + 256 * u, o * o - 1), i = q % o, j = q / o;
      x[u] = a == b ? K[blk + max(i, j) + ov * min(i, j)] : K[blk + i + ov * j];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int q = q0 + 256 * u;
      if (q < o * o) X[q % o + ld * (q / o)] = x[u];
    }
  }
  __syncthreads();
  const double eab = -eps[o + a] - eps[o + b];
  double s = 0.0, row[2] = {0.0, 0.0};
  if (!GRAD)
    for (int q = threadIdx.x; q < o * o; q += 256) {
      const int i = q % o, j = q / o;
      const double x = X[i + ld * j];
      s += x * ((2.0 * x - X[j + ld * i]) / (eps[i] + eps[j] + eab));
    }
  for (int j = wave; GRAD && j < o; j += 4) {
    double col = 0.0;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = lane + 64 * u;
      if (i >= o) continue;
      const double x = X[i + ld * j], d = eps[i] + eps[j] + eab, q = (2.0 * x - X[j + ld * i]) / d;
      s += x * q;
      G[blk + i + ov * j] = 2.0 * q;
      if (rpart) {
        const double w = x * q / d;
        row[u] += w;
        col += w;
      }
    }
    if (rpart) {
      for (int off = 32; off > 0; off >>= 1) col += __shfl_down(col, off, 64);
      if (lane == 0 && a != b) rpart[a + (long)v * (j + (long)o * b)] = col;
    }
  }
  if constexpr (GRAD) {
    if (a != b)  // the mirrored block: lanes j
      for (int i = wave; i < o; i += 4)
        for (int j = lane; j < o; j += 64)
          G[mir + j + ov * i] = 2.0 * ((2.0 * X[i + ld * j] - X[j + ld * i]) / (eps[i] + eps[j] + eab));
    if (rpart) {
      double* R = X + (long)ld * o;
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (lane + 64 * u < o) R[wave * o + lane + 64 * u] = row[u];
      __syncthreads();
      for (int i = threadIdx.x; i < o; i += 256)
        rpart[b + (long)v * (i + (long)o * a)] = (R[i] + R[o + i]) + (R[2 * o + i] + R[3 * o + i]);
    }
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if (lane == 0) sh[wave] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (a == b ? 1.0 : 2.0) * ((sh[0] + sh[1]) + (sh[2] + sh[3]));
}

// out = sum of `count` partial sums in a fixed order, four of a thread's loads in flight (with one at a time the
// 23436 of 216 virtual orbitals took 60 us)
__global__ __launch_bounds__(1024) void sum_pairs_kernel(const double* __restrict__ part, int count,
                                                         double* __restrict__ out) {
  __shared__ double sh[16];
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  for (int i = threadIdx.x; i < count; i += 4096)
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i + 1024 * u < count) s[u] += part[i + 1024 * u];
  double t = (s[0] + s[1]) + (s[2] + s[3]);
  for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = 0.0;
    for (int w = 0; w < 16; ++w) r += sh[w];
    out[0] = r;
  }
}

// r[ia] = 2 sum_b rpart[b, ia] (w is symmetric: its row sums are its column sums), a wavefront per row
__global__ __launch_bounds__(256) void mp2_lower_r_kernel(const double* __restrict__ rpart, int v, long ov,
                                                          double* __restrict__ r) {
  const int lane = threadIdx.x & 63;
  const long ia = blockIdx.x * 4L + (threadIdx.x >> 6);
  if (ia >= ov) return;
  double s = 0.0;
  for (int b = lane; b < v; b += 64) s += rpart[b + v * ia];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if (lane == 0) r[ia] = 2.0 * s;
}

// UMP2 blocks (UMP2.jl:30-77).  One block per (J,B) column of K[i,a,J,B] = (ia|JB).
// same != 0 (alpha-alpha or beta-beta, K square): accumulates (ia|jb)((ia|jb) - (ib|ja)) / D,
// half of which is the sum over i > j, a > b of <ij||ab>^2 / D; otherwise (ia|JB)^2 / D.
template <typename T>
__global__ __launch_bounds__(256) void ump2_energy_kernel(const T* __restrict__ K, const double* __restrict__ eA,
                                                          const double* __restrict__ eB, int oA, int vA, int oB,
                                                          int same, double* __restrict__ part) {
  __shared__ double sh[4];
  const int ovA = oA * vA;
  const int jb = blockIdx.x;
  const int j = jb % oB, b = jb / oB;
  const double ejb = eB[j] - eB[oB + b];
  const long col = (long)jb * ovA;
  double s = 0.0;
  for (int ia = threadIdx.x; ia < ovA; ia += 256) {
    const int i = ia % oA, a = ia / oA;
    const double k = (double)K[col + ia];
    const double d = eA[i] - eA[oA + a] + ejb;
    if (same) {
      const double kx = (double)K[(long)(i + oA * b) + (long)ovA * (j + oA * a)];  // (ib|ja)
      s += k * (k - kx) / d;
    } else {
      s += k * k / d;
    }
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[jb] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

}  // namespace

template <typename T>
double ump2_block_dev(jues_ctx* ctx, const T* K, const double* eA, const double* eB, int oA, int vA, int oB, int vB,
                      bool same) {
  const int cols = oB * vB;
  double* part = static_cast<double*>(scratch(ctx, 14, sizeof(double) * (size_t)(cols + 1)));
  {
    KTimer t(ctx, "ump2_energy", 4.0 * oA * vA * (double)cols, (double)oA * vA * cols * sizeof(T) * (same ? 2 : 1));
    hipLaunchKernelGGL((ump2_energy_kernel<T>), dim3(cols), dim3(256), 0, ctx->stream, K, eA, eB, oA, vA, oB,
                       same ? 1 : 0, part);
    hipLaunchKernelGGL(sum_fixed_kernel, dim3(1), dim3(256), 0, ctx->stream, part, cols, part + cols);
    JUES_HIP(hipGetLastError());
  }
  double E = 0.0;
  d2h(ctx, &E, part + cols, sizeof(double));
  return same ? 0.5 * E : E;
}

template <typename T>
double mp2_energy_dev(jues_ctx* ctx, const T* K, const double* eps, int o, int v) {
  const int ov = o * v;
  double* part = static_cast<double*>(scratch(ctx, 14, sizeof(double) * (size_t)(ov + 1)));
  {
    KTimer t(ctx, "mp2_energy", 6.0 * ov * ov, (double)ov * ov * sizeof(T) * 2);
    hipLaunchKernelGGL((mp2_energy_kernel<T>), dim3(ov), dim3(256), 0, ctx->stream, K, eps, o, v, part);
    hipLaunchKernelGGL(sum_fixed_kernel, dim3(1), dim3(256), 0, ctx->stream, part, ov, part + ov);
    JUES_HIP(hipGetLastError());
  }
  double E = 0.0;
  d2h(ctx, &E, part + ov, sizeof(double));
  return E;
}

double mp2_lower_dev(jues_ctx* ctx, const double* K, const double* eps, int o, int v, double* G, double* r,
                     double* work) {
  JUES_REQUIRE(o >= LOWER_MIN_O && o <= LOWER_MAX_O && (!r || (G && work)), "mp2_lower: bad arguments");
  const long ov = (long)o * v, pairs = (long)v * (v + 1) / 2;
  JUES_REQUIRE(pairs < (1L << 31), "mp2_lower: too many pairs");
  double* part = static_cast<double*>(scratch(ctx, 14, sizeof(double) * (size_t)(pairs + 1)));
  const size_t lds = sizeof(double) * (size_t)(o * (o + 1) + (r ? 4 * o : 0));
  {
    KTimer t(ctx, G ? "mp2_grad_g" : "mp2_energy", 6.0 * ov * ov / 2, (double)ov * ov * (G ? 12.0 : 4.0));
    if (G)
      hipLaunchKernelGGL(mp2_lower_kernel<true>, dim3((unsigned)pairs), dim3(256), lds, ctx->stream, K, eps, o, v, G,
                         r ? work : nullptr, part);
    else
      hipLaunchKernelGGL(mp2_lower_kernel<false>, dim3((unsigned)pairs), dim3(256), lds, ctx->stream, K, eps, o, v,
                         nullptr, nullptr, part);
    hipLaunchKernelGGL(sum_pairs_kernel, dim3(1), dim3(1024), 0, ctx->stream, part, (int)pairs, part + pairs);
    if (r)
      hipLaunchKernelGGL(mp2_lower_r_kernel, dim3((unsigned)((ov + 3) / 4)), dim3(256), 0, ctx->stream, work, v, ov, r);
    JUES_HIP(hipGetLastError());
  }
  double E = 0.0;
  d2h(ctx, &E, part + pairs, sizeof(double));
  return E;
}

template void mo_factors_dev<double>(jues_ctx*, const double*, int, const double*, int, double*);
template void mo_factors_dev<float>(jues_ctx*, const float*, int, const float*, int, float*);
template void mo_factors_dev<double>(jues_ctx*, const double*, int, const double*, int, double*, double*);
template void mo_factors_dev<float>(jues_ctx*, const float*, int, const float*, int, float*, float*);
template void tei_transform_dev<double>(jues_ctx*, const double*, int, const double*, int, const double*, int,
                                        const double*, int, double*);
template void tei_transform_dev<float>(jues_ctx*, const float*, int, const float*, int, const float*, int,
                                       const float*, int, float*);
template double mp2_energy_dev<double>(jues_ctx*, const double*, const double*, int, int);
template double mp2_energy_dev<float>(jues_ctx*, const float*, const double*, int, int);
template double ump2_block_dev<double>(jues_ctx*, const double*, const double*, const double*, int, int, int, int,
                                       bool);
template double ump2_block_dev<float>(jues_ctx*, const float*, const double*, const double*, int, int, int, int,
                                      bool);

}  // namespace jues
