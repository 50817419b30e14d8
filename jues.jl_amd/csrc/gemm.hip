// MFMA GEMM for gfx950 (FP64 and FP32), column-major, batched: LDS-staged kernels with 128x128, 64x64
// and 48 / 64 x 256 tiles, a direct kernel for products with few output tiles, and the dispatch
// between them.
//
// Every kernel works in 16x16 MFMA blocks (v_mfma_f64_16x16x4f64 / v_mfma_f32_16x16x4f32), issued with
// the operands swapped (B^T * A^T) so that each lane's accumulator column is an m index: lanes 0..15
// then hold 16 consecutive rows of C and the epilogue stores are 16-element contiguous runs along the
// leading dimension.
//
// Workgroup ids are remapped so that each of the 8 XCDs (each with its own L2) receives a contiguous
// range of tiles, and tiles are walked in groups of 8 tile-rows to reuse B columns within an L2.
#include "gemm_tail.h"
#include "jues_internal.h"

#include <algorithm>
#include <cstring>

namespace jues {
namespace {

typedef double dvec4 __attribute__((ext_vector_type(4)));
typedef float fvec4 __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma;
template <> struct Mfma<double> {
  typedef dvec4 acc;
  // accumulator element r of lane l is row (l/16) + 4r of the 16x16 block
  __device__ static inline int row(int lane, int r) { return (lane >> 4) + 4 * r; }
  __device__ static inline acc op(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma<float> {
  typedef fvec4 acc;
  // accumulator element r of lane l is row 4(l/16) + r of the 16x16 block
  __device__ static inline int row(int lane, int r) { return 4 * (lane >> 4) + r; }
  __device__ static inline acc op(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

constexpr int NT = 256, NXCD = TAIL_XCD;

// Raw buffer loads: the 64-bit base lives in a scalar resource descriptor, the
// per-lane part is one 32-bit byte offset and the per-element part a scalar
// offset, so an interior tile's loads hold no 64-bit address registers.
constexpr int kBufferDword3 = 0x00020000;  // gfx9-family raw buffer descriptor word 3
__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, 0x7fffffff, kBufferDword3);
}
template <typename T> __device__ inline T bload(__amdgpu_buffer_rsrc_t r, int voff, int soff);
template <> __device__ inline double bload<double>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
template <> __device__ inline float bload<float>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

// Place of a workgroup in a launch of many batch entries or K chunks: x among an entry's gridDim.x workgroups and
// the entry z.  Workgroups go to the 8 XCDs in turn, so a launch whose gridDim.z is a multiple of 8 (padded to
// it by the host; entries past the last one return) is dealt so that an entry's workgroups stay on one XCD, whose L2
// then holds the entry's operands once.  Dealt in turn, each L2 fetched nearly all of them: FP32 34 x 34 x 1227400
// in 128 chunks took 357 us, 142 this way (60 at the copy rate).  Returns whether it was.
__device__ inline bool entry_place(int& x, int& z) {
  x = (int)blockIdx.x;
  z = (int)blockIdx.z;
  if (gridDim.z == 1 || gridDim.z % NXCD != 0) return false;
  const long id = x + (long)gridDim.x * z, slot = id / NXCD;
  x = (int)(slot % gridDim.x);
  z = (int)(slot / gridDim.x) * NXCD + (int)(id % NXCD);
  return true;
}

// A value that is the same in all lanes, in scalar registers: the operand offsets that a two-segment launch reads from its
// table.  In vector registers they had gemm32_nn_kernel spill in its loop: the FP32 W products of the triples at v = 340
// reach 94 TFLOP/s that way, 101 this way.
__device__ inline long uniform(long x) {
  return (long)((unsigned long)(unsigned)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32 |
                (unsigned)__builtin_amdgcn_readfirstlane((int)x));
}

// Tile of workgroup pid of nwg, of which only the first tiles_m * tiles_n carry a tile (a launch
// padded to a multiple of NXCD); false for the padding ids.  plain: the workgroups are on one XCD already.
__device__ inline bool tile_coords_bounded(int pid, int nwg, int tiles_m, int tiles_n, int& tm, int& tn,
                                           bool plain = false) {
  // XCD-aware remap (bijective for any nwg): consecutive hardware ids go to different XCDs; give
  // each XCD a contiguous block of logical tile ids
  const int per = (nwg + NXCD - 1) / NXCD;
  int tall = nwg % NXCD;
  if (tall == 0) tall = NXCD;
  const int xcd = pid % NXCD, loc = pid / NXCD;
  const int p2 = plain ? pid : xcd < tall ? xcd * per + loc : tall * per + (xcd - tall) * (per - 1) + loc;
  if (p2 >= tiles_m * tiles_n) return false;
  grouped_tile(p2, tiles_m, tiles_n, tm, tn);
  return true;
}

// One product of a high-occupancy kernel launch: C = alpha A op(B) + beta C, batched over
// blockIdx.z with strides sA, sB, sC.  A launch carries one or two of them (two
// independent products sharing the grid, so that neither leaves a partly idle last round).
template <typename T>
struct GemmSide {
  const T* A;
  const T* B;
  T* C;
  long lda, ldb, ldc, sA, sB, sC;
  int M, N, K, tiles_m, tiles_n;
  int Klast;  // K of the last batch entry (a split-K launch's shorter last chunk), else K
  // optional second contraction segment: C += alpha A1 op(B1) over K1 more columns (same lda,
  // ldb and batch strides); with K1 > 0, K and K1 are multiples of 16
  const T* A1;
  const T* B1;
  int K1;
  // SEG launches: batch entry z is entry z % inner of group z / inner, whose operands A, B, A1, B1 are offset
  // by tab[4 group + 0..3] elements and whose C by group * sG
  const long* tab = nullptr;
  int inner = 1;
  long sG = 0;
  int nz = 1;  // batch entries or K chunks of the launch
  TailMap tail;      // TAIL launches
  T* part = nullptr;
  // FP32 products that write an FP64 result (the OUT64 instantiation; C is not used there)
  double* C64 = nullptr;
};

// FP32 C = alpha A op(B) + beta C with A m-contiguous and B k-contiguous (NN) or
// n-contiguous (NT), 128x128 tile, 4 wavefronts of 64x64.
// The K slice is 16 deep, so a workgroup needs 32 KB of LDS and at most 128 VGPRs per
// lane: four workgroups (16 wavefronts) share a CU and cover each other's load and
// barrier latency (two workgroups of 32-deep slices reach 73% MFMA-busy, this form 91% with the
// last slice peeled off the main loop and the last round of tiles shared, ~89% with a conditional loop body).
// LDS holds each slice as 64-byte rows of 16 k-values per m (A) or n (B); the 16-byte
// chunk q of row r sits at chunk q ^ ((r >> 2) & 3), so slices are written with 16-byte
// stores and fragments read with 16-byte loads.  Lane l of a 16x16x4 MFMA supplies
// k = 4 (l / 16) + s at step s = 0..3 (the same permutation for both operands): one
// 16-byte read per 16-row block.  B's four fragment blocks are held for the slice and A's
// are streamed one block ahead of the MFMAs that use them.  Rows of the last tile row or
// column beyond M or N load a clamped row and are not stored.  A K tail (16 not dividing K)
// is the first slice: zero-padded, loaded element by element once in the prologue.  TA (A
// k-contiguous, TN / TT) stages A like a k-contiguous B; SEG instantiations add a second contraction
// segment (A1, B1 over K1 columns).
typedef float f4v __attribute__((ext_vector_type(4)));

__device__ inline int g32_chunk(int q, int r) { return q ^ ((r >> 2) & 3); }

// Workgroups [0, nt0) run product p0 (nt0 padded up to a multiple of NXCD when a second
// product follows), the rest p1.  OUT64: C = alpha A op(B) is written to the FP64 array C64
// (beta = 0).
template <int KIND, bool TB, bool TA = false, bool SEG = false, bool OUT64 = false, int BT = 128, bool TAIL = false>
__global__ __launch_bounds__(256, 4) void gemm32_nn_kernel(GemmSide<float> p0, GemmSide<float> p1, int nt0,
                                                           float alpha, float beta) {
  constexpr int BM = BT, BN = BT, BK = 16;
  // 64-row shares per thread, 16-row MFMA blocks per wavefront side, wavefront tile edge
  constexpr int NJ = BT / 64, NB = BT / 32;
  __shared__ __attribute__((aligned(16))) float As[2][BM * BK];
  __shared__ __attribute__((aligned(16))) float Bs[2][BN * BK];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  // a wavefront's 16-row and 16-column blocks alternate with its neighbour's, so that a tile at the edge of M
  // or N keeps all of them at work on the blocks it has
  const auto mrow = [&](int i) { return (2 * i + wm) * 16; };
  const auto ncol = [&](int j) { return (2 * j + wn) * 16; };
  int bx, bz;
  const bool placed = entry_place(bx, bz), second = !TAIL && bx >= nt0;
  const GemmSide<float> g = second ? p1 : p0;
  const int M = g.M, N = g.N, K = bz == g.nz - 1 ? g.Klast : g.K;
  if (bz >= g.nz) return;
  const long lda = g.lda, ldb = g.ldb, ldc = g.ldc;
  const int grp = SEG ? __builtin_amdgcn_readfirstlane(bz / g.inner) : 0;  // the table only in the SEG instantiations
  const long zb = (long)bz - (SEG ? (long)grp * g.inner : 0L);
  const long* tab = SEG ? g.tab + 4L * grp : nullptr;
  const float* __restrict__ A = g.A + zb * g.sA + (SEG ? uniform(tab[0]) : 0L);
  const float* __restrict__ B = g.B + zb * g.sB + (SEG ? uniform(tab[1]) : 0L);
  float* __restrict__ C = OUT64 ? nullptr : g.C + zb * g.sC + (SEG ? grp * g.sG : 0L);
  // a second contraction segment (A1, B1 over K1 columns) only in the SEG instantiations
  const int K1 = SEG ? g.K1 : 0;
  const float* A1 = SEG ? g.A1 + zb * g.sA + uniform(tab[2]) : A;
  const float* B1 = SEG ? g.B1 + zb * g.sB + uniform(tab[3]) : B;
  // slices: the K tail (columns 16 floor(K/16) .. K-1, zero-padded) first when there is one, then the full
  // slices from k = 0; the tail is loaded in the prologue
  const int K16 = K / BK * BK, tail = K > K16 ? 1 : 0;
  const int nk = K16 / BK + tail + K1 / BK;
  int tm, tn, ka = 0, kb = nk, wg = 0;
  bool shared = false;  // the workgroup's result is a part of its tile
  if (TAIL && bx >= g.tail.whole) {
    int t = 0, c = 0, nc = 1;
    g.tail.part(bx - g.tail.whole, t, c, nc, wg);
    shared = nc > 1;
    ka = (int)((long)nk * c / nc);
    kb = (int)((long)nk * (c + 1) / nc);
    g.tail.coords(g.tail.whole + t, tm, tn);
  } else if (TAIL) {
    const int per = g.tail.whole / NXCD;
    g.tail.coords(bx % NXCD * per + bx / NXCD, tm, tn);
  } else if (!tile_coords_bounded(second ? bx - nt0 : bx, second ? (int)gridDim.x - nt0 : nt0, g.tiles_m, g.tiles_n,
                                  tm, tn, placed)) {
    return;
  }
  const int m0 = tm * BM, n0 = tn * BN;

  // A share: row am, 4-k chunks ac0 and ac0 + 2; B share: rows bn and bn + 64, chunk bc
  // (ac0 is uniform within a wavefront: in a scalar register the per-k offsets are scalar too)
  const int am = tid & (BT - 1), ac0 = __builtin_amdgcn_readfirstlane(tid / BT);
  const int bn = tid >> 2, bc = tid & 3;
  float ra[4 * NJ];
  f4v rat[NJ];  // TA (A k-contiguous): shared like a k-contiguous B, rows bn and bn + 64, chunk bc
  f4v rb[NJ];
  // rows past the edge of M or N load the last row instead (their results are not stored).
  // B k-contiguous (TB false): 16-byte loads of 4 k; B n-contiguous (TB true, op(B) = B^T):
  // loaded like A, one dword per k with row n = am of the tile.
  const int a_voff = 4 * (min(m0 + am, M - 1) - m0);
  const int bt_voff = 4 * (min(n0 + am, N - 1) - n0);
  const int b_voff0 = 4 * (4 * bc + (min(n0 + bn, N - 1) - n0) * (int)ldb);
  const int b_voff1 = 4 * (4 * bc + (min(n0 + bn + 64, N - 1) - n0) * (int)ldb);
  // TA: k-contiguous rows addressed from two bases, rows m0.. and m1 = min(m0 + 64, M - 1).., so that a
  // byte offset spans at most 63 rows (the same for B in the TA instantiations)
  const int m1 = min(m0 + 64, M - 1), n1 = min(n0 + 64, N - 1);
  const int at_voff0 = 4 * (4 * bc + (min(m0 + bn, M - 1) - m0) * (int)lda);
  const int at_voff1 = 4 * (4 * bc + (min(m0 + bn + 64, M - 1) - m1) * (int)lda);
  const int b2_voff1 = 4 * (4 * bc + (min(n0 + bn + 64, N - 1) - n1) * (int)ldb);
  auto load_seg = [&](const float* Ab, const float* Bb, int k0) {
    if constexpr (TA) {
      const auto rA0 = make_rsrc(Ab + k0 + (long)m0 * lda);
      const auto rA1 = make_rsrc(Ab + k0 + (long)m1 * lda);
      rat[0] = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rA0, at_voff0, 0, 0));
      if constexpr (NJ == 2) rat[1] = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rA1, at_voff1, 0, 0));
    } else {
      const auto rA = make_rsrc(Ab + m0 + (long)k0 * lda);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          ra[4 * j + u] = bload<float>(rA, a_voff, 4 * (4 * (ac0 + 2 * j) + u) * (int)lda);
    }
    if constexpr (TB) {
      const auto rB = make_rsrc(Bb + n0 + (long)k0 * ldb);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          rb[j][u] = bload<float>(rB, bt_voff, 4 * (4 * (ac0 + 2 * j) + u) * (int)ldb);
    } else if constexpr (TA) {
      const auto rB0 = make_rsrc(Bb + k0 + (long)n0 * ldb);
      const auto rB1 = make_rsrc(Bb + k0 + (long)n1 * ldb);
      rb[0] = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rB0, b_voff0, 0, 0));
      if constexpr (NJ == 2) rb[1] = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rB1, b2_voff1, 0, 0));
    } else {
      const auto rB = make_rsrc(Bb + k0 + (long)n0 * ldb);
      rb[0] = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rB, b_voff0, 0, 0));
      if constexpr (NJ == 2) rb[1] = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rB, b_voff1, 0, 0));
    }
  };
  // full slice s of the contraction: segment 0's K / BK slices, then segment 1's
  const int nk0 = K / BK;
  auto load = [&](int s) {
    if constexpr (SEG) {
      if (s < nk0) load_seg(A, B, s * BK);
      else load_seg(A1, B1, (s - nk0) * BK);
    } else {
      load_seg(A, B, s * BK);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if constexpr (TA) {
        const int m = bn + 64 * j;
        *reinterpret_cast<f4v*>(&As[buf][m * BK + 4 * g32_chunk(bc, m)]) = rat[j];
      } else {
        const int c = ac0 + 2 * j;
        *reinterpret_cast<f4v*>(&As[buf][am * BK + 4 * g32_chunk(c, am)]) =
            f4v{ra[4 * j], ra[4 * j + 1], ra[4 * j + 2], ra[4 * j + 3]};
      }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if constexpr (TB) {
        const int c = ac0 + 2 * j;
        *reinterpret_cast<f4v*>(&Bs[buf][am * BK + 4 * g32_chunk(c, am)]) = rb[j];
      } else {
        const int n = bn + 64 * j;
        *reinterpret_cast<f4v*>(&Bs[buf][n * BK + 4 * g32_chunk(bc, n)]) = rb[j];
      }
    }
  };

  fvec4 acc[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = fvec4{0, 0, 0, 0};

  const int fr = lane & 15, fk = lane >> 4;
  if (tail && ka == 0) {
    if constexpr (TA) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int gk = K16 + 4 * bc + u;
          const int m = min(m0 + bn + 64 * j, M - 1);
          const float val = A[(long)min(gk, K - 1) + (long)m * lda];
          rat[j][u] = gk < K ? val : 0.f;
        }
    } else {
      const float* Ar = A + m0 + (a_voff >> 2);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int gk = K16 + 4 * (ac0 + 2 * j) + u;
          const float val = Ar[(long)min(gk, K - 1) * lda];
          ra[4 * j + u] = gk < K ? val : 0.f;
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float val;
        if constexpr (TB) {
          const int gk = K16 + 4 * (ac0 + 2 * j) + u;
          val = gk < K ? B[n0 + (bt_voff >> 2) + (long)min(gk, K - 1) * ldb] : 0.f;
        } else {
          const int gk = K16 + 4 * bc + u;
          const int n = min(n0 + bn + 64 * j, N - 1);
          val = gk < K ? B[(long)min(gk, K - 1) + (long)n * ldb] : 0.f;
        }
        rb[j][u] = val;
      }
  } else {
    load(ka - tail);
  }
  store(0);
  __syncthreads();
  auto compute = [&](int cur) {
    f4v bf[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int r = ncol(j) + fr;
      bf[j] = *reinterpret_cast<const f4v*>(&Bs[cur][r * BK + 4 * g32_chunk(fk, r)]);
    }
    f4v a0 = *reinterpret_cast<const f4v*>(&As[cur][(mrow(0) + fr) * BK + 4 * g32_chunk(fk, mrow(0) + fr)]);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      f4v a1;
      if (i + 1 < NB) {
        const int r = mrow(i + 1) + fr;
        a1 = *reinterpret_cast<const f4v*>(&As[cur][r * BK + 4 * g32_chunk(fk, r)]);
      }
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[j][s2], a0[s2], acc[i][j], 0, 0, 0);
      if (i + 1 < NB) a0 = a1;
    }
  };
  // the last slice is peeled off, so that the loop body is one block without conditions (a schedule
  // that keeps the matrix pipe about 5% busier on the ring products than the conditional form)
  // a tile past the edge of M or N: only the blocks that hold results
  const int ilim = __builtin_amdgcn_readfirstlane(min(NB, (M - m0 - 16 * wm + 31) / 32));
  const int jlim = __builtin_amdgcn_readfirstlane(min(NB, (N - n0 - 16 * wn + 31) / 32));
  auto compute_edge = [&](int cur) {
    if (ilim <= 0 || jlim <= 0) return;
    f4v bf[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int r = ncol(j) + fr;
      bf[j] = *reinterpret_cast<const f4v*>(&Bs[cur][r * BK + 4 * g32_chunk(fk, r)]);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (i >= ilim) break;
      const int r = mrow(i) + fr;
      const f4v a = *reinterpret_cast<const f4v*>(&As[cur][r * BK + 4 * g32_chunk(fk, r)]);
#pragma unroll
      for (int j = 0; j < NB; ++j)
        if (j < jlim)
#pragma unroll
          for (int s2 = 0; s2 < 4; ++s2)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[j][s2], a[s2], acc[i][j], 0, 0, 0);
    }
  };
  const auto loop = [&](auto slice) {
    for (int kt = ka; kt + 1 < kb; ++kt) {
      const int cur = (kt - ka) & 1;
      load(kt + 1 - tail);
      slice(cur);
      store(cur ^ 1);
      __syncthreads();
    }
    slice((kb - 1 - ka) & 1);
  };
  // (in the two-segment and FP64-output instantiations the second loop costs spills)
  if constexpr (SEG || OUT64) {
    loop(compute);
  } else {
    if (ilim == NB && jlim == NB) loop(compute);
    else loop(compute_edge);
  }
  if (TAIL && shared) {
    // a partial tile, as the registers hold it, for gemm_tail_kernel
    float* __restrict__ P = g.part + (long)wg * (BM * BN) + tid;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) P[((i * NB + j) * 4 + r) * 256] = alpha * acc[i][j][r];
    return;
  }

  if constexpr (OUT64) {
    double* __restrict__ C64 = g.C64 + (long)bz * g.sC;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int m = m0 + mrow(i) + (lane & 15);
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = n0 + ncol(j) + 4 * (lane >> 4) + r;
          if (n < N) C64[(long)m + (long)n * ldc] = (double)(alpha * acc[i][j][r]);
        }
      }
    }
    return;
  }
  if (beta != 0.f && m0 + BM <= M && n0 + BN <= N) {
    // interior tile accumulating into C: per 16-row block, all of the lane's C loads before
    // its stores (an element-wise load -> store round trip would serialise the epilogue)
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const long m = m0 + mrow(i) + (lane & 15);
      float cv[NB][4];
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) cv[j][r] = C[m + (long)(n0 + ncol(j) + 4 * (lane >> 4) + r) * ldc];
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          C[m + (long)(n0 + ncol(j) + 4 * (lane >> 4) + r) * ldc] = alpha * acc[i][j][r] + beta * cv[j][r];
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int m = m0 + mrow(i) + (lane & 15);
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + ncol(j) + 4 * (lane >> 4) + r;
        if (n < N) {
          const long off = (long)m + (long)n * ldc;
          float v = alpha * acc[i][j][r];
          if (beta != 0.f) v += beta * C[off];
          C[off] = v;
        }
      }
    }
  }
}

// FP64 C = alpha A op(B) + beta C with A m-contiguous and B k-contiguous (NN) or
// n-contiguous (NT): 128x128 tile over 8 wavefronts of 64x32, so the accumulators take 64
// VGPRs and a lane stays within 128 -- two 512-thread workgroups (16 wavefronts) per CU.
// K slices are 16 doubles deep, held in LDS as 128-byte rows per m (A) or n (B) with the
// 16-byte chunk q of row r at chunk q ^ (r & 7); lane l supplies k = 4 (l / 16) + s at MFMA
// step s = 0..3 for both operands (two 16-byte fragment reads per 16-row block).  B's two
// blocks are held for the slice and A's four streamed one ahead.  Rows past M or N load a
// clamped row and are not stored; a K tail is the first slice, zero-padded, loaded in the prologue.
// BT = 64: 64x64 tiles over 4 wavefronts of 32x32, twice the operand traffic for four times the workgroups: 1125^3 takes
// 85 us (148 with 128x128 tiles), 66 in three chunks of K (71).
typedef double d2v __attribute__((ext_vector_type(2)));

__device__ inline int g64_chunk(int q, int r) { return q ^ (r & 7); }

template <int KIND, bool TB, bool TA = false, bool SEG = false, int BT = 128, bool TAIL = false>
__global__ __launch_bounds__(4 * BT, 4) void gemm64_kernel(GemmSide<double> p0, GemmSide<double> p1, int nt0,
                                                        double alpha, double beta) {
  constexpr int BM = BT, BN = BT, BK = 16;
  constexpr int HT = BT / 2, IB = BT / 32;  // half tile; 16-row MFMA blocks of a wavefront (HT rows)
  __shared__ __attribute__((aligned(16))) double As[2][BM * BK];
  __shared__ __attribute__((aligned(16))) double Bs[2][BN * BK];
  const int tid = threadIdx.x, lane = tid & 63, wave = BT == 64 ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;  // 2 x (BT / 32) wavefronts of HT x 32
  int bx, bz;
  const bool placed = entry_place(bx, bz), second = !TAIL && bx >= nt0;
  const GemmSide<double> g = second ? p1 : p0;
  const int M = g.M, N = g.N, K = bz == g.nz - 1 ? g.Klast : g.K;
  if (bz >= g.nz) return;
  const long lda = g.lda, ldb = g.ldb, ldc = g.ldc;
  const int grp = SEG ? bz / g.inner : 0;  // the table only in the SEG instantiations
  const long zb = (long)bz - (SEG ? (long)grp * g.inner : 0L);
  const long* tab = SEG ? g.tab + 4L * grp : nullptr;
  const double* __restrict__ A = g.A + zb * g.sA + (SEG ? tab[0] : 0L);
  const double* __restrict__ B = g.B + zb * g.sB + (SEG ? tab[1] : 0L);
  double* __restrict__ C = g.C + zb * g.sC + (SEG ? grp * g.sG : 0L);
  // a second contraction segment (A1, B1 over K1 columns) only in the SEG instantiations
  const int K1 = SEG ? g.K1 : 0;
  const double* A1 = SEG ? g.A1 + zb * g.sA + tab[2] : A;
  const double* B1 = SEG ? g.B1 + zb * g.sB + tab[3] : B;
  // slices: the K tail (columns 16 floor(K/16) .. K-1, zero-padded) first when there is one, then the full
  // slices from k = 0; the tail is loaded in the prologue
  const int K16 = K / BK * BK, tail = K > K16 ? 1 : 0;
  const int nk = K16 / BK + tail + K1 / BK;
  int tm, tn, ka = 0, kb = nk, wg = 0;
  bool shared = false;  // the workgroup's result is a part of its tile
  if (TAIL && bx >= g.tail.whole) {
    int t = 0, c = 0, nc = 1;
    g.tail.part(bx - g.tail.whole, t, c, nc, wg);
    shared = nc > 1;
    ka = (int)((long)nk * c / nc);
    kb = (int)((long)nk * (c + 1) / nc);
    g.tail.coords(g.tail.whole + t, tm, tn);
  } else if (TAIL) {
    const int per = g.tail.whole / NXCD;
    g.tail.coords(bx % NXCD * per + bx / NXCD, tm, tn);
  } else if (!tile_coords_bounded(second ? bx - nt0 : bx, second ? (int)gridDim.x - nt0 : nt0, g.tiles_m, g.tiles_n,
                                  tm, tn, placed)) {
    return;
  }
  const int m0 = tm * BM, n0 = tn * BN;
  // A (and n-contiguous B) share: row am, k = 4 kq + u; k-contiguous B share: rows bn, bn + HT, chunk bc
  // (a k-contiguous A, TA, is shared like a k-contiguous B)
  const int am = tid & (BT - 1), kq = __builtin_amdgcn_readfirstlane(tid / BT);
  const int bn = tid >> 3, bc = tid & 7;
  double ra[4];
  d2v rat[2];
  d2v rb[2];
  const int a_voff = 8 * (min(m0 + am, M - 1) - m0);
  const int bt_voff = 8 * (min(n0 + am, N - 1) - n0);
  const int b_voff0 = 8 * (2 * bc + (min(n0 + bn, N - 1) - n0) * (int)ldb);
  const int b_voff1 = 8 * (2 * bc + (min(n0 + bn + HT, N - 1) - n0) * (int)ldb);
  // TA: k-contiguous rows addressed from two bases, rows m0.. and m1 = min(m0 + HT, M - 1).., so that a
  // byte offset spans at most 63 rows (the same for B in the TA instantiations)
  const int m1 = min(m0 + HT, M - 1), n1 = min(n0 + HT, N - 1);
  const int at_voff0 = 8 * (2 * bc + (min(m0 + bn, M - 1) - m0) * (int)lda);
  const int at_voff1 = 8 * (2 * bc + (min(m0 + bn + HT, M - 1) - m1) * (int)lda);
  const int b2_voff1 = 8 * (2 * bc + (min(n0 + bn + HT, N - 1) - n1) * (int)ldb);
  auto load_seg = [&](const double* Ab, const double* Bb, int k0) {
    if constexpr (TA) {
      const auto rA0 = make_rsrc(Ab + k0 + (long)m0 * lda);
      const auto rA1 = make_rsrc(Ab + k0 + (long)m1 * lda);
      rat[0] = __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(rA0, at_voff0, 0, 0));
      rat[1] = __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(rA1, at_voff1, 0, 0));
    } else {
      const auto rA = make_rsrc(Ab + m0 + (long)k0 * lda);
#pragma unroll
      for (int u = 0; u < 4; ++u) ra[u] = bload<double>(rA, a_voff, 8 * (4 * kq + u) * (int)lda);
    }
    if constexpr (TB) {
      const auto rB = make_rsrc(Bb + n0 + (long)k0 * ldb);
#pragma unroll
      for (int u = 0; u < 4; ++u) rb[u >> 1][u & 1] = bload<double>(rB, bt_voff, 8 * (4 * kq + u) * (int)ldb);
    } else if constexpr (TA) {
      const auto rB0 = make_rsrc(Bb + k0 + (long)n0 * ldb);
      const auto rB1 = make_rsrc(Bb + k0 + (long)n1 * ldb);
      rb[0] = __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(rB0, b_voff0, 0, 0));
      rb[1] = __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(rB1, b2_voff1, 0, 0));
    } else {
      const auto rB = make_rsrc(Bb + k0 + (long)n0 * ldb);
      rb[0] = __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(rB, b_voff0, 0, 0));
      rb[1] = __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(rB, b_voff1, 0, 0));
    }
  };
  // full slice s of the contraction: segment 0's K / BK slices, then segment 1's
  const int nk0 = K / BK;
  auto load = [&](int s) {
    if constexpr (SEG) {
      if (s < nk0) load_seg(A, B, s * BK);
      else load_seg(A1, B1, (s - nk0) * BK);
    } else {
      load_seg(A, B, s * BK);
    }
  };
  auto store = [&](int buf) {
    if constexpr (TA) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int m = bn + HT * j;
        *reinterpret_cast<d2v*>(&As[buf][m * BK + 2 * g64_chunk(bc, m)]) = rat[j];
      }
    } else {
      *reinterpret_cast<d2v*>(&As[buf][am * BK + 2 * g64_chunk(2 * kq, am)]) = d2v{ra[0], ra[1]};
      *reinterpret_cast<d2v*>(&As[buf][am * BK + 2 * g64_chunk(2 * kq + 1, am)]) = d2v{ra[2], ra[3]};
    }
    if constexpr (TB) {
      *reinterpret_cast<d2v*>(&Bs[buf][am * BK + 2 * g64_chunk(2 * kq, am)]) = rb[0];
      *reinterpret_cast<d2v*>(&Bs[buf][am * BK + 2 * g64_chunk(2 * kq + 1, am)]) = rb[1];
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = bn + HT * j;
        *reinterpret_cast<d2v*>(&Bs[buf][n * BK + 2 * g64_chunk(bc, n)]) = rb[j];
      }
    }
  };

  dvec4 acc[IB][2];
#pragma unroll
  for (int i = 0; i < IB; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = dvec4{0, 0, 0, 0};
  const int fr = lane & 15, fk = lane >> 4;
  if (tail && ka == 0) {
    if constexpr (TA) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int gk = K16 + 2 * bc + u;
          const int m = min(m0 + bn + HT * j, M - 1);
          const double val = A[(long)min(gk, K - 1) + (long)m * lda];
          rat[j][u] = gk < K ? val : 0.0;
        }
    } else {
      const double* Ar = A + m0 + (a_voff >> 3);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int gk = K16 + 4 * kq + u;
        const double val = Ar[(long)min(gk, K - 1) * lda];
        ra[u] = gk < K ? val : 0.0;
      }
    }
    if constexpr (TB) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int gk = K16 + 4 * kq + u;
        const double val = B[n0 + (bt_voff >> 3) + (long)min(gk, K - 1) * ldb];
        rb[u >> 1][u & 1] = gk < K ? val : 0.0;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int gk = K16 + 2 * bc + u;
          const int n = min(n0 + bn + HT * j, N - 1);
          const double val = B[(long)min(gk, K - 1) + (long)n * ldb];
          rb[j][u] = gk < K ? val : 0.0;
        }
    }
  } else {
    load(ka - tail);
  }
  store(0);
  __syncthreads();
  // the 16-row and 16-column blocks of a wavefront: in turn with its neighbours' (erow, ecol) in 64x64 tiles, one piece in
  // whole 128x128 tiles, where turns cost a 20400^3 product 6%, and in turn in those with blocks past the edge of M or N,
  // so that all wavefronts have some of the others
  constexpr bool TURN = BT == 64;
  const auto erow = [&](int i) { return (2 * i + wm) * 16; };
  const auto ecol = [&](int j) { return (BT / 32 * j + wn) * 16; };
  const auto frow = [&](int i) { return TURN ? erow(i) : wm * HT + i * 16; };
  const auto fcol = [&](int j) { return TURN ? ecol(j) : wn * 32 + j * 16; };
  auto compute = [&](int cur) {
    d2v bf[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = fcol(j) + fr;
      bf[j][0] = *reinterpret_cast<const d2v*>(&Bs[cur][r * BK + 2 * g64_chunk(2 * fk, r)]);
      bf[j][1] = *reinterpret_cast<const d2v*>(&Bs[cur][r * BK + 2 * g64_chunk(2 * fk + 1, r)]);
    }
    d2v a0[2], a1[2];
    {
      const int r = frow(0) + fr;
      a0[0] = *reinterpret_cast<const d2v*>(&As[cur][r * BK + 2 * g64_chunk(2 * fk, r)]);
      a0[1] = *reinterpret_cast<const d2v*>(&As[cur][r * BK + 2 * g64_chunk(2 * fk + 1, r)]);
    }
#pragma unroll
    for (int i = 0; i < IB; ++i) {
      if (i + 1 < IB) {
        const int r = frow(i + 1) + fr;
        a1[0] = *reinterpret_cast<const d2v*>(&As[cur][r * BK + 2 * g64_chunk(2 * fk, r)]);
        a1[1] = *reinterpret_cast<const d2v*>(&As[cur][r * BK + 2 * g64_chunk(2 * fk + 1, r)]);
      }
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf[j][s2 >> 1][s2 & 1], a0[s2 >> 1][s2 & 1], acc[i][j],
                                                           0, 0, 0);
      if (i + 1 < IB) { a0[0] = a1[0]; a0[1] = a1[1]; }
    }
  };
  // the last slice is peeled off, so that the loop body is one block without conditions
  const int ilim = __builtin_amdgcn_readfirstlane(min(IB, (M - m0 - 16 * wm + 31) / 32));
  const int jlim = __builtin_amdgcn_readfirstlane(min(2, (N - n0 - 16 * wn + HT - 1) / HT));
  const bool edge = TURN ? ilim < IB || jlim < 2 : M - m0 <= BM - 16 || N - n0 <= BN - 16;
  // only the blocks that hold results
  auto compute_edge = [&](int cur) {
    if (ilim <= 0 || jlim <= 0) return;
    d2v bf[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = ecol(j) + fr;
      bf[j][0] = *reinterpret_cast<const d2v*>(&Bs[cur][r * BK + 2 * g64_chunk(2 * fk, r)]);
      bf[j][1] = *reinterpret_cast<const d2v*>(&Bs[cur][r * BK + 2 * g64_chunk(2 * fk + 1, r)]);
    }
#pragma unroll
    for (int i = 0; i < IB; ++i) {
      if (i >= ilim) break;
      const int r = erow(i) + fr;
      const d2v a[2] = {*reinterpret_cast<const d2v*>(&As[cur][r * BK + 2 * g64_chunk(2 * fk, r)]),
                        *reinterpret_cast<const d2v*>(&As[cur][r * BK + 2 * g64_chunk(2 * fk + 1, r)])};
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (j < jlim)
#pragma unroll
          for (int s2 = 0; s2 < 4; ++s2)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf[j][s2 >> 1][s2 & 1], a[s2 >> 1][s2 & 1], acc[i][j],
                                                             0, 0, 0);
    }
  };
  const auto loop = [&](auto slice) {
    for (int kt = ka; kt + 1 < kb; ++kt) {
      const int cur = (kt - ka) & 1;
      load(kt + 1 - tail);
      slice(cur);
      store(cur ^ 1);
      __syncthreads();
    }
    slice((kb - 1 - ka) & 1);
  };
  if (edge) loop(compute_edge);
  else loop(compute);
  const auto mrow = [&](int i) { return edge ? erow(i) : frow(i); };
  const auto ncol = [&](int j) { return edge ? ecol(j) : fcol(j); };
  if (TAIL && shared) {
    // a partial tile, as the registers hold it, for gemm_tail_kernel
    double* __restrict__ P = g.part + (long)wg * (BM * BN) + tid;
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) P[((i * 2 + j) * 4 + r) * (4 * BT)] = alpha * acc[i][j][r];
    return;
  }

  // acc[i][j][r]: C(m, n) with m = lane % 16 of block i, n = lane / 16 + 4 r of block j
  if (beta != 0.0 && m0 + BM <= M && n0 + BN <= N) {
    // interior tile accumulating into C: per 16-row block, the loads before the stores
#pragma unroll
    for (int i = 0; i < IB; ++i) {
      const long m = m0 + mrow(i) + (lane & 15);
      double cv[2][4];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) cv[j][r] = C[m + (long)(n0 + ncol(j) + (lane >> 4) + 4 * r) * ldc];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          C[m + (long)(n0 + ncol(j) + (lane >> 4) + 4 * r) * ldc] = alpha * acc[i][j][r] + beta * cv[j][r];
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < IB; ++i) {
    const int m = m0 + mrow(i) + (lane & 15);
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + ncol(j) + (lane >> 4) + 4 * r;
        if (n < N) {
          const long off = (long)m + (long)n * ldc;
          double v = alpha * acc[i][j][r];
          if (beta != 0.0) v += beta * C[off];
          C[off] = v;
        }
      }
    }
  }
}

// C = alpha op(A) op(B) + beta C for products with few output tiles (M = 1 vectors, o x o and o x v
// blocks, the (ov) x (ov) products of a small basis): a (16 IM) x (16 JN) tile per workgroup, whose NW
// wavefronts share the contraction instead of the tile.  Wavefront w takes the 16-deep k-slabs w, w + NW,
// ...: it loads their fragments from global memory straight into registers (nothing is shared between
// wavefronts, so nothing is staged in LDS and the loop has no barrier), two slabs in flight, and the
// NW partial tiles are added in a fixed order through LDS at the end, in FP64 as every sum of partial results here.  Lane l supplies
// k = 4 (l / 16) + s at MFMA step s, so a k-contiguous operand is read 4 consecutive k per lane and an
// m-contiguous one in runs of 16 rows.  Rows past M or N load a clamped row and are not stored; the K
// tail is a predicated slab after the full ones.
// Bound by the latency of a wavefront's loads (two slabs in flight), and from a few thousand tiles on by the L2s, since
// operands are read once a tile.  FP64, 128-row tiles before: 1 x 2000 x 2000 275 us and 17 here, 5 x 5 x 1805 251 and 6,
// 20 x 20 x 200000 about 130 and 26.
template <typename T, bool TA, bool TB, int NW, int IM, int JN>
__global__ __launch_bounds__(64 * NW) void gemm_direct_kernel(GemmSide<T> g, T alpha, T beta) {
  constexpr int BM = 16 * IM, BN = 16 * JN;
  typedef T t4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  __shared__ T red[NW][BN * BM];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int bx, bz;
  const bool placed = entry_place(bx, bz);
  if (bz >= g.nz) return;
  const int M = g.M, N = g.N, K = bz == g.nz - 1 ? g.Klast : g.K;
  const long lda = g.lda, ldb = g.ldb;
  const T* __restrict__ A = g.A + (long)bz * g.sA;
  const T* __restrict__ B = g.B + (long)bz * g.sB;
  T* __restrict__ C = g.C + (long)bz * g.sC;
  int tm, tn;
  if (!tile_coords_bounded(bx, (int)gridDim.x, g.tiles_m, g.tiles_n, tm, tn, placed)) return;
  const int m0 = tm * BM, n0 = tn * BN, fr = lane & 15, fk = lane >> 4;
  const T *Ap[IM], *Bp[JN];
#pragma unroll
  for (int i = 0; i < IM; ++i) Ap[i] = A + (long)min(m0 + 16 * i + fr, M - 1) * (TA ? lda : 1L);
#pragma unroll
  for (int j = 0; j < JN; ++j) Bp[j] = B + (long)min(n0 + 16 * j + fr, N - 1) * (TB ? 1L : ldb);
  T ra[2][IM][4], rb[2][JN][4];
  auto load = [&](int slot, int s) {
    const long k = 16L * s + 4 * fk;
#pragma unroll
    for (int i = 0; i < IM; ++i) {
      if constexpr (TA) {
        const t4 x = *reinterpret_cast<const t4*>(Ap[i] + k);
#pragma unroll
        for (int u = 0; u < 4; ++u) ra[slot][i][u] = x[u];
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) ra[slot][i][u] = Ap[i][(k + u) * lda];
      }
    }
#pragma unroll
    for (int j = 0; j < JN; ++j) {
      if constexpr (TB) {
#pragma unroll
        for (int u = 0; u < 4; ++u) rb[slot][j][u] = Bp[j][(k + u) * ldb];
      } else {
        const t4 x = *reinterpret_cast<const t4*>(Bp[j] + k);
#pragma unroll
        for (int u = 0; u < 4; ++u) rb[slot][j][u] = x[u];
      }
    }
  };
  typename Mfma<T>::acc acc[IM][JN];
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j) acc[i][j] = typename Mfma<T>::acc{0, 0, 0, 0};
  auto mma = [&](int slot) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j) acc[i][j] = Mfma<T>::op(rb[slot][j][u], ra[slot][i][u], acc[i][j]);
  };
  // this wavefront's full slabs: wave, wave + NW, ... below K / 16
  const int full = K / 16, mine = full > wave ? (full - wave + NW - 1) / NW : 0;
  if (mine > 0) load(0, wave);
  int it = 0;
  for (; it + 2 < mine; it += 2) {
    load(1, wave + (it + 1) * NW);
    mma(0);
    load(0, wave + (it + 2) * NW);
    mma(1);
  }
  if (mine - it == 2) {
    load(1, wave + (it + 1) * NW);
    mma(0);
    mma(1);
  } else if (mine - it == 1) {
    mma(0);
  }
  if (K > 16 * full && full % NW == wave) {  // the K tail, zero-padded
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int gk = 16 * full + 4 * fk + u;
      const long kc = min(gk, K - 1);
#pragma unroll
      for (int i = 0; i < IM; ++i) {
        const T x = Ap[i][TA ? kc : kc * lda];
        ra[0][i][u] = gk < K ? x : T(0);
      }
#pragma unroll
      for (int j = 0; j < JN; ++j) {
        const T x = Bp[j][TB ? kc * ldb : kc];
        rb[0][j][u] = gk < K ? x : T(0);
      }
    }
    mma(0);
  }
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[wave][(16 * j + Mfma<T>::row(lane, r)) * BM + 16 * i + fr] = acc[i][j][r];
  __syncthreads();
  for (int e = tid; e < BM * BN; e += 64 * NW) {
    double v = (double)red[0][e];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += (double)red[w][e];
    const int m = m0 + e % BM, n = n0 + e / BM;
    if (m < M && n < N) {
      const long off = (long)m + (long)n * g.ldc;
      v *= (double)alpha;
      if (beta != T(0)) v += (double)beta * (double)C[off];
      C[off] = (T)v;
    }
  }
}

template <typename T>
__global__ void scale_kernel(T* C, long M, long N, long ldc, T beta) {
  const long total = M * N;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const long m = e % M, n = e / M;
    C[m + n * ldc] = beta == T(0) ? T(0) : beta * C[m + n * ldc];
  }
}

// C = (sum of the parts of a TAIL launch's tile, in FP64 and in the order of its slabs) + beta C.  blockIdx.x: tile
// of the tail, blockIdx.y: 1024 of its 128 x 128 results, in the order of the workgroups' registers.  Bound by reading
// the parts.
template <typename T>
__global__ __launch_bounds__(256) void gemm_tail_kernel(GemmSide<T> g, T beta) {
  constexpr int BT = 128, NTH = sizeof(T) == 8 ? 512 : 256, NJ = sizeof(T) == 8 ? 2 : 4;
  const TailMap& tail = g.tail;
  int tm, tn, q = 3, first = 0;  // the tile's run and its parts' place
  tail.coords(tail.whole + (int)blockIdx.x, tm, tn);
  while (q > 0 && (int)blockIdx.x < tail.first_tile(q)) --q;
  if (tail.s[q] == 1) return;  // written by its workgroup
  for (int k = 1; k <= 3 && k != q; ++k) first += tail.n[k] * tail.s[k];
  const int t = (int)blockIdx.x - tail.first_tile(q);
  const int q0 = (int)blockIdx.y * 1024 + threadIdx.x;
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
  for (int c = 0; c < tail.s[q]; ++c) {
    const T* P = g.part + (long)(first + c * tail.n[q] + t) * (BT * BT) + q0;
#pragma unroll
    for (int u = 0; u < 4; ++u) sum[u] += (double)P[256 * u];
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int x = q0 + 256 * u, th = x % NTH, e = x / NTH, lane = th & 63, wm = (th >> 6) & 1, wn = th >> 7;
    const int i = e / (4 * NJ), j = e / 4 % NJ, r = e % 4;
    // (the wavefronts' blocks as in the kernels: in turn in FP32 and, in FP64, in tiles that some are missing from)
    const bool turn = sizeof(T) == 4 || g.M - tm * BT <= BT - 16 || g.N - tn * BT <= BT - 16;
    const int m = tm * BT + (turn ? (2 * i + wm) * 16 : wm * 64 + i * 16) + (lane & 15);
    const int n = tn * BT + (sizeof(T) == 8 ? (turn ? (4 * j + wn) * 16 : wn * 32 + j * 16) + (lane >> 4) + 4 * r
                                            : (2 * j + wn) * 16 + 4 * (lane >> 4) + r);
    if (m >= g.M || n >= g.N) continue;
    T* c = g.C + m + (long)n * g.ldc;
    *c = (T)(beta != T(0) ? sum[u] + (double)beta * (double)*c : sum[u]);
  }
}

// C = beta*C + sum_s W[s] (in FP64, fixed order), W[s] is M x N with leading dimension M.  Eight loads are in
// flight per thread: with one element per thread and a few hundred partial products (a 20 x 20 result
// of K = 200000) the sum is otherwise a chain of as many memory latencies.
template <typename T>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const T* __restrict__ W, int S, long M, long N,
                                                            T* __restrict__ C, long ldc, T beta) {
  const long total = M * N;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    double acc = 0.0;
    int q = 0;
    for (; q + 8 <= S; q += 8) {
      T w[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) w[u] = W[(long)(q + u) * total + e];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += (double)w[u];
    }
    for (; q < S; ++q) acc += (double)W[(long)q * total + e];
    const long m = e % M, n = e / M;
    const long off = m + n * ldc;
    if (beta != T(0)) acc += (double)beta * (double)C[off];
    C[off] = (T)acc;
  }
}

}  // namespace

// FP32 NN C = alpha A B + beta C for a short, wide product (M <= 64): a (16 IM)x256 tile over four
// wavefronts of (16 IM)x64 side by side (gemm32_nn_kernel's wavefront tile for IM = 4), four
// workgroups per CU.  K must be a multiple of 16.  Slices, swizzle and edge clamping as in
// gemm32_nn_kernel.
template <int IM>
__global__ __launch_bounds__(256, 4) void gemm32_sk_kernel(GemmSide<float> g, float alpha, float beta) {
  constexpr int BM = 16 * IM, BN = 256, BK = 16;
  __shared__ __attribute__((aligned(16))) float As[2][BM * BK];
  __shared__ __attribute__((aligned(16))) float Bs[2][BN * BK];
  const int tid = threadIdx.x, lane = tid & 63, wn = tid >> 6;
  const int M = g.M, N = g.N, K = g.K;
  const long lda = g.lda, ldb = g.ldb, ldc = g.ldc;
  const float* __restrict__ A = g.A + (long)blockIdx.z * g.sA;
  const float* __restrict__ B = g.B + (long)blockIdx.z * g.sB;
  float* __restrict__ C = g.C + (long)blockIdx.z * g.sC;
  int tm, tn;
  if (!tile_coords_bounded((int)blockIdx.x, (int)gridDim.x, g.tiles_m, g.tiles_n, tm, tn)) return;
  const int m0 = tm * BM, n0 = tn * BN;
  // A share: row am = lane (lanes below BM), 4-k chunk ac = wavefront; B share: rows bn + 64 j
  // (j < 4), 16-byte chunk bc
  const int am = lane, ac = __builtin_amdgcn_readfirstlane(wn);
  const bool a_share = lane < BM;
  const int bn = tid >> 2, bc = tid & 3;
  // A (at most 64 rows, L2-resident) is loaded one slice ahead.  B streams from HBM: for IM <= 3
  // it is loaded two slices ahead into two register stages, so that its loads have two slices of
  // MFMA work to arrive; IM = 4 has the registers for one stage.
  constexpr int NSB = IM <= 3 ? 2 : 1;
  float ra[4];
  f4v rb[NSB][4];
  const int a_voff = 4 * (min(m0 + am, M - 1) - m0);
  const int nlim = N - 1 - n0, ldbi = (int)ldb;
  const float* At = A + m0;
  const float* Bt = B + (long)n0 * ldb;
  auto load_a = [&](int k0) {
    if (a_share) {
      const auto rA = make_rsrc(At + (long)k0 * lda);
#pragma unroll
      for (int u = 0; u < 4; ++u) ra[u] = bload<float>(rA, a_voff, 4 * (4 * ac + u) * (int)lda);
    }
  };
  auto load_b = [&](int k0, f4v (&r)[4]) {
    const auto rB = make_rsrc(Bt + k0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      r[j] = __builtin_bit_cast(
          f4v, __builtin_amdgcn_raw_buffer_load_b128(rB, 4 * (4 * bc + min(bn + 64 * j, nlim) * ldbi), 0, 0));
  };
  auto store = [&](int buf, const f4v (&r)[4]) {
    if (a_share) *reinterpret_cast<f4v*>(&As[buf][am * BK + 4 * g32_chunk(ac, am)]) = f4v{ra[0], ra[1], ra[2], ra[3]};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = bn + 64 * j;
      *reinterpret_cast<f4v*>(&Bs[buf][n * BK + 4 * g32_chunk(bc, n)]) = r[j];
    }
  };

  fvec4 acc[IM][4];
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = fvec4{0, 0, 0, 0};
  const int fr = lane & 15, fk = lane >> 4;
  const int nk = K / BK;
  auto compute = [&](int cur) {
    f4v bf[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = wn * 64 + j * 16 + fr;
      bf[j] = *reinterpret_cast<const f4v*>(&Bs[cur][r * BK + 4 * g32_chunk(fk, r)]);
    }
#pragma unroll
    for (int i = 0; i < IM; ++i) {
      const int r = i * 16 + fr;
      const f4v a0 = *reinterpret_cast<const f4v*>(&As[cur][r * BK + 4 * g32_chunk(fk, r)]);
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[j][s2], a0[s2], acc[i][j], 0, 0, 0);
    }
  };
  if constexpr (NSB == 2) {
    // On entry to slice t (t even in the loop): LDS buffer 0 holds slice t, rb[1] holds slice
    // t + 1 (in flight) and rb[0] is free.  A is issued before B each time, so that waiting for A
    // leaves the newer B loads in flight.  Two slices per trip, so that the stages are named
    // statically; the last one to three slices are peeled off, so that the loop body has no
    // conditions.
    load_a(0);
    load_b(0, rb[0]);
    if (nk > 1) load_b(BK, rb[1]);
    store(0, rb[0]);
    __syncthreads();
    int t = 0;
    for (; t + 3 < nk; t += 2) {
      load_a((t + 1) * BK);
      load_b((t + 2) * BK, rb[0]);
      compute(0);
      store(1, rb[1]);
      __syncthreads();
      load_a((t + 2) * BK);
      load_b((t + 3) * BK, rb[1]);
      compute(1);
      store(0, rb[0]);
      __syncthreads();
    }
    if (t + 1 < nk) load_a((t + 1) * BK);
    if (t + 2 < nk) load_b((t + 2) * BK, rb[0]);
    compute(0);
    if (t + 1 < nk) {
      store(1, rb[1]);
      __syncthreads();
      if (t + 2 < nk) load_a((t + 2) * BK);
      compute(1);
      if (t + 2 < nk) {
        store(0, rb[0]);
        __syncthreads();
        compute(0);
      }
    }
  } else {
    load_a(0);
    load_b(0, rb[0]);
    store(0, rb[0]);
    __syncthreads();
    // the last slice is peeled off, so that the loop body is one block without conditions
    for (int kt = 0; kt + 1 < nk; ++kt) {
      const int cur = kt & 1;
      load_a((kt + 1) * BK);
      load_b((kt + 1) * BK, rb[0]);
      compute(cur);
      store(cur ^ 1, rb[0]);
      __syncthreads();
    }
    compute((nk - 1) & 1);
  }

#pragma unroll
  for (int i = 0; i < IM; ++i) {
    const int m = m0 + i * 16 + fr;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + wn * 64 + j * 16 + 4 * fk + r;
        if (n < N) {
          const long off = (long)m + (long)n * ldc;
          float v = alpha * acc[i][j][r];
          if (beta != 0.f) v += beta * C[off];
          C[off] = v;
        }
      }
    }
  }
}

// FP64 NN C = alpha A B + beta C for a short, wide product (M <= 64, e.g. the first quarter
// of the AO->MO transform, M = o): a (16 IM)x256 tile over eight wavefronts of (16 IM)x32 side by
// side (the FP64 kernel's wavefront tile for IM = 4), two workgroups per CU.  K must be a
// multiple of 16.  Slices, swizzle and edge clamping as in gemm64_kernel.
template <int IM>
__global__ __launch_bounds__(512, 4) void gemm64_sk_kernel(GemmSide<double> g, double alpha, double beta) {
  constexpr int BM = 16 * IM, BN = 256, BK = 16;
  __shared__ __attribute__((aligned(16))) double As[2][BM * BK];
  __shared__ __attribute__((aligned(16))) double Bs[2][BN * BK];
  const int tid = threadIdx.x, lane = tid & 63, wn = tid >> 6;
  const int M = g.M, N = g.N, K = g.K;
  const long lda = g.lda, ldb = g.ldb, ldc = g.ldc;
  const double* __restrict__ A = g.A + (long)blockIdx.z * g.sA;
  const double* __restrict__ B = g.B + (long)blockIdx.z * g.sB;
  double* __restrict__ C = g.C + (long)blockIdx.z * g.sC;
  int tm, tn;
  if (!tile_coords_bounded((int)blockIdx.x, (int)gridDim.x, g.tiles_m, g.tiles_n, tm, tn)) return;
  const int m0 = tm * BM, n0 = tn * BN;
  // A share: row am = lane (lanes below BM), 16-byte chunk ka = wavefront (k = 2 ka, 2 ka + 1);
  // B share: rows bn + 64 j, chunk bc
  const int am = lane, ka = __builtin_amdgcn_readfirstlane(wn);
  const bool a_share = lane < BM;
  const int bn = tid >> 3, bc = tid & 7;
  // A (at most 64 rows, L2-resident) is loaded one slice ahead.  B streams from HBM: for IM <= 3
  // it is loaded two slices ahead into two register stages, so that its loads have two slices of
  // MFMA work to arrive (K is short in these products); IM = 4 has the registers for one stage.
  constexpr int NSB = IM <= 3 ? 2 : 1;
  double ra[2];
  d2v rb[NSB][4];
  const int a_voff = 8 * (min(m0 + am, M - 1) - m0);
  // B rows past N load row N - 1 (uniform limit; the offsets are recomputed per load rather
  // than held in registers)
  const int nlim = N - 1 - n0, ldbi = (int)ldb;
  const double* At = A + m0;
  const double* Bt = B + (long)n0 * ldb;
  auto load_a = [&](int k0) {
    if (a_share) {
      const auto rA = make_rsrc(At + (long)k0 * lda);
#pragma unroll
      for (int u = 0; u < 2; ++u) ra[u] = bload<double>(rA, a_voff, 8 * (2 * ka + u) * (int)lda);
    }
  };
  auto load_b = [&](int k0, d2v (&r)[4]) {
    const auto rB = make_rsrc(Bt + k0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      r[j] = __builtin_bit_cast(
          d2v, __builtin_amdgcn_raw_buffer_load_b128(rB, 8 * (2 * bc + min(bn + 64 * j, nlim) * ldbi), 0, 0));
  };
  auto store = [&](int buf, const d2v (&r)[4]) {
    if (a_share) *reinterpret_cast<d2v*>(&As[buf][am * BK + 2 * g64_chunk(ka, am)]) = d2v{ra[0], ra[1]};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = bn + 64 * j;
      *reinterpret_cast<d2v*>(&Bs[buf][n * BK + 2 * g64_chunk(bc, n)]) = r[j];
    }
  };

  dvec4 acc[IM][2];
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = dvec4{0, 0, 0, 0};
  const int fr = lane & 15, fk = lane >> 4;
  const int nk = K / BK;
  auto compute = [&](int cur) {
    d2v bf[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = wn * 32 + j * 16 + fr;
      bf[j][0] = *reinterpret_cast<const d2v*>(&Bs[cur][r * BK + 2 * g64_chunk(2 * fk, r)]);
      bf[j][1] = *reinterpret_cast<const d2v*>(&Bs[cur][r * BK + 2 * g64_chunk(2 * fk + 1, r)]);
    }
    // (A's fragments are read as they are used: with four wavefronts per SIMD the LDS latency
    // is hidden, and the registers a one-ahead copy would take are not there)
#pragma unroll
    for (int i = 0; i < IM; ++i) {
      const int r = i * 16 + fr;
      d2v a0[2];
      a0[0] = *reinterpret_cast<const d2v*>(&As[cur][r * BK + 2 * g64_chunk(2 * fk, r)]);
      a0[1] = *reinterpret_cast<const d2v*>(&As[cur][r * BK + 2 * g64_chunk(2 * fk + 1, r)]);
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf[j][s2 >> 1][s2 & 1], a0[s2 >> 1][s2 & 1], acc[i][j],
                                                           0, 0, 0);
    }
  };
  if constexpr (NSB == 2) {
    // On entry to slice t (t even in the loop): LDS buffer 0 holds slice t, rb[1] holds slice
    // t + 1 (in flight) and rb[0] is free.  A is issued before B each time, so that waiting for A
    // leaves the newer B loads in flight.  Two slices per trip, so that the stages are named
    // statically; the last one to three slices are peeled off, so that the loop body has no
    // conditions.
    load_a(0);
    load_b(0, rb[0]);
    if (nk > 1) load_b(BK, rb[1]);
    store(0, rb[0]);
    __syncthreads();
    int t = 0;
    for (; t + 3 < nk; t += 2) {
      load_a((t + 1) * BK);
      load_b((t + 2) * BK, rb[0]);
      compute(0);
      store(1, rb[1]);
      __syncthreads();
      load_a((t + 2) * BK);
      load_b((t + 3) * BK, rb[1]);
      compute(1);
      store(0, rb[0]);
      __syncthreads();
    }
    if (t + 1 < nk) load_a((t + 1) * BK);
    if (t + 2 < nk) load_b((t + 2) * BK, rb[0]);
    compute(0);
    if (t + 1 < nk) {
      store(1, rb[1]);
      __syncthreads();
      if (t + 2 < nk) load_a((t + 2) * BK);
      compute(1);
      if (t + 2 < nk) {
        store(0, rb[0]);
        __syncthreads();
        compute(0);
      }
    }
  } else {
    load_a(0);
    load_b(0, rb[0]);
    store(0, rb[0]);
    __syncthreads();
    // the last slice is peeled off, so that the loop body is one block without conditions
    for (int kt = 0; kt + 1 < nk; ++kt) {
      const int cur = kt & 1;
      load_a((kt + 1) * BK);
      load_b((kt + 1) * BK, rb[0]);
      compute(cur);
      store(cur ^ 1, rb[0]);
      __syncthreads();
    }
    compute((nk - 1) & 1);
  }

  // acc[i][j][r]: C(m, n) with m = 16 i + lane % 16, n = n0 + 32 wn + 16 j + lane / 16 + 4 r
#pragma unroll
  for (int i = 0; i < IM; ++i) {
    const int m = m0 + i * 16 + fr;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + wn * 32 + j * 16 + fk + 4 * r;
        if (n < N) {
          const long off = (long)m + (long)n * ldc;
          double v = alpha * acc[i][j][r];
          if (beta != 0.0) v += beta * C[off];
          C[off] = v;
        }
      }
    }
  }
}

// FP64 NN C = alpha A B + beta C for a tall, narrow product (N <= 64, M large, e.g. the MP2
// adjoint's g Co half-transform step, N = o): a 256x(16 IN) tile over eight wavefronts of
// 32x(16 IN) stacked in m, two workgroups per CU.  A (m-contiguous, the streamed operand) is
// staged as in gemm64_kernel, B (k-contiguous, at most 64 rows) as gemm64_sk_kernel's B.
// K must be a multiple of 16.
template <int IN>
__global__ __launch_bounds__(512, 4) void gemm64_tall_kernel(GemmSide<double> g, double alpha, double beta) {
  constexpr int BM = 256, BN = 16 * IN, BK = 16;
  __shared__ __attribute__((aligned(16))) double As[2][BM * BK];
  __shared__ __attribute__((aligned(16))) double Bs[2][BN * BK];
  const int tid = threadIdx.x, lane = tid & 63, wm = tid >> 6;
  const int M = g.M, N = g.N, K = g.K;
  const long lda = g.lda, ldb = g.ldb, ldc = g.ldc;
  const double* __restrict__ A = g.A + (long)blockIdx.z * g.sA;
  const double* __restrict__ B = g.B + (long)blockIdx.z * g.sB;
  double* __restrict__ C = g.C + (long)blockIdx.z * g.sC;
  int tm, tn;
  if (!tile_coords_bounded((int)blockIdx.x, (int)gridDim.x, g.tiles_m, g.tiles_n, tm, tn)) return;
  const int m0 = tm * BM, n0 = tn * BN;
  // A share: row am, k = 8 kq + u (u = 0..7); B share (threads below 8 BN): row bn, 16-byte chunk bc
  const int am = tid & 255, kq = __builtin_amdgcn_readfirstlane(tid >> 8);
  const int bn = tid >> 3, bc = tid & 7;
  const bool b_share = tid < 8 * BN;
  double ra[8];
  d2v rb;
  const int a_voff = 8 * (min(m0 + am, M - 1) - m0);
  const int b_voff = 8 * (2 * bc + (min(n0 + bn, N - 1) - n0) * (int)ldb);
  auto load = [&](int k0) {
    const auto rA = make_rsrc(A + m0 + (long)k0 * lda);
#pragma unroll
    for (int u = 0; u < 8; ++u) ra[u] = bload<double>(rA, a_voff, 8 * (8 * kq + u) * (int)lda);
    if (b_share) {
      const auto rB = make_rsrc(B + k0 + (long)n0 * ldb);
      rb = __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(rB, b_voff, 0, 0));
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<d2v*>(&As[buf][am * BK + 2 * g64_chunk(4 * kq + q, am)]) = d2v{ra[2 * q], ra[2 * q + 1]};
    if (b_share) *reinterpret_cast<d2v*>(&Bs[buf][bn * BK + 2 * g64_chunk(bc, bn)]) = rb;
  };

  dvec4 acc[2][IN];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < IN; ++j) acc[i][j] = dvec4{0, 0, 0, 0};
  const int fr = lane & 15, fk = lane >> 4;
  const int nk = K / BK;
  load(0);
  store(0);
  __syncthreads();
  // the last slice is peeled off, so that the loop body is one block without conditions
  auto compute = [&](int cur) {
    // A's two blocks are held for the slice, B's blocks streamed one ahead of their MFMAs (for
    // IN = 4 read as they are used: the one-ahead copy would not fit in 128 VGPRs)
    constexpr bool ahead = IN < 4;
    d2v af[2][2], b0[2], b1[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = wm * 32 + i * 16 + fr;
      af[i][0] = *reinterpret_cast<const d2v*>(&As[cur][r * BK + 2 * g64_chunk(2 * fk, r)]);
      af[i][1] = *reinterpret_cast<const d2v*>(&As[cur][r * BK + 2 * g64_chunk(2 * fk + 1, r)]);
    }
    if (ahead) {
      b0[0] = *reinterpret_cast<const d2v*>(&Bs[cur][fr * BK + 2 * g64_chunk(2 * fk, fr)]);
      b0[1] = *reinterpret_cast<const d2v*>(&Bs[cur][fr * BK + 2 * g64_chunk(2 * fk + 1, fr)]);
    }
#pragma unroll
    for (int j = 0; j < IN; ++j) {
      if (!ahead) {
        const int r = j * 16 + fr;
        b0[0] = *reinterpret_cast<const d2v*>(&Bs[cur][r * BK + 2 * g64_chunk(2 * fk, r)]);
        b0[1] = *reinterpret_cast<const d2v*>(&Bs[cur][r * BK + 2 * g64_chunk(2 * fk + 1, r)]);
      } else if (j + 1 < IN) {
        const int r = (j + 1) * 16 + fr;
        b1[0] = *reinterpret_cast<const d2v*>(&Bs[cur][r * BK + 2 * g64_chunk(2 * fk, r)]);
        b1[1] = *reinterpret_cast<const d2v*>(&Bs[cur][r * BK + 2 * g64_chunk(2 * fk + 1, r)]);
      }
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b0[s2 >> 1][s2 & 1], af[i][s2 >> 1][s2 & 1], acc[i][j],
                                                           0, 0, 0);
      if (ahead && j + 1 < IN) { b0[0] = b1[0]; b0[1] = b1[1]; }
    }
  };
  for (int kt = 0; kt + 1 < nk; ++kt) {
    const int cur = kt & 1;
    load((kt + 1) * BK);
    compute(cur);
    store(cur ^ 1);
    __syncthreads();
  }
  compute((nk - 1) & 1);

  // acc[i][j][r]: C(m, n) with m = m0 + 32 wm + 16 i + lane % 16, n = n0 + 16 j + lane / 16 + 4 r
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + wm * 32 + i * 16 + fr;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < IN; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + j * 16 + fk + 4 * r;
        if (n < N) {
          const long off = (long)m + (long)n * ldc;
          double v = alpha * acc[i][j][r];
          if (beta != 0.0) v += beta * C[off];
          C[off] = v;
        }
      }
    }
  }
}

// FP32 NN C = alpha A B + beta C for a tall, narrow product (N <= 64, M large): a 256x(16 IN) tile over
// four wavefronts of 64x(16 IN) stacked in m, four workgroups per CU.  A (m-contiguous) is staged as in
// gemm32_nn_kernel, each thread holding one row's four 16-byte k-chunks; B (k-contiguous, at most 64
// rows) as gemm32_nn_kernel's B.  K must be a multiple of 16.
template <int IN>
__global__ __launch_bounds__(256, 4) void gemm32_tall_kernel(GemmSide<float> g, float alpha, float beta) {
  constexpr int BM = 256, BN = 16 * IN, BK = 16;
  __shared__ __attribute__((aligned(16))) float As[2][BM * BK];
  __shared__ __attribute__((aligned(16))) float Bs[2][BN * BK];
  const int tid = threadIdx.x, lane = tid & 63, wm = tid >> 6;
  const int M = g.M, N = g.N, K = g.K;
  const long lda = g.lda, ldb = g.ldb, ldc = g.ldc;
  const float* __restrict__ A = g.A + (long)blockIdx.z * g.sA;
  const float* __restrict__ B = g.B + (long)blockIdx.z * g.sB;
  float* __restrict__ C = g.C + (long)blockIdx.z * g.sC;
  int tm, tn;
  if (!tile_coords_bounded((int)blockIdx.x, (int)gridDim.x, g.tiles_m, g.tiles_n, tm, tn)) return;
  const int m0 = tm * BM, n0 = tn * BN;
  // A share: row am = tid, k = 4 c + u (c, u = 0..3); B share (threads below 4 BN): row bn, chunk bc
  const int am = tid;
  const int bn = tid >> 2, bc = tid & 3;
  const bool b_share = tid < 4 * BN;
  float ra[16];
  f4v rb;
  const int a_voff = 4 * (min(m0 + am, M - 1) - m0);
  const int b_voff = 4 * (4 * bc + (min(n0 + bn, N - 1) - n0) * (int)ldb);
  auto load = [&](int k0) {
    const auto rA = make_rsrc(A + m0 + (long)k0 * lda);
#pragma unroll
    for (int q = 0; q < 16; ++q) ra[q] = bload<float>(rA, a_voff, 4 * q * (int)lda);
    if (b_share) {
      const auto rB = make_rsrc(B + k0 + (long)n0 * ldb);
      rb = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rB, b_voff, 0, 0));
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      *reinterpret_cast<f4v*>(&As[buf][am * BK + 4 * g32_chunk(c, am)]) =
          f4v{ra[4 * c], ra[4 * c + 1], ra[4 * c + 2], ra[4 * c + 3]};
    if (b_share) *reinterpret_cast<f4v*>(&Bs[buf][bn * BK + 4 * g32_chunk(bc, bn)]) = rb;
  };

  fvec4 acc[4][IN];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < IN; ++j) acc[i][j] = fvec4{0, 0, 0, 0};
  const int fr = lane & 15, fk = lane >> 4;
  const int nk = K / BK;
  load(0);
  store(0);
  __syncthreads();
  // B's blocks are held for the slice, A's streamed one ahead of their MFMAs
  auto compute = [&](int cur) {
    f4v bf[IN];
#pragma unroll
    for (int j = 0; j < IN; ++j) {
      const int r = j * 16 + fr;
      bf[j] = *reinterpret_cast<const f4v*>(&Bs[cur][r * BK + 4 * g32_chunk(fk, r)]);
    }
    f4v a0 = *reinterpret_cast<const f4v*>(&As[cur][(wm * 64 + fr) * BK + 4 * g32_chunk(fk, wm * 64 + fr)]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f4v a1;
      if (i + 1 < 4) {
        const int r = wm * 64 + (i + 1) * 16 + fr;
        a1 = *reinterpret_cast<const f4v*>(&As[cur][r * BK + 4 * g32_chunk(fk, r)]);
      }
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
        for (int j = 0; j < IN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[j][s2], a0[s2], acc[i][j], 0, 0, 0);
      if (i + 1 < 4) a0 = a1;
    }
  };
  // the last slice is peeled off, so that the loop body is one block without conditions
  for (int kt = 0; kt + 1 < nk; ++kt) {
    const int cur = kt & 1;
    load((kt + 1) * BK);
    compute(cur);
    store(cur ^ 1);
    __syncthreads();
  }
  compute((nk - 1) & 1);

  // acc[i][j][r]: C(m, n) with m = m0 + 64 wm + 16 i + lane % 16, n = n0 + 16 j + 4 (lane / 16) + r
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + wm * 64 + i * 16 + fr;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < IN; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + j * 16 + 4 * fk + r;
        if (n < N) {
          const long off = (long)m + (long)n * ldc;
          float v = alpha * acc[i][j][r];
          if (beta != 0.f) v += beta * C[off];
          C[off] = v;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// dispatch
// ---------------------------------------------------------------------------
// Kernel forms of one product.  TILE128 / TILE64: the LDS-staged kernels with 128x128 / 64x64 tiles;
// SHORT / TALL: their 48 or 64 by 256 tiles for M <= 64 / N <= 64 (NN only); the DIRECT forms:
// gemm_direct_kernel with 32x32, 32x16, 16x32 (four wavefronts) and 16x16 tiles (eight).
enum GemmForm { TILE128, TILE64, SHORT, TALL, DIRECT22, DIRECT21, DIRECT12, DIRECT11, GEMM_FORMS };

struct GemmPlan {
  int form = DIRECT22;
  long split = 1;   // chunks of the contraction, each a launch-z entry with its own partial product
  TailMap tail;     // wgs > 0: a TAIL launch of 128x128 tiles
  double us = 1e300;
  long chain = 0;   // the longest sum over k in one accumulator
};

static inline long cdiv(long a, long b) { return (a + b - 1) / b; }

// gridDim.z of a launch of nz entries of `tiles` workgroups (entry_place); at most 65528 entries.  Not padded where the
// XCDs' shares would differ too much: in FP32, 17 chunks of 600 x 1500 x 20000 take 483 us in three entries for some XCDs
// and two for others, 361 dealt tile by tile; 15 chunks of 2800 x 1500 x 33600, each more than an XCD holds at once, 2.77
// and 2.57 ms.
static inline unsigned grid_z(int nz, long tiles) {
  const long padded = cdiv(nz, NXCD) * NXCD;
  const bool even = 3 * padded <= 4L * nz && (tiles <= 128 || 16 * padded <= 17L * nz);
  return (unsigned)(nz >= NXCD && even ? padded : nz);
}

static void form_tile(int form, long M, long N, long& bm, long& bn) {
  switch (form) {
    case TILE128: bm = bn = 128; break;
    case TILE64: bm = bn = 64; break;
    case SHORT: bm = M <= 48 ? 48 : 64; bn = 256; break;
    case TALL: bm = 256; bn = N <= 48 ? 48 : 64; break;
    case DIRECT22: bm = bn = 32; break;
    case DIRECT21: bm = 32; bn = 16; break;
    case DIRECT12: bm = 16; bn = 32; break;
    default: bm = bn = 16; break;
  }
}

// Whether a form takes the product.  The LDS-staged kernels address a tile's k-slice with 32-bit byte
// offsets from one buffer base: an m-contiguous A (n-contiguous B) spans 16 columns of lda (ldb), a
// k-contiguous operand the tile's rows of it (in the 128-row TN / TT instantiations 64 rows from each
// of two bases).  The direct kernel addresses with 64 bits and takes everything.
template <typename T>
static bool form_ok(int form, bool ta, bool tb, long M, long N, long K, long lda, long ldb) {
  const auto fits = [](long rows, long ld) { return (long)sizeof(T) * rows * (ld + 1) < (1L << 31); };
  switch (form) {
    case TILE128:
    case TILE64: {
      const long rows = form == TILE128 && !ta ? 128 : 64;
      return fits(ta ? rows : 16, lda) && fits(tb ? 16 : rows, ldb);
    }
    case SHORT: return M <= 64 && !ta && !tb && K % 16 == 0 && fits(256 + 64, std::max(lda, ldb));
    case TALL: return N <= 64 && !ta && !tb && K % 16 == 0 && fits(16, lda) && fits(64, ldb);
    default: return true;
  }
}

// Estimated time (us) of `products` tiles-sets sharing one launch: tiles workgroups in all, each
// walking `slabs` 16-deep k-slabs.  Per compute unit the larger of three times: the workgroups' k-loops one
// after another at the kernel's reach of the MFMA rate (a 16x16 block of a slab is 0.107 us of one SIMD's
// FP64 pipe, half that in FP32), one workgroup's own latency-bound loop, and for the direct kernel, whose
// wavefronts share nothing, the cache traffic of its fragments; over the chip the traffic from HBM
// (`bytes`).  The constants are fitted to measurements of all forms over 62 shapes (95^3 to 8640^2 x 768,
// M = 1 vectors, 34 x 34 x 1227400, batches of 20 x 108 x 128; FP64 and FP32): the form picked is on
// average 2% from the best measured one.
template <typename T>
static double form_us(int form, long tiles, long slabs, double bytes) {
  const double f = sizeof(T) == 8 ? 1.0 : 0.5;
  const double cu = (double)cdiv(tiles, 256);  // workgroups per compute unit
  const double hbm = bytes / 5.6e6;
  switch (form) {
    case TILE128: return 8.5 + std::max(hbm, (slabs + 1) * std::max(f == 1.0 ? 2.5 : 1.4, cu * 1.71 * f / 0.86));
    case TILE64: {
      // twice TILE128's operand traffic: at 8.4 TB/s from the L2s it is what bounds a 6460^3 FP64 product
      // (9.0 ms; 7.7 with 128x128 tiles)
      const double cache = (double)tiles * slabs * 2048.0 * sizeof(T) / 8.4e6;
      return 7.0 + std::max(std::max(hbm, cache), (slabs + 1) * std::max(f == 1.0 ? 0.8 : 0.72, cu * 0.427 * f / (f == 1.0 ? 0.8 : 0.85)));
    }
    case SHORT:
    case TALL: return 8.0 + std::max(hbm, (slabs + 1) * std::max(1.6 * f, cu * 1.28 * f / 0.75));
    default: {
      const int nw = form == DIRECT11 ? 8 : 4, blocks = form == DIRECT22 ? 4 : form == DIRECT11 ? 1 : 2;
      const int sides = form == DIRECT22 ? 4 : form == DIRECT11 ? 2 : 3;
      const double L = (double)cdiv(slabs, nw), m = 0.107 * blocks * f;
      const double resident = (form == DIRECT22 ? 3.0 : 4.0) * 4 / nw;
      const double own = L * (0.2 + 0.025 * sides + m) * std::max(1.0, cu / resident);
      const double mfma = cu * nw * L * m / 4 / 0.55;
      const double cache = (double)tiles * nw * L * 256.0 * sides * sizeof(T) / 9.0e6;
      return 3.0 + std::max(std::max(own, hbm), std::max(mfma, cache));
    }
  }
}

// time of adding S partial products of `elems` elements (splitk_reduce_kernel)
template <typename T>
static double reduce_us(long S, double elems) {
  return S > 1 ? 2.0 + (S + 1) * elems * sizeof(T) / 4.5e6 + 0.18 * S : 0.0;
}

// 128x128 tiles: 2 x 4 wavefronts of 64x32 in FP64, 2 x 2 of 64x64 in FP32
template <typename T>
constexpr TailShape kTail{128, 128, 2, sizeof(T) == 8 ? 4 : 2, 16, 0.375, 8};

// Estimated time (us) of a TAIL launch: a compute unit's slabs, and 2.5 for each workgroup's start and end, at the
// rate that a long launch of 128x128 tiles reaches (1.87 us in FP64, 0.94 in FP32; more where few workgroups
// share a unit), but at least the latency of each slab of the longest chunk; and the parts, written and read once.
template <typename T>
static double tail_us(const TailMap& t) {
  constexpr bool dp = sizeof(T) == 8;
  int tiles = 0, least = 1 << 30;
  for (int q = 0; q < 4; ++q) {
    tiles += t.n[q];
    if (t.n[q]) least = std::min(least, t.s[q]);
  }
  const int chunks = t.n[0] ? t.s[0] : least;
  const double rounds = (double)cdiv(t.wgs, 256);
  const double slabs = t.whole / 256 * (t.nk + 2.5) + rounds * ((double)t.nk / chunks + 2.5);
  // (an FP32 unit holds four workgroups)
  const double latency = (dp ? 0.88 : 1.2) * (t.nk * (t.whole / (dp ? 256 : 1024) + 1.0 / least) + 2.5);
  const long each = cdiv(t.whole + t.wgs, 256);
  const double few = dp ? (each == 1 ? 1.08 : 1.0) : (each == 1 ? 1.3 : each == 2 ? 1.12 : each == 3 ? 1.05 : 1.0);
  const double parts = t.wgs > tiles ? (2.0 * t.wgs + tiles) * 16384.0 * sizeof(T) / 6.0e6 + 5.0 : 0.0;
  return 11.0 + (dp ? 1.87 : 0.94) * std::max(slabs, latency) * few + parts;
}

static const long kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128};

// The longest sum over k that an accumulator of an FP32 product may form before it is added to others in FP64: the error
// of a long product is that of its accumulators' FP32 sums (it grows as the root of their length: 5.7e-7 of sqrt(K) at
// 1024, 2.5e-6 at 20000), so a form that is faster without splitting K does not give this up.  Products of few 128x128
// tiles get chunks of 1024 and longer ones that make a round of four workgroups a compute unit; long ones of more tiles
// the fewest chunks that fill the rounds; others may sum all of K.
static long chain_limit(long M, long N, long K) {
  if (K < 4096) return K;
  const bool wide = M <= 64 && N >= 8192, tall = N <= 64 && M >= 8192;
  const long tiles = cdiv(M, wide ? 64 : tall ? 256 : 128) * cdiv(N, wide ? 256 : tall ? 64 : 128);
  long S = 1;
  if (tiles < 128) {
    S = std::max(2L, std::min(K / 1024, 1024 / tiles));
  } else if (!wide && !tall && K >= 32768) {
    const auto fill = [&](long s) { return (double)(tiles * s) / (double)(cdiv(tiles * s, 1024) * 1024); };
    for (long s = 2; s <= 16 && fill(1) < 0.8; ++s)
      if (fill(s) > fill(S) + 0.02 && 4.0 * s * M * N <= 2147483648.0) S = s;
  }
  return cdiv(cdiv(K, S), 32) * 32;
}

// The form and split with the smallest estimated time, in FP32 within chain_limit where the splits allow it.  A
// split product's partial results take at most 256 MiB of workspace, 2 GiB when K >= 32768 (RCCSD's o^2 x v.m x v^2
// products over (ia|bc)).
template <typename T>
static GemmPlan gemm_plan(bool ta, bool tb, long M, long N, long K, long lda, long ldb, long sA, long sB, int batch,
                          bool allow_split, bool limited = true) {
  GemmPlan best;
  const long limit = sizeof(T) == 4 && limited && allow_split && batch == 1 ? chain_limit(M, N, K) : K;
  const double bytes = (double)sizeof(T) * ((double)M * K * (sA || batch == 1 ? batch : 1) +
                                            (double)N * K * (sB || batch == 1 ? batch : 1) + (double)M * N * batch);
  const double room = K >= 32768 ? 2147483648.0 : 268435456.0;
  for (int form = 0; form < GEMM_FORMS; ++form) {
    // a transposed short A (the transform's orbital block) is transposed first for SHORT
    const bool copy_a = form == SHORT && ta && !tb && lda == K && batch == 1 && allow_split;
    if (!form_ok<T>(form, copy_a ? false : ta, tb, M, N, K, copy_a ? M : lda, ldb)) continue;
    long bm, bn;
    form_tile(form, M, N, bm, bn);
    const long tiles = cdiv(M, bm) * cdiv(N, bn);
    if (tiles >= (1L << 31)) continue;
    // (operands past the caches' sizes: 4200 x 1500 x 33600 in five chunks takes 4.26 ms with 64x64 tiles, 3.89 with 128x128)
    if (form == TILE64 && limit < K && K >= 32768 && tiles >= 512 && form_ok<T>(TILE128, ta, tb, M, N, K, lda, ldb)) continue;
    const long parts = limit < K ? cdiv(K, limit) : 1;  // the split that the limit comes from, too
    for (int q = parts > 1 ? -1 : 0; q < (int)(sizeof(kSplits) / sizeof(kSplits[0])); ++q) {
      const long s = q < 0 ? parts : kSplits[q];
      if (s > 1 && (!allow_split || batch > 1 || K < 64 * s || tiles * s > 8192 || form == SHORT || form == TALL ||
                    (double)s * M * N * sizeof(T) > room)) {
        if (q < 0) continue;
        break;
      }
      const long slabs = cdiv(cdiv(K, s), 16);
      const long chain = 16 * (form < DIRECT22 ? slabs : cdiv(slabs, form == DIRECT11 ? 8 : 4));
      if (limit < K && chain > limit) continue;
      const double us = form_us<T>(form, tiles * s * batch, slabs, bytes) + reduce_us<T>(s, (double)M * N) +
                        (copy_a ? 6.0 : 0.0);
      if (us < best.us) best = GemmPlan{form, s, TailMap{}, us, chain};
    }
  }
  if (allow_split && batch == 1 && form_ok<T>(TILE128, ta, tb, M, N, K, lda, ldb)) {
    const long full = (M / 128) * (N / 128) / 256 * 256;
    for (const long whole : {full, full - 256})
      for (int chunks = 1; whole >= 0 && chunks <= 32; ++chunks) {
        const TailMap t = tail_map(kTail<T>, M, N, K, whole, chunks);
        if (!t.wgs || t.wgs == t.n[0] + t.n[1] + t.n[2] + t.n[3]) continue;  // (nothing shared: the plain launch)
        const long chain = tail_chain(t, 16);
        if (limit < K && chain > limit) continue;
        const double us = tail_us<T>(t);
        if (us < best.us) best = GemmPlan{TILE128, 1, t, us, chain};
      }
  }
  if (best.us >= 1e300 && limit < K)
    return gemm_plan<T>(ta, tb, M, N, K, lda, ldb, sA, sB, batch, allow_split, false);
  return best;
}

template <typename T>
static GemmSide<T> make_side(long M, long N, long K, const T* A, long lda, long sA, const T* B, long ldb, long sB,
                             T* C, long ldc, long sC, int form = TILE128) {
  long bm, bn;
  form_tile(form, M, N, bm, bn);
  return GemmSide<T>{A, B, C, lda, ldb, ldc, sA, sB, sC, (int)M, (int)N, (int)K, (int)cdiv(M, bm),
                     (int)cdiv(N, bn), (int)K, nullptr, nullptr, 0};
}

// One launch of the LDS-staged kernel with 128x128 or 64x64 tiles over p0 (and p1 when `two`), nb batch
// entries.  The ring and ladder symbols (kind 1 and 2) exist for the 128x128 NN kernels.
template <typename T>
static void tile_launch(jues_ctx* ctx, int form, bool tb, int kind, GemmSide<T> p0, GemmSide<T> p1, bool two, int nb,
                        T alpha, T beta, bool ta = false, bool seg = false) {
  const long t0 = (long)p0.tiles_m * p0.tiles_n;
  const long nt0 = two ? (t0 + NXCD - 1) / NXCD * NXCD : t0;
  const long total = two ? nt0 + (long)p1.tiles_m * p1.tiles_n : t0;
  JUES_REQUIRE(total < (1L << 31), "gemm: too many tiles");
  p0.nz = p1.nz = nb;
  if (!two) p1 = p0;
  const bool tail = p0.tail.wgs > 0;
  const dim3 grid((unsigned)(tail ? p0.tail.whole + p0.tail.wgs : total), 1, grid_z(nb, total));
  if constexpr (sizeof(T) == 4) {
#define JUES_GEMM32(K_, TB_, TA_, SEG_, BT_, ...)                                                                   \
  hipLaunchKernelGGL((gemm32_nn_kernel<K_, TB_, TA_, SEG_, false, BT_, ##__VA_ARGS__>), grid, dim3(NT), 0,          \
                     ctx->stream, p0, p1, (int)nt0, (float)alpha, (float)beta)
#define JUES_GEMM32_TAIL(K_, TB_, TA_) JUES_GEMM32(K_, TB_, TA_, false, 128, true)
#define JUES_GEMM32_SHAPES(BT_)                      \
  if (seg) {                                         \
    if (tb) JUES_GEMM32(0, true, false, true, BT_);  \
    else JUES_GEMM32(0, false, false, true, BT_);    \
  } else if (ta) {                                   \
    if (tb) JUES_GEMM32(0, true, true, false, BT_);  \
    else JUES_GEMM32(0, false, true, false, BT_);    \
  } else if (tb) JUES_GEMM32(0, true, false, false, BT_)
    if (tail) {
      if (ta && tb) JUES_GEMM32_TAIL(0, true, true);
      else if (ta) JUES_GEMM32_TAIL(0, false, true);
      else if (tb) JUES_GEMM32_TAIL(0, true, false);
      else if (kind == 1) JUES_GEMM32_TAIL(1, false, false);
      else if (kind == 2) JUES_GEMM32_TAIL(2, false, false);
      else JUES_GEMM32_TAIL(0, false, false);
    } else if (form == TILE64) {
      JUES_GEMM32_SHAPES(64);
      else JUES_GEMM32(0, false, false, false, 64);
    } else {
      JUES_GEMM32_SHAPES(128);
      else if (kind == 1) JUES_GEMM32(1, false, false, false, 128);
      else if (kind == 2) JUES_GEMM32(2, false, false, false, 128);
      else JUES_GEMM32(0, false, false, false, 128);
    }
#undef JUES_GEMM32_SHAPES
#undef JUES_GEMM32_TAIL
#undef JUES_GEMM32
  } else {
#define JUES_GEMM64(K_, TB_, TA_, SEG_, BT_, ...)                                                                \
  hipLaunchKernelGGL((gemm64_kernel<K_, TB_, TA_, SEG_, BT_, ##__VA_ARGS__>), grid, dim3(4 * BT_), 0, ctx->stream, \
                     p0, p1, (int)nt0, (double)alpha, (double)beta)
#define JUES_GEMM64_TAIL(K_, TB_, TA_) JUES_GEMM64(K_, TB_, TA_, false, 128, true)
#define JUES_GEMM64_SHAPES(BT_)                      \
  if (seg) {                                         \
    if (tb) JUES_GEMM64(0, true, false, true, BT_);  \
    else JUES_GEMM64(0, false, false, true, BT_);    \
  } else if (ta) {                                   \
    if (tb) JUES_GEMM64(0, true, true, false, BT_);  \
    else JUES_GEMM64(0, false, true, false, BT_);    \
  } else if (tb) JUES_GEMM64(0, true, false, false, BT_)
    if (tail) {
      if (ta && tb) JUES_GEMM64_TAIL(0, true, true);
      else if (ta) JUES_GEMM64_TAIL(0, false, true);
      else if (tb) JUES_GEMM64_TAIL(0, true, false);
      else if (kind == 1) JUES_GEMM64_TAIL(1, false, false);
      else if (kind == 2) JUES_GEMM64_TAIL(2, false, false);
      else JUES_GEMM64_TAIL(0, false, false);
    } else if (form == TILE64) {
      JUES_GEMM64_SHAPES(64);
      else JUES_GEMM64(0, false, false, false, 64);
    } else {
      JUES_GEMM64_SHAPES(128);
      else if (kind == 1) JUES_GEMM64(1, false, false, false, 128);
      else if (kind == 2) JUES_GEMM64(2, false, false, false, 128);
      else JUES_GEMM64(0, false, false, false, 128);
    }
#undef JUES_GEMM64_SHAPES
#undef JUES_GEMM64_TAIL
#undef JUES_GEMM64
  }
  if (tail) {
    JUES_HIP(hipGetLastError());
    int tiles = 0;
    for (const int n : p0.tail.n) tiles += n;
    if (p0.tail.wgs > tiles)
      hipLaunchKernelGGL((gemm_tail_kernel<T>), dim3((unsigned)tiles, 16), dim3(256), 0, ctx->stream, p0, beta);
  }
  JUES_HIP(hipGetLastError());
}

template <typename T>
static void short_launch(jues_ctx* ctx, bool tall, GemmSide<T> p, int nb, T alpha, T beta) {
  const dim3 grid((unsigned)((long)p.tiles_m * p.tiles_n), 1, nb);
  const bool three = (tall ? p.N : p.M) <= 48;  // 16-row (16-column) blocks: 3 or 4
#define JUES_SHORT(KERNEL_, THREADS_)                                                                      \
  do {                                                                                                     \
    if (three) hipLaunchKernelGGL(KERNEL_<3>, grid, dim3(THREADS_), 0, ctx->stream, p, alpha, beta);       \
    else hipLaunchKernelGGL(KERNEL_<4>, grid, dim3(THREADS_), 0, ctx->stream, p, alpha, beta);             \
  } while (0)
  if constexpr (sizeof(T) == 4) {
    if (tall) JUES_SHORT(gemm32_tall_kernel, 256);
    else JUES_SHORT(gemm32_sk_kernel, 256);
  } else {
    if (tall) JUES_SHORT(gemm64_tall_kernel, 512);
    else JUES_SHORT(gemm64_sk_kernel, 512);
  }
#undef JUES_SHORT
  JUES_HIP(hipGetLastError());
}

template <typename T, bool TA, bool TB>
static void direct_launch_ab(jues_ctx* ctx, int form, GemmSide<T> p, int nb, T alpha, T beta) {
  p.nz = nb;
  const long tiles = (long)p.tiles_m * p.tiles_n;
  const dim3 grid((unsigned)tiles, 1, grid_z(nb, tiles));
#define JUES_DIRECT(NW_, IM_, JN_)                                                                            \
  hipLaunchKernelGGL((gemm_direct_kernel<T, TA, TB, NW_, IM_, JN_>), grid, dim3(64 * NW_), 0, ctx->stream, p, \
                     alpha, beta)
  if (form == DIRECT22) JUES_DIRECT(4, 2, 2);
  else if (form == DIRECT21) JUES_DIRECT(4, 2, 1);
  else if (form == DIRECT12) JUES_DIRECT(4, 1, 2);
  else JUES_DIRECT(8, 1, 1);
#undef JUES_DIRECT
  JUES_HIP(hipGetLastError());
}

// One launch of `form` over nb batch entries of p (made for that form).
template <typename T>
static void form_launch(jues_ctx* ctx, int form, bool ta, bool tb, int kind, const GemmSide<T>& p, int nb, T alpha,
                        T beta) {
  if (form == TILE128 || form == TILE64) tile_launch<T>(ctx, form, tb, kind, p, p, false, nb, alpha, beta, ta);
  else if (form == SHORT || form == TALL) short_launch<T>(ctx, form == TALL, p, nb, alpha, beta);
  else if (ta && tb) direct_launch_ab<T, true, true>(ctx, form, p, nb, alpha, beta);
  else if (ta) direct_launch_ab<T, true, false>(ctx, form, p, nb, alpha, beta);
  else if (tb) direct_launch_ab<T, false, true>(ctx, form, p, nb, alpha, beta);
  else direct_launch_ab<T, false, false>(ctx, form, p, nb, alpha, beta);
}

template <typename T>
static void reduce_launch(jues_ctx* ctx, const T* W, long S, long M, long N, T* C, long ldc, T beta) {
  const unsigned nb = (unsigned)std::max(1L, std::min(cdiv(M * N, 256), 65536L));
  hipLaunchKernelGGL((splitk_reduce_kernel<T>), dim3(nb), dim3(256), 0, ctx->stream, W, (int)S, M, N, C, ldc, beta);
  JUES_HIP(hipGetLastError());
}

// Workspace for partial products, or null when the device has no room for it (the product then runs
// unsplit, which needs none).
template <typename T>
static T* split_work(jues_ctx* ctx, int slot, size_t elems) {
  try {
    return static_cast<T*>(scratch(ctx, slot, sizeof(T) * elems));
  } catch (const Error& e) {
    if (e.st != JUES_OOM) throw;
    return nullptr;
  }
}

static int symbol_kind(const char* tag) {
  return !tag ? 0 : (std::strcmp(tag, "cc_ring") == 0 ? 1 : (std::strcmp(tag, "cc_pp_ladder") == 0 ? 2 : 0));
}

template <typename T>
static void gemm_impl(jues_ctx* ctx, bool ta, bool tb, long M, long N, long K, T alpha, const T* A, long lda,
                      long sA, const T* B, long ldb, long sB, T beta, T* C, long ldc, long sC, int batch,
                      const char* tag, bool allow_split) {
  if (M <= 0 || N <= 0 || batch <= 0) return;
  JUES_REQUIRE(M < (1L << 31) && N < (1L << 31) && K < (1L << 31), "gemm: dimension too large");
  JUES_REQUIRE(ldc >= M, "gemm: ldc < M");
  JUES_REQUIRE(lda >= (ta ? K : M) || K == 0, "gemm: lda too small");
  JUES_REQUIRE(ldb >= (tb ? N : K) || K == 0, "gemm: ldb too small");
  const char* name = tag ? tag : (sizeof(T) == 8 ? "gemm_f64" : "gemm_f32");
  const int kind = symbol_kind(tag);
  if (K <= 0) {
    KTimer t(ctx, name, 0, 0);
    for (int b = 0; b < batch; ++b)
      hipLaunchKernelGGL(scale_kernel<T>, dim3(1024), dim3(256), 0, ctx->stream, C + (long)b * sC, M,
                         N, ldc, beta);
    JUES_HIP(hipGetLastError());
    return;
  }
  const bool split_ok = allow_split && !no_alloc_active();
  GemmPlan plan = gemm_plan<T>(ta, tb, M, N, K, lda, ldb, sA, sB, batch, split_ok);
  if (plan.form == SHORT && ta) {
    // the transposed copy of A that the SHORT form of a TN product reads
    T* At = static_cast<T*>(scratch(ctx, 18, sizeof(T) * (size_t)(M * K)));
    permute<T, T>(ctx, A, {K, M}, {1, 0}, At, 1.0, 0.0, name);
    A = At;
    lda = M;
    ta = false;
  }
  if (plan.split > 1) {
    // chunks of K in one launch, the last one shorter; the partial products are added in a fixed order
    const long kc = cdiv(cdiv(K, plan.split), 16) * 16, S = cdiv(K, kc);
    T* Wk = S > 1 ? split_work<T>(ctx, 9, (size_t)S * M * N) : nullptr;
    if (Wk) {
      {
        KTimer t1(ctx, name, 2.0 * M * N * K, (double)sizeof(T) * ((double)M * K + (double)K * N + (double)S * M * N));
        GemmSide<T> p = make_side<T>(M, N, kc, A, lda, ta ? kc : kc * lda, B, ldb, tb ? kc * ldb : kc, Wk, M, M * N,
                                     plan.form);
        p.Klast = (int)(K - (S - 1) * kc);
        form_launch<T>(ctx, plan.form, ta, tb, kind, p, (int)S, alpha, T(0));
      }
      KTimer t(ctx, name, 0.0, (double)sizeof(T) * S * M * N);
      reduce_launch<T>(ctx, Wk, S, M, N, C, ldc, beta);
      return;
    }
    plan = gemm_plan<T>(ta, tb, M, N, K, lda, ldb, sA, sB, batch, false);
  }
  if (plan.tail.wgs) {
    T* part = split_work<T>(ctx, 9, (size_t)plan.tail.wgs * 128 * 128);
    if (part) {
      KTimer t(ctx, name, 2.0 * M * N * K, (double)sizeof(T) * ((double)M * K + (double)K * N + (double)M * N));
      GemmSide<T> p = make_side<T>(M, N, K, A, lda, 0, B, ldb, 0, C, ldc, 0);
      p.tail = plan.tail;
      p.part = part;
      tile_launch<T>(ctx, TILE128, tb, kind, p, p, false, 1, alpha, beta, ta);
      return;
    }
    plan = gemm_plan<T>(ta, tb, M, N, K, lda, ldb, sA, sB, batch, false);
  }
  const double flops = 2.0 * M * N * K * batch;
  const double bytes = (double)sizeof(T) * ((double)M * K + (double)K * N + (beta != T(0) ? 2.0 : 1.0) * M * N) * batch;
  KTimer timer(ctx, name, flops, bytes);
  for (int b0 = 0; b0 < batch; b0 += 65528) {
    const GemmSide<T> p = make_side<T>(M, N, K, A + (long)b0 * sA, lda, sA, B + (long)b0 * sB, ldb, sB,
                                       C + (long)b0 * sC, ldc, sC, plan.form);
    form_launch<T>(ctx, plan.form, ta, tb, kind, p, std::min(batch - b0, 65528), alpha, beta);
  }
}

template <typename T>
void gemm(jues_ctx* ctx, bool ta, bool tb, long M, long N, long K, T alpha, const T* A, long lda, long sA,
          const T* B, long ldb, long sB, T beta, T* C, long ldc, long sC, int batch, const char* tag) {
  gemm_impl<T>(ctx, ta, tb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, tag, true);
}

// Half the work of the square: 8640 x 8640 x 768 takes 1.09 ms, 1.80 as a whole.
bool gemm_lower(jues_ctx* ctx, long M, long K, const double* L, long ldl, double* C, long ldc, const char* tag) {
  if (M < 128 || K < 1 || M >= (1L << 31) || K >= (1L << 31) || !form_ok<double>(TILE128, false, true, M, M, K, ldl, ldl))
    return false;
  JUES_REQUIRE(ldl >= M && ldc >= M, "gemm_lower: leading dimension too small");
  const long fm = M / 128, full = fm * (fm + 1) / 2 / 256 * 256;
  TailMap best = tail_map(kTail<double>, M, M, K, full, 1, true);  // nothing shared, if there is no workspace
  if (!best.wgs && full >= 256) best = tail_map(kTail<double>, M, M, K, full - 256, 1, true);
  if (!best.wgs) return false;
  double us = tail_us<double>(best);
  double* part = nullptr;
  if (!no_alloc_active()) {
    TailMap shared;
    for (const long whole : {full, full - 256})
      for (int chunks = 2; whole >= 0 && chunks <= 32; ++chunks) {
        const TailMap t = tail_map(kTail<double>, M, M, K, whole, chunks, true);
        if (t.wgs && tail_us<double>(t) < us) shared = t, us = tail_us<double>(t);
      }
    if (shared.wgs && (part = split_work<double>(ctx, 9, (size_t)shared.wgs * 128 * 128))) best = shared;
  }
  // against the whole square (a few tiles leave the chip idle either way)
  const double square = gemm_plan<double>(false, true, M, M, K, ldl, ldl, 0, 0, 1, !no_alloc_active()).us;
  if (square < us) return false;
  const char* name = tag ? tag : "gemm_f64";
  KTimer t(ctx, name, 1.0 * M * (M + 1) * K, 8.0 * (double)M * (K + 0.5 * M));
  GemmSide<double> p = make_side<double>(M, M, K, L, ldl, 0, L, ldl, 0, C, ldc, 0);
  p.tail = best;
  p.part = part;
  tile_launch<double>(ctx, TILE128, true, 0, p, p, false, 1, 1.0, 0.0);
  return true;
}

bool gemm32_out64(jues_ctx* ctx, long M, long N, long K, const float* A, long lda, const float* B, long ldb,
                  double* C, long ldc, const char* tag) {
  if (M <= 0 || N <= 0 || K < 16 || !form_ok<float>(TILE128, false, false, M, N, K, lda, ldb)) return false;
  JUES_REQUIRE(lda >= M && ldb >= K && ldc >= M, "gemm32_out64: leading dimension too small");
  GemmSide<float> p = make_side<float>(M, N, K, A, lda, 0, B, ldb, 0, nullptr, ldc, 0);
  p.C64 = C;
  const long tiles = (long)p.tiles_m * p.tiles_n;
  JUES_REQUIRE(tiles < (1L << 31), "gemm: too many tiles");
  KTimer timer(ctx, tag ? tag : "gemm_f32", 2.0 * M * N * K, 4.0 * ((double)M * K + (double)K * N) + 8.0 * M * N);
  hipLaunchKernelGGL((gemm32_nn_kernel<0, false, false, false, true>), dim3((unsigned)tiles, 1, 1), dim3(NT), 0,
                     ctx->stream, p, p, (int)tiles, 1.0f, 0.0f);
  JUES_HIP(hipGetLastError());
  return true;
}

template <typename T>
void gemm_batch_sum(jues_ctx* ctx, bool ta, bool tb, long M, long N, long K, T alpha, const T* A, long lda, long sA,
                    const T* B, long ldb, long sB, T beta, T* C, long ldc, int batch, T* work, const char* tag) {
  JUES_REQUIRE(batch >= 1 && M > 0 && N > 0, "gemm_batch_sum: empty product");
  const char* name = tag ? tag : (sizeof(T) == 8 ? "gemm_f64" : "gemm_f32");
  gemm_impl<T>(ctx, ta, tb, M, N, K, alpha, A, lda, sA, B, ldb, sB, T(0), work, M, M * N, batch, tag, false);
  KTimer t(ctx, name, 0.0, (double)sizeof(T) * ((double)batch + (beta != T(0) ? 2.0 : 1.0)) * M * N);
  reduce_launch<T>(ctx, work, batch, M, N, C, ldc, beta);
}

template <typename T>
void gemm_pair(jues_ctx* ctx, bool tb, long M0, long N0, long K0, const T* A0, long lda0, const T* B0, long ldb0,
               T* C0, long ldc0, long M1, long N1, long K1, const T* A1, long lda1, const T* B1, long ldb1, T* C1,
               long ldc1, T alpha, T beta, const char* tag) {
  const bool empty0 = M0 <= 0 || N0 <= 0, empty1 = M1 <= 0 || N1 <= 0;
  // One launch of 64x64 or 128x128 tiles, its contractions split over S chunks, against two planned
  // products, by the same estimate.
  // In FP32 both keep to sums over k as long as those of 1024 workgroups, each with at least 1024 of k (chain_limit).
  GemmPlan best;
  if (!empty0 && !empty1 && K0 >= 16 && K1 >= 16) {
    long limit = std::max(K0, K1);
    if (sizeof(T) == 4 && !no_alloc_active()) {
      const long t = cdiv(M0, 128) * cdiv(N0, 128) + cdiv(M1, 128) * cdiv(N1, 128);
      const long S = t < 1024 ? std::min(std::min(K0, K1) / 1024, cdiv(2048, t)) : 1;
      if (S > 1) limit = cdiv(limit, S);
    }
    const double bytes = (double)sizeof(T) * ((double)M0 * K0 + (double)K0 * N0 + (double)M0 * N0 + (double)M1 * K1 +
                                              (double)K1 * N1 + (double)M1 * N1);
    for (const int form : {(int)TILE128, (int)TILE64}) {
      if (!form_ok<T>(form, false, tb, M0, N0, K0, lda0, ldb0) || !form_ok<T>(form, false, tb, M1, N1, K1, lda1, ldb1))
        continue;
      const long bt = form == TILE128 ? 128 : 64;
      const long tiles = cdiv(M0, bt) * cdiv(N0, bt) + cdiv(M1, bt) * cdiv(N1, bt);
      const double elems = (double)M0 * N0 + (double)M1 * N1;
      for (const long s : kSplits) {
        if (s > 1 && (no_alloc_active() || s > 16 || std::min(K0, K1) < 64 * s || tiles * s > 8192 ||
                      (double)s * elems * sizeof(T) > 268435456.0))
          break;
        if (cdiv(std::max(K0, K1), s) > limit) continue;
        const double us = form_us<T>(form, tiles * s, cdiv(cdiv(std::max(K0, K1), s), 16), bytes) +
                          (s > 1 ? 2.0 : 0.0) + reduce_us<T>(s, elems);
        if (us < best.us) best = GemmPlan{form, s, TailMap{}, us};
      }
    }
    const GemmPlan a0 = gemm_plan<T>(false, tb, M0, N0, K0, lda0, ldb0, 0, 0, 1, !no_alloc_active()),
                   a1 = gemm_plan<T>(false, tb, M1, N1, K1, lda1, ldb1, 0, 0, 1, !no_alloc_active());
    const bool within = limit == std::max(K0, K1) || std::max(a0.chain, a1.chain) <= cdiv(limit, 16) * 16;
    if (a0.us + a1.us <= best.us && (within || best.us >= 1e300)) best.us = 1e300;
  }
  T* Wk = nullptr;
  long S = best.split;
  if (best.us < 1e300 && S > 1) {
    Wk = split_work<T>(ctx, 16, (size_t)S * (M0 * N0 + M1 * N1));
    if (!Wk) best.us = 1e300;
  }
  if (best.us >= 1e300) {
    gemm<T>(ctx, false, tb, M0, N0, K0, alpha, A0, lda0, 0, B0, ldb0, 0, beta, C0, ldc0, 0, 1, tag);
    gemm<T>(ctx, false, tb, M1, N1, K1, alpha, A1, lda1, 0, B1, ldb1, 0, beta, C1, ldc1, 0, 1, tag);
    return;
  }
  JUES_REQUIRE(M0 < (1L << 31) && N0 < (1L << 31) && K0 < (1L << 31) && M1 < (1L << 31) && N1 < (1L << 31) &&
                   K1 < (1L << 31),
               "gemm: dimension too large");
  JUES_REQUIRE(ldc0 >= M0 && ldc1 >= M1, "gemm: ldc < M");
  JUES_REQUIRE(lda0 >= M0 && lda1 >= M1, "gemm: lda too small");
  JUES_REQUIRE(ldb0 >= (tb ? N0 : K0) && ldb1 >= (tb ? N1 : K1), "gemm: ldb too small");
  const char* name = tag ? tag : (sizeof(T) == 8 ? "gemm_f64" : "gemm_f32");
  const int kind = symbol_kind(tag);
  const double sz = sizeof(T), bf = beta != T(0) ? 2.0 : 1.0;
  const double flops = 2.0 * M0 * N0 * K0 + 2.0 * M1 * N1 * K1;
  const long n0 = M0 * N0, n1 = M1 * N1;
  const double in = sz * ((double)M0 * K0 + (double)K0 * N0 + (double)M1 * K1 + (double)K1 * N1);
  if (Wk) {
    // both K ranges in S chunks (the last chunk of each shorter): the partial products go to the
    // workspace and are added to C0 / C1 in a fixed order
    const long kc0 = cdiv(K0, S), kc1 = cdiv(K1, S);
    {
      KTimer timer(ctx, name, flops, in + sz * S * (n0 + n1));
      GemmSide<T> p0 = make_side<T>(M0, N0, kc0, A0, lda0, kc0 * lda0, B0, ldb0, tb ? kc0 * ldb0 : kc0, Wk, M0, n0,
                                    best.form);
      GemmSide<T> p1 = make_side<T>(M1, N1, kc1, A1, lda1, kc1 * lda1, B1, ldb1, tb ? kc1 * ldb1 : kc1, Wk + S * n0,
                                    M1, n1, best.form);
      p0.Klast = (int)(K0 - (S - 1) * kc0);
      p1.Klast = (int)(K1 - (S - 1) * kc1);
      tile_launch<T>(ctx, best.form, tb, kind, p0, p1, true, (int)S, alpha, T(0));
    }
    KTimer t(ctx, name, 0.0, sz * (S + bf) * (n0 + n1));
    reduce_launch<T>(ctx, Wk, S, M0, N0, C0, ldc0, beta);
    reduce_launch<T>(ctx, Wk + S * n0, S, M1, N1, C1, ldc1, beta);
    return;
  }
  KTimer timer(ctx, name, flops, in + sz * bf * (n0 + n1));
  tile_launch<T>(ctx, best.form, tb, kind,
                 make_side<T>(M0, N0, K0, A0, lda0, 0, B0, ldb0, 0, C0, ldc0, 0, best.form),
                 make_side<T>(M1, N1, K1, A1, lda1, 0, B1, ldb1, 0, C1, ldc1, 0, best.form), true, 1, alpha, beta);
}

template <typename T>
void gemm_ksum(jues_ctx* ctx, bool tb, long M, long N, long K, const T* A0, const T* B0, const T* A1, const T* B1,
               const long* tab, int groups, int inner, long lda, long ldb, long sA, long sB, T alpha, T beta, T* C,
               long ldc, long sC, long sG, const char* tag) {
  if (M <= 0 || N <= 0 || groups <= 0 || inner <= 0) return;
  JUES_REQUIRE(M < (1L << 31) && N < (1L << 31) && 2 * K < (1L << 31), "gemm: dimension too large");
  JUES_REQUIRE(K >= 16 && K % 16 == 0 && (long)groups * inner <= 65528, "gemm_ksum: bad contraction or batch");
  JUES_REQUIRE(ldc >= M && lda >= M && ldb >= (tb ? N : K), "gemm: leading dimension too small");
  const long batch = (long)groups * inner;
  const double bytes = (double)sizeof(T) * batch * (2.0 * M * K + 2.0 * N * K + (beta != T(0) ? 2.0 : 1.0) * M * N);
  GemmPlan best;
  for (const int form : {(int)TILE128, (int)TILE64}) {
    if (!form_ok<T>(form, false, tb, M, N, K, lda, ldb)) continue;
    const long bt = form == TILE128 ? 128 : 64;
    const double us = form_us<T>(form, cdiv(M, bt) * cdiv(N, bt) * batch, 2 * K / 16, 0.0);
    if (us < best.us) best = GemmPlan{form, 1, TailMap{}, us};
  }
  JUES_REQUIRE(best.us < 1e300, "gemm_ksum: leading dimension too large");
  const char* name = tag ? tag : (sizeof(T) == 8 ? "gemm_f64" : "gemm_f32");
  KTimer timer(ctx, name, 4.0 * M * N * K * batch, bytes);
  GemmSide<T> p = make_side<T>(M, N, K, A0, lda, sA, B0, ldb, sB, C, ldc, sC, best.form);
  p.A1 = A1;
  p.B1 = B1;
  p.K1 = (int)K;
  p.tab = tab;
  p.inner = inner;
  p.sG = sG;
  tile_launch<T>(ctx, best.form, tb, 0, p, p, false, (int)batch, alpha, beta, false, true);
}

template void gemm_ksum<double>(jues_ctx*, bool, long, long, long, const double*, const double*, const double*,
                                const double*, const long*, int, int, long, long, long, long, double, double, double*,
                                long, long, long, const char*);
template void gemm_ksum<float>(jues_ctx*, bool, long, long, long, const float*, const float*, const float*,
                               const float*, const long*, int, int, long, long, long, long, float, float, float*, long,
                               long, long, const char*);

template void gemm_pair<double>(jues_ctx*, bool, long, long, long, const double*, long, const double*, long, double*,
                                long, long, long, long, const double*, long, const double*, long, double*, long,
                                double, double, const char*);
template void gemm_pair<float>(jues_ctx*, bool, long, long, long, const float*, long, const float*, long, float*, long,
                               long, long, long, const float*, long, const float*, long, float*, long, float, float,
                               const char*);

template void gemm_batch_sum<double>(jues_ctx*, bool, bool, long, long, long, double, const double*, long, long,
                                     const double*, long, long, double, double*, long, int, double*, const char*);
template void gemm_batch_sum<float>(jues_ctx*, bool, bool, long, long, long, float, const float*, long, long,
                                    const float*, long, long, float, float*, long, int, float*, const char*);
template void gemm<double>(jues_ctx*, bool, bool, long, long, long, double, const double*, long, long,
                           const double*, long, long, double, double*, long, long, int, const char*);
template void gemm<float>(jues_ctx*, bool, bool, long, long, long, float, const float*, long, long,
                          const float*, long, long, float, float*, long, long, int, const char*);

}  // namespace jues
