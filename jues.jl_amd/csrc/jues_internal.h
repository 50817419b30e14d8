// Internal declarations shared by the libjues_hip translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <list>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "../../include/jues.h"

namespace jues {

struct Error : std::exception {
  jues_status st;
  std::string msg;
  Error(jues_status s, std::string m) : st(s), msg(std::move(m)) {}
  const char* what() const noexcept override { return msg.c_str(); }
};

#define JUES_HIP(x)                                                                    \
  do {                                                                                 \
    hipError_t e_ = (x);                                                               \
    if (e_ != hipSuccess)                                                              \
      throw ::jues::Error(JUES_HIP_ERROR, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

#define JUES_REQUIRE(cond, msg)                                          \
  do {                                                                   \
    if (!(cond)) throw ::jues::Error(JUES_BAD_ARG, std::string(msg));    \
  } while (0)

// Device blocks that a context's buffers released and may use again.  A solve, a gradient or a transform
// allocates and frees tens of buffers of up to hundreds of megabytes, and hipMalloc / hipFree cost from
// tens of microseconds to several milliseconds each (the driver maps and clears the memory, and hipFree waits
// for the device): at n = 256 they took 2.2 of the 8.7 ms of a factor-route MP2 gradient, and 40 ms of it when
// three contexts took turns.
// One pool per context, so every block is reused in the order of that context's stream.  Kept are at most a
// sixteenth of the device's memory and 256 blocks, the least recently released going first; jues_release
// and jues_destroy give all of them back, and an allocation that the device refuses is tried again after
// every pool of the process has given its blocks back.
class BlockPool {
 public:
  explicit BlockPool(int device);
  ~BlockPool();
  void* take(size_t bytes, size_t& capacity);  // a kept block of at least `bytes`, or null
  void give(void* p, size_t capacity);         // keeps or frees the block
  void trim();                                 // frees every kept block
  void close();                                // trim, and free what is given from now on
  size_t kept();
  int device() const { return device_; }

 private:
  struct Block {
    void* p;
    size_t capacity;
  };
  std::mutex mu_;
  std::list<Block> blocks_;  // oldest first
  size_t kept_ = 0, limit_ = 0;
  int device_;
  bool open_ = true;
};

// While one is active on the calling thread, DevBuf::alloc uses the given pool.
struct PoolScope {
  std::shared_ptr<BlockPool> prev;
  explicit PoolScope(const std::shared_ptr<BlockPool>& pool);
  ~PoolScope();
};

// Owning device allocation.  Allocation failure raises JUES_OOM.
struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  DevBuf() = default;
  explicit DevBuf(size_t nbytes) { alloc(nbytes); }
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  DevBuf(DevBuf&& o) noexcept { swap(o); }
  DevBuf& operator=(DevBuf&& o) noexcept {
    if (this != &o) { release(); swap(o); }
    return *this;
  }
  ~DevBuf() { release(); }
  void alloc(size_t nbytes);
  void release();
  template <typename T> T* as() const { return static_cast<T*>(p); }

 private:
  void swap(DevBuf& o) noexcept {
    std::swap(p, o.p);
    std::swap(bytes, o.bytes);
    std::swap(capacity, o.capacity);
    pool.swap(o.pool);
  }
  size_t capacity = 0;              // of the block, at least `bytes`
  std::shared_ptr<BlockPool> pool;  // where the block goes on release
};

// Device memory allocated by the process (buffers in use and kept blocks)
size_t device_bytes_in_use();
// Free and total memory of the context's device; kept blocks, which the next allocation may take, count as free
void device_memory(jues_ctx* ctx, size_t* free_bytes, size_t* total_bytes);

// Allocation-free scope: while one is active on the calling thread, DevBuf::alloc and
// scratch() raise instead of allocating, and gemm() avoids its workspace paths (split-K,
// the transposed copy of a short A).  Used by the entry points that must not allocate.
struct NoAllocScope {
  bool prev;
  NoAllocScope();
  ~NoAllocScope();
};
bool no_alloc_active();
// looks up the device address of the allocation-free entry point's static scratch array on
// `device` (current) once; called by jues_create (noalloc.hip)
void noalloc_attach(int device);

struct KStat {
  double ms = 0, calls = 0, flops = 0, bytes = 0;
};

struct CCState;  // cc.hip
struct CCDeleter {
  void operator()(CCState* p) const;  // defined in cc.hip
};

}  // namespace jues

struct jues_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  std::shared_ptr<jues::BlockPool> pool;
  jues::DevBuf scratch[20];  // temporaries, grown on demand (jues::scratch)
  // AO integrals: exactly one of gao (n^4) / Bfac (n*n*naux) is set.
  int n = 0, naux = 0;
  jues::DevBuf gao;
  jues::DevBuf Bfac;
  jues::DevBuf gao32, Bfac32;  // FP32 copies, made on first FP32 use
  // kernel timing (HIP events on `stream`)
  bool timing = false;
  std::map<std::string, jues::KStat> kstats;
  struct Pending { std::string name; hipEvent_t a, b; double flops, bytes; };
  std::vector<Pending> pending;
  std::vector<hipEvent_t> event_pool;
  std::unique_ptr<jues::CCState, jues::CCDeleter> cc;
  jues_ctx();
  ~jues_ctx();
};

namespace jues {

// Scoped kernel timer: records events around the enclosed launches when timing is on.
struct KTimer {
  jues_ctx* ctx;
  bool on;
  size_t slot = 0;
  KTimer(jues_ctx* c, const char* name, double flops, double bytes);
  ~KTimer();
};
void flush_timers(jues_ctx* ctx);  // synchronises and folds pending events into kstats

// ---- GEMM (gemm.hip) -------------------------------------------------------
// Column-major C[M,N] = alpha*op(A)*op(B) + beta*C, batched with element strides.
template <typename T>
void gemm(jues_ctx* ctx, bool ta, bool tb, long M, long N, long K, T alpha, const T* A, long lda,
          long sA, const T* B, long ldb, long sB, T beta, T* C, long ldc, long sC, int batch = 1,
          const char* tag = nullptr);

// C = L L^T (M x M, L M x K) in the tiles of the lower triangle only (what lies above the diagonal's tiles is left
// as it is); returns false, launching nothing, where the whole square is faster or the kernel does not apply.
bool gemm_lower(jues_ctx* ctx, long M, long K, const double* L, long ldl, double* C, long ldc,
                const char* tag = nullptr);

// C = A B in FP32 MFMA work with the FP64 result written directly (NN, beta = 0, one product), on
// the high-occupancy FP32 kernel; returns false, launching nothing, where that kernel does not apply.
bool gemm32_out64(jues_ctx* ctx, long M, long N, long K, const float* A, long lda, const float* B, long ldb,
                  double* C, long ldc, const char* tag = nullptr);

// C = alpha sum_z op(A_z) op(B_z) + beta C over a batch (strides sA, sB): the batch's products are
// written to work (batch * M * N elements) and added in a fixed order, so the result is the same
// on every call.
template <typename T>
void gemm_batch_sum(jues_ctx* ctx, bool ta, bool tb, long M, long N, long K, T alpha, const T* A, long lda, long sA,
                    const T* B, long ldb, long sB, T beta, T* C, long ldc, int batch, T* work,
                    const char* tag = nullptr);

// Two independent products C_i = alpha A_i op(B_i) + beta C_i (A_i m-contiguous, op the same
// for both) in one launch, so that the second fills the first one's last partial round of
// workgroups; falls back to two gemm calls where the high-occupancy kernels do not apply.
template <typename T>
void gemm_pair(jues_ctx* ctx, bool tb, long M0, long N0, long K0, const T* A0, long lda0, const T* B0, long ldb0,
               T* C0, long ldc0, long M1, long N1, long K1, const T* A1, long lda1, const T* B1, long ldb1, T* C1,
               long ldc1, T alpha, T beta, const char* tag = nullptr);

// C = alpha (A0 op(B0) + A1 op(B1)) + beta C over groups x inner batch entries in one launch: products over
// two contraction segments of K (a multiple of 16) each, which share the leading dimensions, so C is read
// and written once.  Entry (g, r) reads A0 + tab[4g] + r sA, B0 + tab[4g+1] + r sB, A1 + tab[4g+2] + r sA and
// B1 + tab[4g+3] + r sB (tab: device, in elements) and writes C + g sG + r sC.
template <typename T>
void gemm_ksum(jues_ctx* ctx, bool tb, long M, long N, long K, const T* A0, const T* B0, const T* A1, const T* B1,
               const long* tab, int groups, int inner, long lda, long ldb, long sA, long sB, T alpha, T beta, T* C,
               long ldc, long sC, long sG, const char* tag = nullptr);

// ---- split-FP16 MFMA GEMM (gemm16.hip) ---------------------------------------
// An FP32 matrix X (rows x cols) as two FP16 planes hi + lo = s X, column-major and
// zero-padded to rows_p (multiple of 32) x cols_p (>= cols + 256), interleaved per
// 32-row block: column c, block b holds 32 hi then 32 lo halves at p + c*2*rows_p + 64b.
// `sexp` is a device int holding k, s = 2^k.
struct Split16 {
  _Float16* p = nullptr;
  int* sexp = nullptr;
  long rows = 0, cols = 0, rows_p = 0, cols_p = 0;
};
struct Split16Buf {
  DevBuf mem;
  Split16 s;
  void ensure(long rows, long cols);  // (re)allocates when the padded size grows
};
// columns [c0, c0 + nc) of a split operand (its planes, padding beyond them included)
inline Split16 split16_cols(const Split16& s, long c0, long nc) {
  Split16 r = s;
  r.p = s.p + c0 * 2 * s.rows_p;
  r.cols = nc;
  r.cols_p = s.cols_p - c0;
  return r;
}
// planes of X; the scale is found on the device (no host synchronisation)
template <typename Ti>
void split16(jues_ctx* ctx, const Ti* X, long rows, long cols, long ldx, Split16Buf& out,
             const char* tag = nullptr);
// planes (rows x cols) of X^T, X stored cols x rows with leading dimension ldx
template <typename Ti>
void split16t(jues_ctx* ctx, const Ti* X, long rows, long cols, long ldx, Split16Buf& out,
              const char* tag = nullptr);
// C[m,n] = alpha sum_k A(k,m) B(k,n) + beta C[m,n], K = A.rows = B.rows, FP32 C
void gemm16_tn(jues_ctx* ctx, long M, long N, float alpha, const Split16& A, const Split16& B, float beta,
               float* C, long ldc, const char* tag = nullptr);

// ---- elementwise / data movement (kernels.hip) -------------------------------
// out = alpha * permutedims(in, perm) + beta * out   (perm 0-based; out dim k = in dim perm[k])
template <typename Ti, typename To>
void permute(jues_ctx* ctx, const Ti* in, const std::vector<long>& in_dims,
             const std::vector<int>& perm, To* out, double alpha, double beta,
             const char* tag = nullptr);
template <typename Ti, typename To>
void convert(jues_ctx* ctx, const Ti* in, To* out, long n);
template <typename T>
void fill(jues_ctx* ctx, T* out, long n, double value);
// y = a*x + b*y
template <typename T>
void axpby(jues_ctx* ctx, long n, double a, const T* x, double b, T* y);
// z = a*x + b*y, formed in FP64 and rounded once to T
template <typename T>
void axpby2(jues_ctx* ctx, long n, double a, const double* x, double b, const double* y, T* z);
// deterministic FP64 dot of two vectors (any element types)
template <typename Ta, typename Tb>
double dot(jues_ctx* ctx, const Ta* x, const Tb* y, long n);
double max_abs(jues_ctx* ctx, const double* x, long n);

// ---- contraction engine (einsum.cpp) -----------------------------------------
template <typename T>
struct Tens {
  T* p = nullptr;
  std::string idx;         // one letter per dimension, first letter fastest
  std::vector<long> dims;
  long size() const { long s = 1; for (long d : dims) s *= d; return s; }
};
// C[idxC] = alpha * sum A[idxA] B[idxB] + beta * C  (any index order; TTGT on the device).
// A permuted copy of an operand or of the product goes to `work` (work_elems elements) when
// given and large enough, else to the context's scratch.
template <typename T>
void contract(jues_ctx* ctx, double alpha, const Tens<T>& A, const Tens<T>& B, double beta,
              const Tens<T>& C, const char* tag = nullptr, T* work = nullptr, long work_elems = 0);
// C[idxC] = alpha * P(A) + beta * C
template <typename Ti, typename To>
void add_perm(jues_ctx* ctx, double alpha, const Tens<Ti>& A, double beta, const Tens<To>& C,
              const char* tag = nullptr);

// scratch pool owned by the context for temporaries of the contraction engine
void* scratch(jues_ctx* ctx, int slot, size_t bytes);

void release_scratch(jues_ctx* ctx);

// ---- integral transformation (transform.hip) -------------------------------------
// AO integrals in precision T (FP32 copies are made on first use and cached).
template <typename T> const T* ao_dense(jues_ctx* ctx);
template <typename T> const T* ao_factors(jues_ctx* ctx);
// out[p,q,r,s] (chemist, d1 x d2 x d3 x d4) from device C_k (n x d_k)
template <typename T>
void tei_transform_dev(jues_ctx* ctx, const T* C1, int d1, const T* C2, int d2, const T* C3, int d3,
                       const T* C4, int d4, T* out);
// MO factors L[p,q,P] = (C1^T B_P C2)[p,q]  (needs factors)
template <typename T>
void mo_factors_dev(jues_ctx* ctx, const T* C1, int d1, const T* C2, int d2, T* L);
// the same with the half-transformed factors in `work` (n * min(d1, d2) * naux elements)
template <typename T>
void mo_factors_dev(jues_ctx* ctx, const T* C1, int d1, const T* C2, int d2, T* L, T* work);
// RMP2 energy from K[i,a,j,b] = (ia|jb) (device, o x v x o x v) and eps (device FP64, n)
template <typename T>
double mp2_energy_dev(jues_ctx* ctx, const T* K, const double* eps, int o, int v);
// The same from the lower triangle (rows >= columns) of a symmetric K = (ia|jb); with G non-null also the whole of
// G[i,a,j,b] = dE/dK = 2 (2 K_iajb - K_ibja) / D and, with r non-null, r[i,a] = the row and column sums of
// K (2 K - K_ibja) / D^2 (device; work: o v^2 doubles).  For o in [LOWER_MIN_O, LOWER_MAX_O].
constexpr int LOWER_MIN_O = 16, LOWER_MAX_O = 88;
double mp2_lower_dev(jues_ctx* ctx, const double* K, const double* eps, int o, int v, double* G = nullptr,
                     double* r = nullptr, double* work = nullptr);
// One UMP2 spin block from K[i,a,J,B] = (ia|JB) (oA vA x oB vB) and the two spins' orbital
// energies (occupied first); same = alpha-alpha or beta-beta (K square, eA == eB).
template <typename T>
double ump2_block_dev(jues_ctx* ctx, const T* K, const double* eA, const double* eB, int oA, int vA, int oB, int vB,
                      bool same);

// ---- host <-> device helpers ---------------------------------------------------
void h2d(jues_ctx* ctx, void* dst, const void* src, size_t bytes);
void d2h(jues_ctx* ctx, void* dst, const void* src, size_t bytes);
void sync(jues_ctx* ctx);

}  // namespace jues
