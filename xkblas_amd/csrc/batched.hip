// batched.hip — uneven batches of small GEMMs and lower-triangular TRSMs,
// FP64 and FP32 mixed, in ONE persistent launch (gfx950).
//
// A plan turns the problems into work items — one per 64 x 64 output tile of
// each GEMM, one per 64-column panel of each TRSM — sorted by estimated cost,
// longest first.  The persistent kernel starts as many workgroups as fit on
// the chip at once; each workgroup takes the next item from a device counter
// until the list is exhausted (every workgroup reaches the exit), so large and
// small problems balance without one launch per problem.  A run is two
// launches on one stream: an int fill of the counter (no memset node, so the
// pair can be captured in a hipGraph) and the persistent kernel.
//
// The first items go to the workgroups by position, the others from the counter.
// GEMM tile: 4 waves, 2 x 2 of 32 x 32 quarters as 16 x 16 MFMA blocks
// (v_mfma_f64_16x16x4f64 / v_mfma_f32_16x16x4f32), 32-deep k slices through
// LDS, rows beyond the matrix repeated, the end of the inner dimension zero.
// TRSM panel (Left, Lower, NoTrans, Non-unit; B m x ncols with ncols <= 64),
// left-looking over 64-row blocks: one MFMA tile, 16 columns a wave, forms alpha
// B_kb minus the solved blocks' contribution, then each wave solves its columns
// by itself, 16 rows at a time (rows in lanes, DPP), and the block is written
// back for the next one, all inside the workgroup.
// Shared memory is 40 KB per workgroup, so four fit on a CU.
#include "common.h"
#include "kernels.h"
#include "runtime.h"
#include "../../include/xkblas.h"
#include <algorithm>
#include <cstdio>
#include <vector>

namespace xk {

typedef double bd4 __attribute__((ext_vector_type(4)));
typedef float bf4 __attribute__((ext_vector_type(4)));

struct BatchProblem {
  int kind;   // 0 GEMM, 1 TRSM
  int dtype;  // 0 FP64, 1 FP32
  int ta, tb;
  int m, n, k;
  double alpha, beta;
  const void* A;
  long lda;
  const void* B;
  long ldb;
  void* C;
  long ldc;
};

struct BatchItem {
  int prob;
  int tm, tn;  // GEMM tile indices; TRSM: tn = panel index
  int tile;    // GEMM tile order (64 or 32)
};

__device__ __forceinline__ bd4 bmfma(double a, double b, bd4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ __forceinline__ bf4 bmfma(float a, float b, bf4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

template <typename T> struct BAcc;
template <> struct BAcc<double> { typedef bd4 type; };
template <> struct BAcc<float> { typedef bf4 type; };

// Operands by pointers into global memory: a load through a pointer of unknown
// kind also counts as an LDS access, and every wait for LDS data would wait
// for the prefetched slices too.
template <typename T> using GlobalC = const __attribute__((address_space(1))) T*;
template <typename T> using Global = __attribute__((address_space(1))) T*;

constexpr int TB_BM = 64, TB_BK = 32, TB_LD = TB_BM + 2;

// Shared memory of one workgroup, in doubles: 40 KB, so that four
// workgroups fit in the 160 KB of a CU.  Overlaid uses:
//   GEMM staging  (A, B) x 32 x 66                         4224
//   TRSM          L_kk, 10 tiles of 256, and 4 x 16 columns of 17   3648
//   item index    one int at the start, between items
constexpr int BATCH_SMEM = 5120;

// Thread index hidden from loop-invariant code motion: recomputing the
// swizzled LDS offsets of an item is cheaper than keeping them live (and
// spilled) across the whole persistent loop.
__device__ __forceinline__ int item_tid()
{
  int t = threadIdx.x;
  __asm__ volatile("" : "+v"(t));
  return t;
}

// A barrier for LDS data alone: loads from memory stay in flight over it.
__device__ __forceinline__ void slice_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One operand of a tile: this thread's elements of each 32-deep slice of op(A)
// (`rows` of m) or op(B) (`rows` of n), by pointers that move on one slice at a
// time.  along: the tile's rows are contiguous in memory, else the inner index
// is.  Rows beyond the matrix repeat its last one: they only reach results that
// are not stored.
template <typename T, int TBM>
struct SliceLoad {
  static constexpr int V = TBM / 16, SH = TBM == 64 ? 6 : 5;  // V elements of each half of a slice
  GlobalC<T> p[V];
  T* lds;     // place of element 0
  long step;  // half a slice
  int k0;     // inner index of element 0
  bool along;

  __device__ __forceinline__ SliceLoad(GlobalC<T> A, long ld, bool along_, int row0, int rows, int tid, T* buf)
      : along(along_)
  {
    const int i0 = along ? tid & (TBM - 1) : tid >> 4;
    k0 = along ? tid >> SH : tid & 15;
    step = along ? 16 * ld : 16;
    lds = buf + k0 * TB_LD + i0;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = min(row0 + i0 + (along ? 0 : 16 * v), rows - 1), k = k0 + (along ? 256 / TBM * v : 0);
      p[v] = along ? A + i + (long)k * ld : A + k + (long)i * ld;
    }
  }
  // the next slice; left: what is left of the inner dimension
  __device__ __forceinline__ void load(T (&r)[2 * V], int left, GlobalC<T> A)
  {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        GlobalC<T> q = p[v];
        if (left < TB_BK) q = k0 + (along ? 256 / TBM * v : 0) + 16 * h < left ? q : A;
        r[h * V + v] = *q;
        p[v] += step;
      }
  }
  __device__ __forceinline__ void store(const T (&r)[2 * V], int left) const
  {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      T* d = lds + 16 * h * TB_LD;
      if (left < TB_BK) {
#pragma unroll
        for (int v = 0; v < V; ++v)
          d[along ? 256 / TBM * v * TB_LD : 16 * v] =
              k0 + (along ? 256 / TBM * v : 0) + 16 * h < left ? r[h * V + v] : T(0);
      } else if (along) {
#pragma unroll
        for (int v = 0; v < V; ++v) d[256 / TBM * v * TB_LD] = r[h * V + v];
      } else {
#pragma unroll
        for (int v = 0; v < V; ++v) d[16 * v] = r[h * V + v];
      }
    }
  }
};

// Main loop of the TBM x TBM tile (TBM = 64 or 32) at (m0, n0) of alpha
// op(A) op(B): 4 waves as 2 x 2 quarters of TBM/2 x TBM/2, or (TI = 4, TJ = 1)
// as four strips of 16 columns, each TI x TJ MFMA blocks of 16 x 16; one 32-deep k slice in LDS, the next in
// flight to registers while it is multiplied.  Ends with a barrier after the
// last LDS read, so the caller may overwrite `smem` at once.  A slice takes
// 4.5k cycles alone, 2.0k of them products (FP64, 64 x 64); four workgroups of
// a CU share the rest.  2048 products of order 512: FP64 49.6 TFLOP/s, 44.8
// with 16-deep slices in two buffers and addresses formed for each element.
template <typename T, int TBM, int TI = TBM / 32, int TJ = TBM / 32>
__device__ __forceinline__ void tile_mainloop(int ta, int tb, int M, int N, int K, GlobalC<T> A, long lda,
                                              GlobalC<T> B, long ldb, int m0, int n0, T* smem,
                                              typename BAcc<T>::type (&acc)[TI][TJ])
{
  constexpr int V = TBM / 16;
  T* As = smem;
  T* Bs = smem + TB_BK * TB_LD;
  typedef typename BAcc<T>::type acc_t;
  const int tid = item_tid(), lane = tid & 63, wave = tid >> 6;
  const int wm = TJ == 1 && TBM == 64 ? 0 : wave & 1, wn = TJ == 1 && TBM == 64 ? wave : wave >> 1;
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
  if (K <= 0) return;
  const int lr = lane & 15, lk = lane >> 4;
  SliceLoad<T, TBM> la(A, lda, !ta, m0, M, tid, As), lb(B, ldb, tb, n0, N, tid, Bs);
  const T* ar = As + lk * TB_LD + wm * 16 * TI + lr;
  const T* br = Bs + lk * TB_LD + wn * 16 * TJ + lr;
  T ra[2 * V], rb[2 * V];
  la.load(ra, K, A);
  lb.load(rb, K, B);
  for (int left = K; left > 0; left -= TB_BK) {
    la.store(ra, left);
    lb.store(rb, left);
    slice_barrier();
    if (left > TB_BK) {
      la.load(ra, left - TB_BK, A);
      lb.load(rb, left - TB_BK, B);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (16 * h >= left) break;
#pragma unroll
      for (int ks = 4 * h; ks < 4 * h + 4; ++ks) {
        T af[TI], bf[TJ];
#pragma unroll
        for (int i = 0; i < TI; ++i) af[i] = ar[ks * 4 * TB_LD + i * 16];
#pragma unroll
        for (int j = 0; j < TJ; ++j) bf[j] = br[ks * 4 * TB_LD + j * 16];
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j) acc[i][j] = bmfma(bf[j], af[i], acc[i][j]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    slice_barrier();
  }
}

// Tile element of accumulator register r of block (i, j) held by `lane`:
// row (of op(A) / C) and column (of op(B) / C) inside a TBM x TBM tile.
template <typename T, int TBM = 64>
__device__ __forceinline__ int tile_row(int wave, int lane, int i)
{
  return (wave & 1) * (TBM / 2) + i * 16 + (lane & 15);
}
template <typename T, int TBM = 64>
__device__ __forceinline__ int tile_col(int wave, int lane, int j, int r)
{
  return (wave >> 1) * (TBM / 2) + j * 16 + (sizeof(T) == 8 ? (lane >> 4) + 4 * r : (lane >> 4) * 4 + r);
}

// C tile (tm, tn) of the TBM x TBM tiling of C <- alpha op(A) op(B) + beta C.
template <typename T, int TBM>
__device__ void gemm_tile(int ta, int tb, int M, int N, int K, T alpha, GlobalC<T> A, long lda, GlobalC<T> B, long ldb,
                          T beta, Global<T> C, long ldc, int tm, int tn, T* smem)
{
  constexpr int TQ = TBM / 32;
  typename BAcc<T>::type acc[TQ][TQ];
  const int m0 = tm * TBM, n0 = tn * TBM;
  tile_mainloop<T, TBM>(ta, tb, M, N, K, A, lda, B, ldb, m0, n0, smem, acc);
  const int tid = item_tid(), lane = tid & 63, wave = tid >> 6;
  // C is read whole before it is written: one wait for all, where a load and
  // its use in turn behind each bounds test cost 16 memory latencies a tile
  T c[TQ][TQ][4];
  if (beta != T(0)) {
#pragma unroll
    for (int j = 0; j < TQ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const GlobalC<T> q = C + (long)min(n0 + tile_col<T, TBM>(wave, lane, j, r), N - 1) * ldc;
#pragma unroll
        for (int i = 0; i < TQ; ++i) c[i][j][r] = q[min(m0 + tile_row<T, TBM>(wave, lane, i), M - 1)];
      }
  }
#pragma unroll
  for (int j = 0; j < TQ; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gn = n0 + tile_col<T, TBM>(wave, lane, j, r);
#pragma unroll
      for (int i = 0; i < TQ; ++i) {
        const int gm = m0 + tile_row<T, TBM>(wave, lane, i);
        T v = alpha * acc[i][j][r];
        if (beta != T(0)) v += beta * c[i][j][r];
        if (gm < M && gn < N) C[gm + (long)gn * ldc] = v;
      }
    }
}

// d += (y of lane J of this lane's row of 16 lanes) * m
template <int J>
__device__ __forceinline__ void fmac_row(double& d, double y, double m)
{
  asm volatile("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(d) : "v"(y), "v"(m), "n"(J));
}
template <int J>
__device__ __forceinline__ void fmac_row(float& d, float y, float m)
{
  asm volatile("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(d) : "v"(y), "v"(m), "n"(J));
}

// L x = d for one 16 x 16 block of L: lane i of each row of 16 lanes holds row
// i of -L (l; zero from the diagonal on), 1 / L(i, i) and row i of four columns
// of d.  Row J of the solution is taken when it is complete: what the later
// steps do to it (zero times an infinite solution) stays out.
template <typename T, typename V, int J, int END>
__device__ __forceinline__ void solve16(V& d, V& x, const T (&l)[16], T rinv, int i)
{
  if constexpr (J < END) {
    V y;
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = d[r] * rinv;
    // two wait states between a vector write and its DPP read: the compiler
    // does not look into fmac_row, the selections stand between
    asm volatile("" : "+v"(y));
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = i == J ? y[r] : x[r];
    asm volatile("" : "+v"(x));
    if constexpr (J < 15) {
      const T m = l[J];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        T t = d[r];
        fmac_row<J>(t, y[r], m);
        d[r] = t;
      }
    }
    solve16<T, V, J + 1, END>(d, x, l, rinv, i);
  }
}

// One 64-column panel of a lower-triangular solve L X = alpha B, in place,
// left-looking over 64-row blocks kb, 16 columns a wave:
//   X_kb <- alpha B_kb - L[kb, 0:kb] X[0:kb]   four MFMA blocks a wave
//   X_kb <- L_kk^-1 X_kb                       L_kk in LDS, no barriers
//   X_kb -> global                             (read back by later blocks)
// A wave goes down its 64 x 16 part in strips of 16 rows: solve16 on the strip,
// whose solutions reach the operand layout through LDS, and one product for each
// block below.
// Bound by latency.  Order 1024 with 64 columns alone: 566 us; with the products
// in quarters of 32 x 32, redistributed through LDS, and each strip's part of L
// from memory: 636; with one wave solving a strip of all columns for the others,
// three barriers a strip, and B read one element after the other: 755.  1024
// solves of order 32 to 1024: 739, 799 and 1406 us.  Products by single waves
// straight from memory, without LDS (each wave then loads what the four now
// share): 550 us alone, but 1250 for the 1024 solves.
template <typename T>
__device__ void trsm_panel(const BatchProblem& p, int panel, T* smem)
{
  typedef typename BAcc<T>::type V;
  constexpr int XLD = 17;
  const int tid = item_tid(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int m = p.m, ncp = min(64, p.n - panel * 64), nc = ncp - wave * 16;
  const GlobalC<T> L = (GlobalC<T>)(uintptr_t)p.A;
  const Global<T> Bq = (Global<T>)(uintptr_t)p.C + (long)panel * 64 * p.ldc, Bp = Bq + (long)wave * 16 * p.ldc;
  const long ldl = p.lda, ldb = p.ldc;
  const T alpha = (T)p.alpha;
  T* Ls = smem;                             // tiles (a, b), b <= a, of L_kk by columns
  T* Xt = smem + 2560 + wave * 16 * XLD;    // a strip's solution, for its transpose
  auto col = [&](int r) { return sizeof(T) == 8 ? g + 4 * r : 4 * g + r; };
  for (int kb = 0; kb < m; kb += 64) {
    // addresses are formed anew for each block and strip, not carried along
    int r0 = kb;
    asm volatile("" : "+s"(r0));
    const int h = min(64, m - r0);
    V acc[4][1];
    tile_mainloop<T, 64, 4, 1>(0, 0, h, ncp, r0, L + r0, ldl, Bq, ldb, 0, 0, smem, acc);
    // L_kk to LDS, the diagonal's reciprocals in its place; rows and columns
    // beyond m repeat the last: what they reach is not stored (a tile row at a
    // time: all ten tiles in flight take the registers of the products)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      if (16 * a >= h) break;
      const int ti = tid & 15, q = tid >> 4;
      const GlobalC<T> Lr = L + min(r0 + 16 * a + ti, m - 1);
      T x[4];
#pragma unroll
      for (int b = 0; b <= a; ++b) x[b] = Lr[(long)min(r0 + 16 * b + q, m - 1) * ldl];
      if (ti == q) x[a] = T(1) / x[a];
#pragma unroll
      for (int b = 0; b <= a; ++b) Ls[(a * (a + 1) / 2 + b) * 256 + q * 16 + ti] = x[b];
    }
    if (nc > 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const GlobalC<T> q = Bp + r0 + (long)min(col(r), nc - 1) * ldb;
        T v[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = q[min(16 * b + i, h - 1)];
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[b][0][r] = 16 * b + i < h && col(r) < nc ? alpha * v[b] - acc[b][0][r] : T(0);
      }
    }
    __syncthreads();
    if (nc > 0) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (16 * s >= h) break;
        const T* D = Ls + (s * (s + 1) / 2 + s) * 256;
        T l[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const T v = D[q * 16 + i];
          l[q] = q < i ? -v : T(0);
        }
        V x = {0, 0, 0, 0};
        solve16<T, V, 0, 16>(acc[s][0], x, l, D[17 * i], i);
        const int row = r0 + 16 * s + i;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = col(r);
          if (row < m && c < nc) Bp[row + (long)c * ldb] = x[r];
          Xt[c * XLD + i] = x[r];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        T xo[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) xo[u] = -Xt[i * XLD + 4 * u + g];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int b = s + 1; b < 4; ++b) {
          if (16 * b >= h) break;
          const T* E = Ls + (b * (b + 1) / 2 + s) * 256;
#pragma unroll
          for (int u = 0; u < 4; ++u) acc[b][0] = bmfma(xo[u], E[(4 * u + g) * 16 + i], acc[b][0]);
        }
      }
    }
    __syncthreads();  // X_kb visible to the workgroup's next block; Ls free
  }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void batch_kernel(
    const BatchProblem* __restrict__ probs, const BatchItem* __restrict__ items, int nitems, int* counter)
{
  __shared__ double smem_d[BATCH_SMEM];
  int* next = reinterpret_cast<int*>(smem_d);
  // The first items, the longest, go by position: workgroups c, c + 256, .. share
  // a CU, so that each CU starts with one of the longest; by the counter, in
  // the order of arrival, some start with several (1024 solves of order 32 ..
  // 1024, FP64: 1018 us, then 799).
  for (int it = blockIdx.x; it < nitems;) {
    const BatchItem w = items[it];
    const BatchProblem p = probs[w.prob];
    if (p.kind == 0) {
      const int ta = p.ta != NoTrans, tb = p.tb != NoTrans;
      if (p.dtype == 0) {
        const GlobalC<double> A = (GlobalC<double>)(uintptr_t)p.A;
        const GlobalC<double> B = (GlobalC<double>)(uintptr_t)p.B;
        const Global<double> C = (Global<double>)(uintptr_t)p.C;
        if (w.tile == 32)
          gemm_tile<double, 32>(ta, tb, p.m, p.n, p.k, p.alpha, A, p.lda, B, p.ldb, p.beta, C, p.ldc, w.tm, w.tn,
                                smem_d);
        else
          gemm_tile<double, 64>(ta, tb, p.m, p.n, p.k, p.alpha, A, p.lda, B, p.ldb, p.beta, C, p.ldc, w.tm, w.tn,
                                smem_d);
      } else {
        const GlobalC<float> A = (GlobalC<float>)(uintptr_t)p.A;
        const GlobalC<float> B = (GlobalC<float>)(uintptr_t)p.B;
        const Global<float> C = (Global<float>)(uintptr_t)p.C;
        float* sm = reinterpret_cast<float*>(smem_d);
        if (w.tile == 32)
          gemm_tile<float, 32>(ta, tb, p.m, p.n, p.k, (float)p.alpha, A, p.lda, B, p.ldb, (float)p.beta, C, p.ldc,
                               w.tm, w.tn, sm);
        else
          gemm_tile<float, 64>(ta, tb, p.m, p.n, p.k, (float)p.alpha, A, p.lda, B, p.ldb, (float)p.beta, C, p.ldc,
                               w.tm, w.tn, sm);
      }
    } else {
      // a TRSM panel is a chain of dependent blocks and the longest ones set
      // the batch's time: its waves issue ahead of the GEMM items beside them
      __builtin_amdgcn_s_setprio(2);
      if (p.dtype == 0) trsm_panel<double>(p, w.tn, smem_d);
      else trsm_panel<float>(p, w.tn, reinterpret_cast<float*>(smem_d));
      __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();  // smem free for the next item index
    if (threadIdx.x == 0) *next = (int)gridDim.x + atomicAdd(counter, 1);
    __syncthreads();
    it = __builtin_amdgcn_readfirstlane(*next);
    __syncthreads();
  }
}

// ---------------------------------------------------------------- plan
struct BatchPlan {
  BatchProblem* d_probs = nullptr;
  BatchItem* d_items = nullptr;
  int* d_counter = nullptr;
  int nitems = 0, nprobs = 0;
  int grid = 0;
  double flops = 0.0, bytes = 0.0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

static void enqueue_run(BatchPlan* pl, hipStream_t s)
{
  fill_int(s, pl->d_counter, 1, 0);
  hipLaunchKernelGGL(batch_kernel, dim3(pl->grid), dim3(256), 0, s, pl->d_probs, pl->d_items, pl->nitems,
                     pl->d_counter);
  XK_HIP(hipGetLastError());
}

// Work list of a batch: one item per 64 x 64 GEMM tile and per 64-column
// TRSM panel, sorted by estimated cost, longest first (ties keep problem
// order).  batch_count_items counts the items; batch_build fills hp[count]
// and work[], returns the item count and adds the batch's flops and bytes.
struct BatchCost {
  double c;
  long seq;
  BatchItem w;
};

// GEMM item shape: 1 = 32 x 32 tiles for a problem whose 32 x 32 tiling
// covers at most 3/4 of the area the 64 x 64 one does (a small m or n), 2 =
// 32 x 32 only, 3 = 64 x 64 only, 0 (default) = rule 1 for FP64 problems and
// 64 x 64 for FP32 ones (XKBLAS_BATCH_TILE).  On the uneven batch of 4096
// GEMMs + 1024 TRSMs (MI355X, two draws of sizes), FP64: per problem 1342 and
// 1407 us, 64 x 64 1312 and 1378, 32 x 32 1790 and 1846 (the documented default
// stays, 2 % from the best); FP32: 64 x 64 857 and 896, per problem 923 and
// 958, 32 x 32 1444 and 1489.
static int g_batch_tile = getenv("XKBLAS_BATCH_TILE") ? atoi(getenv("XKBLAS_BATCH_TILE")) : 0;

static int gemm_item_tile(int m, int n, int dtype)
{
  const int mode = g_batch_tile == 0 ? (dtype == 0 ? 1 : 3) : g_batch_tile;
  if (mode == 3) return 64;
  if (mode == 2) return 32;
  const long a64 = (long)((m + 63) / 64) * ((n + 63) / 64) * 4096;
  const long a32 = (long)((m + 31) / 32) * ((n + 31) / 32) * 1024;
  return 4 * a32 <= 3 * a64 ? 32 : 64;
}

static long batch_count_items(const xkblas_batch_problem_t* probs, int count)
{
  long n = 0;
  for (int i = 0; i < count; ++i) {
    const xkblas_batch_problem_t& q = probs[i];
    if (q.m <= 0 || q.n <= 0) continue;
    if (q.kind == XKBLAS_BATCH_GEMM) {
      const int t = gemm_item_tile(q.m, q.n, q.dtype);
      n += (long)((q.m + t - 1) / t) * ((q.n + t - 1) / t);
    } else {
      n += (q.n + 63) / 64;
    }
  }
  return n;
}

static long batch_build(const xkblas_batch_problem_t* probs, int count, BatchProblem* hp, BatchCost* work,
                        double* flops, double* bytes)
{
  long nw = 0;
  for (int i = 0; i < count; ++i) {
    const xkblas_batch_problem_t& q = probs[i];
    BatchProblem& p = hp[i];
    p.kind = q.kind; p.dtype = q.dtype; p.ta = q.transA; p.tb = q.transB;
    p.m = q.m; p.n = q.n; p.k = q.k; p.alpha = q.alpha; p.beta = q.beta;
    p.A = q.A; p.lda = q.lda; p.B = q.B; p.ldb = q.ldb; p.C = q.C; p.ldc = q.ldc;
    const double elt = q.dtype == 0 ? 8.0 : 4.0;
    XK_CHECK(q.kind == XKBLAS_BATCH_GEMM || q.kind == XKBLAS_BATCH_TRSM, "batch: unknown problem kind");
    XK_CHECK(q.dtype == 0 || q.dtype == 1, "batch: dtype must be 0 (FP64) or 1 (FP32)");
    if (q.m <= 0 || q.n <= 0) continue;
    if (q.kind == XKBLAS_BATCH_GEMM) {
      const int t = gemm_item_tile(q.m, q.n, q.dtype);
      const int tmx = (q.m + t - 1) / t, tnx = (q.n + t - 1) / t;
      // a tile's k-loop work plus a fixed overhead (a 32 x 32 tile runs at a
      // quarter of the MFMA work per slice, hence the same time per k as half
      // of a 64 x 64 one)
      const double c = t == 64 ? 2.0 * 64 * 64 * std::max(q.k, 1) + 64 * 64 * 8.0
                               : 2.0 * 64 * 32 * std::max(q.k, 1) + 64 * 64 * 8.0;
      for (int a = 0; a < tmx; ++a)
        for (int b = 0; b < tnx; ++b) {
          work[nw] = BatchCost{c, nw, BatchItem{i, a, b, t}};
          ++nw;
        }
      *flops += 2.0 * q.m * q.n * (double)q.k;
      *bytes += elt * ((double)q.m * q.k + (double)q.k * q.n + 2.0 * q.m * q.n);
    } else {
      const int np = (q.n + 63) / 64;
      // left-looking blocks: one tile of k = 64 kb each plus the block's
      // solve, priced like a tile of k = 128
      const double nbk = (q.m + 63) / 64;
      const double c = 2.0 * 64 * 64 * 64 * nbk * (nbk - 1) / 2 + nbk * 2.0 * 64 * 64 * 128;
      for (int b = 0; b < np; ++b) {
        work[nw] = BatchCost{c, nw, BatchItem{i, 0, b, 64}};
        ++nw;
      }
      *flops += (double)q.m * q.m * q.n;
      *bytes += elt * (0.5 * (double)q.m * q.m + 2.0 * q.m * q.n);
    }
  }
  std::sort(work, work + nw,
            [](const BatchCost& a, const BatchCost& b) { return a.c > b.c || (a.c == b.c && a.seq < b.seq); });
  return nw;
}

// workgroups of the persistent kernel: as many as can be resident at once
static int batch_grid(long nitems)
{
  int dev = 0, cus = 0, per_cu = 0;
  XK_HIP(hipGetDevice(&dev));
  XK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  XK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, batch_kernel, 256, 0));
  return (int)std::max(1L, std::min((long)cus * std::max(per_cu, 1), std::max(nitems, 1L)));
}

// ---- allocation-free runs
// xkblas_batch_run_noalloc serves callers that cannot allocate device
// memory: its counter, problem list and work list live in one fixed device
// array (`scratch`, below; one copy per GPU, held until the process ends),
// whose device address hipGetSymbolAddress gives at initialisation.  The
// host-side lists are built in fixed host arrays, so the call allocates
// nothing on the host either.  Calls share the array: they are ordered on
// the library's compute stream, and calls that overlap on one GPU from
// other streams would race.
constexpr int NOALLOC_MAX_PROBS = 8192;
constexpr long NOALLOC_MAX_ITEMS = 196608;
constexpr size_t NOALLOC_PROBS_OFF = 256;  // the work counter comes first
constexpr size_t NOALLOC_ITEMS_OFF = NOALLOC_PROBS_OFF + sizeof(BatchProblem) * NOALLOC_MAX_PROBS;
constexpr size_t NOALLOC_BYTES = NOALLOC_ITEMS_OFF + sizeof(BatchItem) * NOALLOC_MAX_ITEMS;
constexpr int NOALLOC_MAX_DEVICES = 64;

static char* g_noalloc_dev[NOALLOC_MAX_DEVICES];  // device address of `scratch`, per GPU
static BatchProblem g_noalloc_probs[NOALLOC_MAX_PROBS];
static BatchCost g_noalloc_work[NOALLOC_MAX_ITEMS];
static BatchItem g_noalloc_items[NOALLOC_MAX_ITEMS];
static hipEvent_t g_noalloc_staged = nullptr;  // the last run's copies have read the host lists

}  // namespace xk

// 3.9 MB: counter, NOALLOC_MAX_PROBS problems, NOALLOC_MAX_ITEMS work items.
// In host code this name is only the symbol's host-side handle: kernels get
// the address hipGetSymbolAddress returns.
static __device__ __align__(256) char scratch[xk::NOALLOC_BYTES];

namespace xk {

void batch_noalloc_init()
{
  int dev = 0;
  XK_HIP(hipGetDevice(&dev));
  XK_CHECK(dev >= 0 && dev < NOALLOC_MAX_DEVICES, "device ordinal beyond the allocation-free table");
  if (g_noalloc_dev[dev]) return;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(::scratch));
  if (e != hipSuccess || !p) fatal("hipGetSymbolAddress(scratch)", __FILE__, __LINE__, hipGetErrorString(e));
  g_noalloc_dev[dev] = static_cast<char*>(p);
  if (!g_noalloc_staged) XK_HIP(hipEventCreateWithFlags(&g_noalloc_staged, hipEventDisableTiming));
}

}  // namespace xk

using namespace xk;

extern "C" {

void* xkblas_batch_create(const xkblas_batch_problem_t* probs, int count)
{
  if (count < 0 || (count > 0 && !probs)) return nullptr;
  xkblas_init();
  BatchPlan* pl = new BatchPlan();
  std::vector<BatchProblem> hp(std::max(count, 1));
  std::vector<BatchCost> work(std::max(batch_count_items(probs, count), 1L));
  const long nw = batch_build(probs, count, hp.data(), work.data(), &pl->flops, &pl->bytes);
  std::vector<BatchItem> items(std::max(nw, 1L));
  for (long i = 0; i < nw; ++i) items[i] = work[i].w;
  pl->nitems = (int)nw;
  pl->nprobs = count;
  XK_HIP(hipMalloc(&pl->d_probs, sizeof(BatchProblem) * std::max(count, 1)));
  XK_HIP(hipMalloc(&pl->d_items, sizeof(BatchItem) * items.size()));
  XK_HIP(hipMalloc(&pl->d_counter, sizeof(int)));
  if (count) XK_HIP(hipMemcpy(pl->d_probs, hp.data(), sizeof(BatchProblem) * count, hipMemcpyHostToDevice));
  if (nw) XK_HIP(hipMemcpy(pl->d_items, items.data(), sizeof(BatchItem) * nw, hipMemcpyHostToDevice));
  pl->grid = batch_grid(nw);
  return pl;
}

int xkblas_batch_run(void* plan)
{
  BatchPlan* pl = static_cast<BatchPlan*>(plan);
  if (!pl) return -1;
  std::lock_guard<std::mutex> lock(api_mutex());
  Runtime& r = rt();
  r.begin_compute("batch", pl->flops, nullptr);
  if (pl->exec) XK_HIP(hipGraphLaunch(pl->exec, r.s_comp));
  else enqueue_run(pl, r.s_comp);
  r.prof_end();
  return 0;
}

int xkblas_batch_run_noalloc(const xkblas_batch_problem_t* problems, int count)
{
  if (count < 0 || (count > 0 && !problems)) return -1;
  if (count > NOALLOC_MAX_PROBS) {
    fprintf(stderr, "[xkblas_amd] xkblas_batch_run_noalloc: %d problems exceed the maximum of %d\n", count,
            NOALLOC_MAX_PROBS);
    return -2;
  }
  const long nw = batch_count_items(problems, count);
  if (nw > NOALLOC_MAX_ITEMS) {
    fprintf(stderr, "[xkblas_amd] xkblas_batch_run_noalloc: %ld work items exceed the maximum of %ld\n", nw,
            NOALLOC_MAX_ITEMS);
    return -3;
  }
  std::lock_guard<std::mutex> lock(api_mutex());
  Runtime& r = rt();
  if (!r.device_ready) {
    fprintf(stderr, "[xkblas_amd] xkblas_batch_run_noalloc: call xkblas_init first\n");
    return -4;
  }
  int dev = 0;
  XK_HIP(hipGetDevice(&dev));
  XK_CHECK(dev >= 0 && dev < NOALLOC_MAX_DEVICES && g_noalloc_dev[dev], "allocation-free array not set up");
  char* base = g_noalloc_dev[dev];
  // the previous run's copies must have read the host lists before they change
  XK_HIP(hipEventSynchronize(g_noalloc_staged));
  double flops = 0.0, bytes = 0.0;
  batch_build(problems, count, g_noalloc_probs, g_noalloc_work, &flops, &bytes);
  for (long i = 0; i < nw; ++i) g_noalloc_items[i] = g_noalloc_work[i].w;
  BatchProblem* d_probs = reinterpret_cast<BatchProblem*>(base + NOALLOC_PROBS_OFF);
  BatchItem* d_items = reinterpret_cast<BatchItem*>(base + NOALLOC_ITEMS_OFF);
  int* d_counter = reinterpret_cast<int*>(base);
  r.stamp_written("batch", flops, nullptr);
  r.before_compute();
  if (count)
    XK_HIP(hipMemcpyAsync(d_probs, g_noalloc_probs, sizeof(BatchProblem) * count, hipMemcpyHostToDevice, r.s_comp));
  if (nw) XK_HIP(hipMemcpyAsync(d_items, g_noalloc_items, sizeof(BatchItem) * nw, hipMemcpyHostToDevice, r.s_comp));
  XK_HIP(hipEventRecord(g_noalloc_staged, r.s_comp));
  fill_int(r.s_comp, d_counter, 1, 0);
  hipLaunchKernelGGL(batch_kernel, dim3(batch_grid(nw)), dim3(256), 0, r.s_comp, d_probs, d_items, (int)nw,
                     d_counter);
  XK_HIP(hipGetLastError());
  return 0;
}

void xkblas_set_batch_tile(int mode)
{
  std::lock_guard<std::mutex> lock(api_mutex());
  g_batch_tile = mode < 0 || mode > 3 ? 0 : mode;
}

int xkblas_batch_use_graph(void* plan, int on)
{
  BatchPlan* pl = static_cast<BatchPlan*>(plan);
  if (!pl) return -1;
  std::lock_guard<std::mutex> lock(api_mutex());
  Runtime& r = rt();
  if (pl->exec) {
    XK_HIP(hipGraphExecDestroy(pl->exec));
    XK_HIP(hipGraphDestroy(pl->graph));
    pl->exec = nullptr;
    pl->graph = nullptr;
  }
  if (!on) return 0;
  XK_HIP(hipStreamSynchronize(r.s_comp));
  XK_HIP(hipStreamBeginCapture(r.s_comp, hipStreamCaptureModeThreadLocal));
  enqueue_run(pl, r.s_comp);
  XK_HIP(hipStreamEndCapture(r.s_comp, &pl->graph));
  XK_HIP(hipGraphInstantiate(&pl->exec, pl->graph, nullptr, nullptr, 0));
  return 0;
}

int xkblas_batch_info(void* plan, int* nitems, int* grid, double* flops, double* bytes)
{
  BatchPlan* pl = static_cast<BatchPlan*>(plan);
  if (!pl) return -1;
  if (nitems) *nitems = pl->nitems;
  if (grid) *grid = pl->grid;
  if (flops) *flops = pl->flops;
  if (bytes) *bytes = pl->bytes;
  return 0;
}

void xkblas_batch_destroy(void* plan)
{
  BatchPlan* pl = static_cast<BatchPlan*>(plan);
  if (!pl) return;
  XK_HIP(hipDeviceSynchronize());
  if (pl->exec) {
    (void)hipGraphExecDestroy(pl->exec);
    (void)hipGraphDestroy(pl->graph);
  }
  (void)hipFree(pl->d_probs);
  (void)hipFree(pl->d_items);
  (void)hipFree(pl->d_counter);
  delete pl;
}

void* xkblas_device_malloc(size_t bytes)
{
  xkblas_init();
  void* p = nullptr;
  if (hipMalloc(&p, bytes ? bytes : 1) != hipSuccess) return nullptr;
  return p;
}

void xkblas_device_free(void* p)
{
  if (p) {
    (void)hipDeviceSynchronize();
    (void)hipFree(p);
  }
}

int xkblas_memcpy_htod(void* dst, const void* src, size_t bytes)
{
  return hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice) == hipSuccess ? 0 : -1;
}

int xkblas_memcpy_dtoh(void* dst, const void* src, size_t bytes)
{
  return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost) == hipSuccess ? 0 : -1;
}

}  // extern "C"
