// gemm.hip — FP64/FP32 MFMA GEMM for gfx950 (the tile body of every BLAS-3
// call in the library): gemm_dma_kernel for aligned operands, gemm_kernel for
// the rest.
//
// Work decomposition of gemm_kernel.  One workgroup (4 waves, 256 lanes) owns a BM x BN
// macro tile of C; each wave owns a (BM/2) x (BN/2) quarter as (BM/32) x
// (BN/32) accumulators of 16x16 (v_mfma_*_16x16x4: 4 doubles / floats per
// lane).  The k loop streams BK-deep slices of op(A) and op(B) through two
// LDS buffers: the next slice is loaded from HBM into registers while the
// current one feeds the MFMAs, then written to the other buffer; one barrier
// per slice.  LDS rows are k-major (op(A)[k][m], op(B)[k][n]) so every MFMA
// operand read is 16 consecutive elements per 16 lanes.
//
// The MFMA is issued with op(B) as its first operand, so the accumulator holds
// C^T in the hardware's output layout: lane l, register r holds
// C[m = 16*tile + l%16][n = 16*tile + q(l,r)] with q = l/16 + 4r for
// v_mfma_f64_16x16x4f64 and q = 4(l/16) + r for v_mfma_f32_16x16x4f32.
// Sixteen consecutive lanes then store 16 consecutive rows of one column:
// 128-byte segments of the column-major C.
//
// Tile order.  Workgroup ids are dealt round-robin to the 8 XCDs; the id is
// remapped so each XCD receives a contiguous range of tiles, and tiles are
// rastered in groups of 8 tile rows so that concurrently running tiles of one
// XCD share op(A) panels in its L2.
#include "common.h"
#include <algorithm>
#include <cmath>
#include <type_traits>
#include "tiles.h"
#include "kernels.h"

namespace xk {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

template <typename T> struct AccT;
template <> struct AccT<double> { typedef d4_t type; };
template <> struct AccT<float> { typedef f4_t type; };

__device__ __forceinline__ d4_t mfma16(double a, double b, d4_t c)
{
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4_t mfma16(float a, float b, f4_t c)
{
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <typename T>
struct GemmParams {
  int m, n, k;
  int tiles_m, tiles_n;
  int tri;
  int trap;        // triangle-masked output that is not square: full tile raster, tiles outside it leave at once
  int whole;       // tiles of gemm_dma_mixed_kernel's first part
  int kmode;       // inner range per tile for a triangular operand (KRANGE_*)
  int kpart;       // > 0: batch entry z multiplies the z-th kpart of the inner dimension
  int vecA, vecB;  // 16-byte vector loads allowed (base and ld aligned)
  int prio;        // raise the waves' issue priority (latency-bound chain steps)
  T alpha, beta;
  const T* A;
  long lda, sA;
  const T* B;
  long ldb, sB;
  T* C;
  long ldc, sC;
};

typedef __attribute__((address_space(3))) void lds_void;

// at most CNT vector memory operations still in flight
template <int CNT>
__device__ __forceinline__ void wait_vmcnt()
{
  static_assert(CNT < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((CNT & 15) | ((CNT >> 4) << 14) | 0x0f70);
}

// A barrier behind which LDS data written with stores or, once wait_vmcnt has
// seen it land, with direct loads is there for every wave; direct loads not
// waited for stay in flight over it.  (A release fence of the workgroup would
// wait for them: the compiler counts them as LDS writes.)
__device__ __forceinline__ void stage_barrier()
{
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// Load V consecutive elements starting at p (16-byte aligned when vec).
template <typename T, int V>
__device__ __forceinline__ void load_run(const T* p, T (&r)[V])
{
  static_assert((V * sizeof(T)) % 16 == 0, "run must be a multiple of 16 bytes");
  typedef float4 v16;
  const v16* q = reinterpret_cast<const v16*>(p);
#pragma unroll
  for (int i = 0; i < (int)(V * sizeof(T) / 16); ++i) {
    v16 x = q[i];
    __builtin_memcpy(reinterpret_cast<char*>(r) + 16 * i, &x, 16);
  }
}

// Tile (tm, tn) at place `at` of the raster: groups of 8 tile rows, column by
// column inside a group; a square triangle's tiles only.
template <typename T>
__device__ __forceinline__ void tile_raster(const GemmParams<T>& p, int at, int& tm, int& tn)
{
  if (p.tri == TRI_FULL || p.trap) {
    constexpr int GM = 8;
    const int group = GM * p.tiles_n;
    const int g = at / group;
    const int first = g * GM;
    const int gm = min(p.tiles_m - first, GM);
    const int r = at - g * group;
    tm = first + r % gm;
    tn = r / gm;
  } else {
    int i, j;
    tri_raster<8>(at, p.tiles_m, i, j);
    if (p.tri == TRI_LOWER) { tm = i; tn = j; }
    else { tm = j; tn = i; }
  }
}

// Whether a BM x BN tile at (m0, n0) holds anything to write.
template <int BM, int BN, typename T>
__device__ __forceinline__ bool tile_holds(const GemmParams<T>& p, int m0, int n0)
{
  if (m0 >= p.m || n0 >= p.n) return false;
  return p.tri == TRI_FULL || (p.tri == TRI_LOWER ? m0 + BM > n0 : n0 + BN > m0);
}

// First row and column of this workgroup's BM x BN tile; false when there is
// nothing of it to write.
template <int BM, int BN, typename T>
__device__ __forceinline__ bool tile_origin(const GemmParams<T>& p, int& m0, int& n0)
{
  int at = blockIdx.x, tm, tn;
  // a limited inner range makes the work per tile grow along the tile rows or
  // columns: no XCD blocking then (consecutive ids go to different XCDs, which
  // then share light and heavy tiles alike), and the heaviest tiles are
  // dispatched first
  if (p.kmode == KRANGE_ALL) at = xcd_range(at, gridDim.x);
  tile_raster(p, at, tm, tn);
  if (p.kmode == KRANGE_A_LOWER) tm = p.tiles_m - 1 - tm;
  else if (p.kmode == KRANGE_B_UPPER) tn = p.tiles_n - 1 - tn;
  m0 = tm * BM;
  n0 = tn * BN;
  return tile_holds<BM, BN>(p, m0, n0);
}

// C = alpha acc + beta C on the selected triangle: the wave's TM x TN blocks
// of 16 x 16 at rows gm0, columns gn0.
template <typename T, int TM, int TN>
__device__ __forceinline__ void store_tile(const GemmParams<T>& p, T* __restrict__ C, int gm0, int gn0, int lane,
                                           const typename AccT<T>::type (&acc)[TM][TN])
{
  const T alpha = p.alpha, beta = p.beta;
  const int lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int gm = gm0 + i * 16 + lr;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // output row of the 16x16 MFMA block held by (lane, r): f64 uses
        // lane/16 + 4r, f32 uses 4(lane/16) + r (measured on gfx950)
        const int gn = gn0 + j * 16 + (sizeof(T) == 8 ? lk + 4 * r : lk * 4 + r);
        bool ok = gm < p.m && gn < p.n;
        if (p.tri == TRI_LOWER) ok = ok && gm >= gn;
        else if (p.tri == TRI_UPPER) ok = ok && gm <= gn;
        if (ok) {
          T* c = C + (long)gm + (long)gn * p.ldc;
          T v = alpha * acc[i][j][r];
          if (beta != T(0)) v += beta * *c;
          *c = v;
        }
      }
    }
  }
}

template <typename T, int BM, int BN, int BK, bool TA, bool TB>
__global__ __launch_bounds__(256) void gemm_kernel(GemmParams<T> p)
{
  constexpr int PAD = 16 / sizeof(T);
  constexpr int LA = BM + PAD, LB = BN + PAD;
  constexpr int VA = BM * BK / 256;  // elements of op(A) per lane per slice
  constexpr int VB = BN * BK / 256;
  constexpr int WTM = BM / 2, WTN = BN / 2;  // wave tile
  constexpr int TM = WTM / 16, TN = WTN / 16;
  typedef typename AccT<T>::type acc_t;

  __shared__ T As[2][BK][LA];
  __shared__ T Bs[2][BK][LB];
  if (p.prio) __builtin_amdgcn_s_setprio(3);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;

  const T* __restrict__ A = p.A + (long)blockIdx.z * p.sA;
  const T* __restrict__ B = p.B + (long)blockIdx.z * p.sB;
  T* __restrict__ C = p.C + (long)blockIdx.z * p.sC;

  const int M = p.m, N = p.n, K = p.kpart ? min(p.kpart, p.k - (int)blockIdx.z * p.kpart) : p.k;
  int m0, n0;
  if (!tile_origin<BM, BN>(p, m0, n0)) return;

  // ---- per-lane load coordinates
  // op(A) slice BM x BK.  !TA: runs along m.  TA: runs along k.
  int a_r, a_c;  // row (m) and column (k) of the run start inside the slice
  if (!TA) { a_c = tid / (BM / VA); a_r = (tid % (BM / VA)) * VA; }
  else     { a_r = tid / (BK / VA); a_c = (tid % (BK / VA)) * VA; }
  // op(B) slice BK x BN.  !TB: runs along k.  TB: runs along n.
  int b_r, b_c;  // k and n of the run start
  if (!TB) { b_c = tid / (BK / VB); b_r = (tid % (BK / VB)) * VB; }
  else     { b_r = tid / (BN / VB); b_c = (tid % (BN / VB)) * VB; }

  T ra[VA], rb[VB];

  auto load_slice = [&](int k0) {
    const bool fullA = p.vecA && (m0 + BM <= M) && (k0 + BK <= K);
    const bool fullB = p.vecB && (n0 + BN <= N) && (k0 + BK <= K);
    if (!TA) {
      const T* src = A + (long)(m0 + a_r) + (long)(k0 + a_c) * p.lda;
      if (fullA) load_run<T, VA>(src, ra);
      else {
#pragma unroll
        for (int v = 0; v < VA; ++v)
          ra[v] = (m0 + a_r + v < M && k0 + a_c < K) ? src[v] : T(0);
      }
    } else {
      const T* src = A + (long)(k0 + a_c) + (long)(m0 + a_r) * p.lda;
      if (fullA) load_run<T, VA>(src, ra);
      else {
#pragma unroll
        for (int v = 0; v < VA; ++v)
          ra[v] = (m0 + a_r < M && k0 + a_c + v < K) ? src[v] : T(0);
      }
    }
    if (!TB) {
      const T* src = B + (long)(k0 + b_r) + (long)(n0 + b_c) * p.ldb;
      if (fullB) load_run<T, VB>(src, rb);
      else {
#pragma unroll
        for (int v = 0; v < VB; ++v)
          rb[v] = (k0 + b_r + v < K && n0 + b_c < N) ? src[v] : T(0);
      }
    } else {
      const T* src = B + (long)(n0 + b_c) + (long)(k0 + b_r) * p.ldb;
      if (fullB) load_run<T, VB>(src, rb);
      else {
#pragma unroll
        for (int v = 0; v < VB; ++v)
          rb[v] = (k0 + b_r < K && n0 + b_c + v < N) ? src[v] : T(0);
      }
    }
  };

  auto store_slice = [&](int buf) {
    if (!TA) {
#pragma unroll
      for (int v = 0; v < VA; ++v) As[buf][a_c][a_r + v] = ra[v];
    } else {
#pragma unroll
      for (int v = 0; v < VA; ++v) As[buf][a_c + v][a_r] = ra[v];
    }
    if (!TB) {
#pragma unroll
      for (int v = 0; v < VB; ++v) Bs[buf][b_r + v][b_c] = rb[v];
    } else {
#pragma unroll
      for (int v = 0; v < VB; ++v) Bs[buf][b_r][b_c + v] = rb[v];
    }
  };

  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  // inner range: all of k, or the part where a triangular op(A) / op(B) of
  // this tile row / column is not zero (the rest would add exact zeros)
  int kbeg = 0, kend = K;
  if (p.kmode == KRANGE_A_LOWER) kend = min(K, m0 + BM);
  else if (p.kmode == KRANGE_A_UPPER) kbeg = m0;
  else if (p.kmode == KRANGE_B_UPPER) kend = min(K, n0 + BN);
  else if (p.kmode == KRANGE_B_LOWER) kbeg = n0;
  const int kt0 = kbeg / BK;
  const int nk = (kend + BK - 1) / BK;
  const int lr = lane & 15, lk = lane >> 4;
  if (nk > kt0) {
    load_slice(kt0 * BK);
    store_slice(0);
    __syncthreads();
    int buf = 0;
    for (int kt = kt0; kt < nk; ++kt) {
      const bool more = kt + 1 < nk;
      if (more) load_slice((kt + 1) * BK);
#pragma unroll
      for (int ks = 0; ks < BK / 4; ++ks) {
        T af[TM], bf[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) af[i] = As[buf][ks * 4 + lk][wm * WTM + i * 16 + lr];
#pragma unroll
        for (int j = 0; j < TN; ++j) bf[j] = Bs[buf][ks * 4 + lk][wn * WTN + j * 16 + lr];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = mfma16(bf[j], af[i], acc[i][j]);
      }
      if (more) store_slice(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }

  store_tile<T, TM, TN>(p, C, m0 + wm * WTM, n0 + wn * WTN, lane, acc);
}

// The kernel of aligned operands (16-byte base and leading dimension).  A
// workgroup of four waves owns a BM x BM tile, each wave a quarter; slices of
// 128 bytes of the inner dimension (16 doubles, 32 floats) go from memory
// straight to LDS (1 KB per instruction, no registers between) through a ring
// of NST stages: the loads of NST - 1 stages are in flight while one is
// multiplied, one barrier per stage, which waits for the stage it opens alone
// (with every load waited for, 32 x 32 tiles: FP64 512^3 19.0 us, then 16.7;
// FP32 12.4, 11.7; larger tiles and the quarters alike).
// An operand whose rows (op(A): m, op(B): n) are contiguous in memory is kept
// k-major, block b of 16 elements of row k at b ^ swizzle(k); one whose inner
// index is contiguous is kept row-major (128 bytes a row), chunk c (16 bytes)
// of row m at c ^ (m / 2 % 8): with these places every operand read (b64 or
// b32 per lane) meets each bank once.  Rows beyond the matrix repeat its last
// one (they only reach results that are not stored); a remainder of the inner
// dimension is staged through registers with zeros.  A wave whose quarter
// lies partly or wholly beyond the matrix multiplies only the 16 x 16 blocks
// that hold results.
// The inner order per element is gemm_kernel's: the same bits.
template <typename T, int BM, int NST, bool TA, bool TB>
__device__ __forceinline__ void dma_tile_body(const GemmParams<T>& p, char* S, int m0, int n0)
{
  constexpr int SZ = sizeof(T), E = 16 / SZ, BK = 128 / SZ;
  constexpr int OP = BM * 128;      // bytes of one operand's stage
  constexpr int CR = BM * SZ / 16;  // chunks of a k-major row
  constexpr int Q = BM / 32;        // load instructions per wave, operand and stage
  constexpr int TQ = BM / 32;       // 16 x 16 blocks of a wave's quarter, each way
  typedef typename AccT<T>::type acc_t;
  if (p.prio) __builtin_amdgcn_s_setprio(3);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const T* __restrict__ A = p.A + (long)blockIdx.z * p.sA;
  const T* __restrict__ B = p.B + (long)blockIdx.z * p.sB;
  T* __restrict__ C = p.C + (long)blockIdx.z * p.sC;
  const int M = p.m, N = p.n, K = p.kpart ? min(p.kpart, p.k - (int)blockIdx.z * p.kpart) : p.k;

  // block permutation of k-major row k: rows that the lanes of one read take
  // together (k .. k + 3) fall into different banks
  auto swizzle = [](int k) { return SZ == 8 ? k & 1 : BM == 32 ? (k >> 1) & 1 : k & 3; };
  // Place q of this lane in a stage of an operand: 16 bytes, elements
  // (row, k ..) row-major or (row .., k) k-major of the tile.
  auto place = [&](bool kmajor, int q, int& row, int& k) {
    const int idx = (wave * Q + q) * 64 + lane;
    if (kmajor) {
      k = idx / CR;
      row = ((idx % CR) ^ (swizzle(k) * (16 / E))) * E;
    } else {
      row = idx >> 3;
      k = ((idx & 7) ^ ((row >> 1) & 7)) * E;
    }
  };
  // byte offsets of those elements from the tile's first row at k = 0
  unsigned offA[Q], offB[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    int row, k;
    place(!TA, q, row, k);
    row = TA ? min(row, M - 1 - m0) : min(row, (M - 1) / E * E - m0);
    offA[q] = (unsigned)(TA ? k + row * p.lda : row + k * p.lda) * SZ;
    place(TB, q, row, k);
    row = TB ? min(row, (N - 1) / E * E - n0) : min(row, N - 1 - n0);
    offB[q] = (unsigned)(TB ? row + k * p.ldb : k + row * p.ldb) * SZ;
  }
  const char* A0 = reinterpret_cast<const char*>(TA ? A + m0 * p.lda : A + m0);
  const char* B0 = reinterpret_cast<const char*>(TB ? B + n0 : B + n0 * p.ldb);
  const long stepA = (TA ? 1 : p.lda) * SZ, stepB = (TB ? p.ldb : 1) * SZ;  // bytes per k
  auto issue = [&](int buf, int k0) {
    const char* a = A0 + k0 * stepA;
    const char* b = B0 + k0 * stepB;
    char* s = S + buf * 2 * OP + wave * (Q * 1024);
#pragma unroll
    for (int q = 0; q < Q; ++q)
      __builtin_amdgcn_global_load_lds((const void*)(a + offA[q]), (lds_void*)(s + q * 1024), 16, 0, 0);
#pragma unroll
    for (int q = 0; q < Q; ++q)
      __builtin_amdgcn_global_load_lds((const void*)(b + offB[q]), (lds_void*)(s + OP + q * 1024), 16, 0, 0);
  };
  // the same through registers, zeros from k = kend on
  auto issue_tail = [&](int buf, int k0, int kend) {
#pragma unroll
    for (int op = 0; op < 2; ++op) {
      const bool kmajor = op == 0 ? !TA : TB;
      const char* base = op == 0 ? A0 + k0 * stepA : B0 + k0 * stepB;
      const int rows = op == 0 ? M - m0 : N - n0;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        int row, k;
        place(kmajor, q, row, k);
        T v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const int rr = row + (kmajor ? e : 0), kk = k + (kmajor ? 0 : e);
          v[e] = rr < rows && k0 + kk < kend
                     ? *reinterpret_cast<const T*>(base + (op == 0 ? offA[q] : offB[q]) + e * SZ) : T(0);
        }
        __builtin_memcpy(S + buf * 2 * OP + op * OP + (wave * Q + q) * 1024 + lane * 16, v, 16);
      }
    }
    // a wave all of whose loads here are masked off adds none to the count of
    // those in flight: with the earlier stages landed now, the counted waits
    // of the loop hold whatever it is
    wait_vmcnt<0>();
  };

  acc_t acc[TQ][TQ];
#pragma unroll
  for (int i = 0; i < TQ; ++i)
#pragma unroll
    for (int j = 0; j < TQ; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  const int lr = lane & 15, lk = lane >> 4;
  // operand element of block i, inner index 4 s + lk, in a stage
  auto operand = [&](const char* s, bool kmajor, int w, int i, int ks) -> T {
    const int k = ks * 4 + lk;
    int off;
    if (kmajor) off = k * (BM * SZ) + (((w * TQ + i) ^ swizzle(k)) * 16 + lr) * SZ;
    else off = (w * (BM / 2) + i * 16 + lr) * 128 + ((k / E) ^ ((lr >> 1) & 7)) * 16 + (k % E) * SZ;
    return *reinterpret_cast<const T*>(s + off);
  };

  int kbeg = 0, kend = K;
  if (p.kmode == KRANGE_A_LOWER) kend = min(K, m0 + BM);
  else if (p.kmode == KRANGE_A_UPPER) kbeg = m0;
  else if (p.kmode == KRANGE_B_UPPER) kend = min(K, n0 + BM);
  else if (p.kmode == KRANGE_B_LOWER) kbeg = n0;
  const int nk = (kend - kbeg + BK - 1) / BK;
  auto stage = [&](int kt) {
    const int k0 = kbeg + kt * BK;
    if (k0 + BK <= kend) issue(kt % NST, k0);
    else issue_tail(kt % NST, k0, kend);
  };
  // blocks of this wave's quarter that hold results
  const int ni = min(TQ, max(0, (M - m0 - wm * (BM / 2) + 15) >> 4));
  const int nj = min(TQ, max(0, (N - n0 - wn * (BM / 2) + 15) >> 4));
#pragma unroll
  for (int st = 0; st < NST - 1; ++st)
    if (st < nk) stage(st);
  // the waves of a workgroup meet in the same barriers whichever loop they run
  auto loop = [&](auto whole) {
    for (int kt = 0; kt < nk; ++kt) {
      // this stage has landed for every wave (of the stages after it up to
      // NST - 2 may be in flight), and every wave has read the one whose
      // place the next stage takes
      if (NST > 2 && kt + NST - 2 < nk) wait_vmcnt<(NST - 2) * 2 * Q>();
      else wait_vmcnt<0>();
      stage_barrier();
      if (kt + NST - 1 < nk) stage(kt + NST - 1);
      const char* s = S + (kt % NST) * 2 * OP;
      if constexpr (decltype(whole)::value) {
#pragma unroll
        for (int ks = 0; ks < BK / 4; ++ks) {
          T af[TQ], bf[TQ];
#pragma unroll
          for (int i = 0; i < TQ; ++i) af[i] = operand(s, !TA, wm, i, ks);
#pragma unroll
          for (int j = 0; j < TQ; ++j) bf[j] = operand(s + OP, TB, wn, j, ks);
#pragma unroll
          for (int i = 0; i < TQ; ++i)
#pragma unroll
            for (int j = 0; j < TQ; ++j) acc[i][j] = mfma16(bf[j], af[i], acc[i][j]);
        }
      } else if (ni > 0 && nj > 0) {
#pragma unroll 1
        for (int ks = 0; ks < BK / 4; ++ks) {
          T af[TQ];
#pragma unroll
          for (int i = 0; i < TQ; ++i) af[i] = operand(s, !TA, wm, i, ks);
#pragma unroll
          for (int j = 0; j < TQ; ++j) {
            if (j >= nj) break;
            const T bf = operand(s + OP, TB, wn, j, ks);
#pragma unroll
            for (int i = 0; i < TQ; ++i)
              if (i < ni) acc[i][j] = mfma16(bf, af[i], acc[i][j]);
          }
        }
      }
    }
  };
  if (ni == TQ && nj == TQ) loop(std::true_type{});
  else loop(std::false_type{});
  store_tile<T, TQ, TQ>(p, C, m0 + wm * (BM / 2), n0 + wn * (BM / 2), lane, acc);
}

template <typename T, int BM, int NST, bool TA, bool TB>
__global__ __launch_bounds__(256, 2) void gemm_dma_kernel(GemmParams<T> p)
{
  __shared__ __attribute__((aligned(1024))) char S[NST * 2 * BM * 128];
  int m0, n0;
  if (tile_origin<BM, BM>(p, m0, n0)) dma_tile_body<T, BM, NST, TA, TB>(p, S, m0, n0);
}

// 128 x 128 tiles for the first p.whole places of the raster (whole rounds
// over the chip), then the rest as quarters of 64 x 64 with a ring of four
// stages in the same LDS: the last round takes about its share of the work
// instead of a tile's whole time.
template <typename T, bool TA, bool TB>
__global__ __launch_bounds__(256, 2) void gemm_dma_mixed_kernel(GemmParams<T> p)
{
  __shared__ __attribute__((aligned(1024))) char S[2 * 2 * 128 * 128];
  const int pid = blockIdx.x;
  int tm, tn;
  if (pid < p.whole) {
    tile_raster(p, xcd_range(pid, p.whole), tm, tn);
    if (tile_holds<128, 128>(p, tm * 128, tn * 128)) dma_tile_body<T, 128, 2, TA, TB>(p, S, tm * 128, tn * 128);
  } else {
    const int at = xcd_range(pid - p.whole, gridDim.x - p.whole);
    tile_raster(p, p.whole + (at >> 2), tm, tn);
    const int m0 = tm * 128 + (at & 1) * 64, n0 = tn * 128 + (at & 2) * 32;
    if (tile_holds<64, 64>(p, m0, n0)) dma_tile_body<T, 64, 4, TA, TB>(p, S, m0, n0);
  }
}

static int g_force_tile = 0;
void gemm_set_tile(int bm) { g_force_tile = bm; }

// Products launched on this stream run their waves at raised issue priority
// (the latency-bound diagonal chain of POTRF, beside full-chip updates).
static hipStream_t g_prio_stream = nullptr;
void gemm_set_priority_stream(hipStream_t s) { g_prio_stream = s; }
int gemm_is_priority_stream(hipStream_t s) { return s != nullptr && s == g_prio_stream; }
int gemm_get_tile() { return g_force_tile; }

template <typename T, int BM, int BK>
static void launch_shape(hipStream_t s, bool ta, bool tb, GemmParams<T>& p, int batch)
{
  p.tiles_m = (p.m + BM - 1) / BM;
  p.tiles_n = (p.n + BM - 1) / BM;
  long ntiles = (p.tri == TRI_FULL || p.trap) ? (long)p.tiles_m * p.tiles_n
                                              : (long)p.tiles_m * (p.tiles_m + 1) / 2;
  XK_CHECK(ntiles < (1L << 31), "gemm grid too large");
  dim3 grid((unsigned)ntiles, 1, (unsigned)batch), block(256);
  if (!ta && !tb) hipLaunchKernelGGL((gemm_kernel<T, BM, BM, BK, false, false>), grid, block, 0, s, p);
  else if (!ta && tb) hipLaunchKernelGGL((gemm_kernel<T, BM, BM, BK, false, true>), grid, block, 0, s, p);
  else if (ta && !tb) hipLaunchKernelGGL((gemm_kernel<T, BM, BM, BK, true, false>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((gemm_kernel<T, BM, BM, BK, true, true>), grid, block, 0, s, p);
  XK_HIP(hipGetLastError());
}

template <typename T, int BM, int NST>
static void launch_dma(hipStream_t s, bool ta, bool tb, GemmParams<T>& p, int batch)
{
  p.tiles_m = (p.m + BM - 1) / BM;
  p.tiles_n = (p.n + BM - 1) / BM;
  const long ntiles = (p.tri == TRI_FULL || p.trap) ? (long)p.tiles_m * p.tiles_n
                                                    : (long)p.tiles_m * (p.tiles_m + 1) / 2;
  XK_CHECK(ntiles < (1L << 31), "gemm grid too large");
  dim3 grid((unsigned)ntiles, 1, (unsigned)batch), block(256);
  if (!ta && !tb) hipLaunchKernelGGL((gemm_dma_kernel<T, BM, NST, false, false>), grid, block, 0, s, p);
  else if (!ta && tb) hipLaunchKernelGGL((gemm_dma_kernel<T, BM, NST, false, true>), grid, block, 0, s, p);
  else if (ta && !tb) hipLaunchKernelGGL((gemm_dma_kernel<T, BM, NST, true, false>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((gemm_dma_kernel<T, BM, NST, true, true>), grid, block, 0, s, p);
  XK_HIP(hipGetLastError());
}

template <typename T>
static void launch_mixed(hipStream_t s, bool ta, bool tb, GemmParams<T>& p, int whole, long tiles)
{
  p.tiles_m = (p.m + 127) / 128;
  p.tiles_n = (p.n + 127) / 128;
  p.whole = whole;
  XK_CHECK(4 * tiles < (1L << 31), "gemm grid too large");
  dim3 grid((unsigned)(whole + 4 * (tiles - whole))), block(256);
  if (!ta && !tb) hipLaunchKernelGGL((gemm_dma_mixed_kernel<T, false, false>), grid, block, 0, s, p);
  else if (!ta && tb) hipLaunchKernelGGL((gemm_dma_mixed_kernel<T, false, true>), grid, block, 0, s, p);
  else if (ta && !tb) hipLaunchKernelGGL((gemm_dma_mixed_kernel<T, true, false>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((gemm_dma_mixed_kernel<T, true, true>), grid, block, 0, s, p);
  XK_HIP(hipGetLastError());
}

// Tile of gemm_dma_kernel for t128 / t64 tiles of 128 / 64 of inner dimension
// k; mixed: the last round of 128 x 128 tiles goes in quarters.  Rates with the
// chip full: FP64 70-71 TFLOP/s with 128 x 128 tiles (two workgroups per CU),
// 66 with 64 x 64 (five per CU); FP32 136 and 120.  A last round that fills a
// part f of its places takes about 0.6 + 0.95 f of a round with 128 (up to
// 1.12; a workgroup alone on its CU runs faster, but two of the last ones may
// share one) and 0.1 + 1.2 f in quarters, an only round 0.62 up to half of the
// places; with 64 0.5 + 0.5 f.  Filling the ring and storing cost as much as
// 150 and 57 of k.  Measured, 128 / 64: FP64 4096^3 62.4 / 59.3, 2048^3 53.9 /
// 55.5, 1536^3 31.8 / 42.0, 2500^2 x 512 43.1 / 46.5, 12000 x 1000 x 3000 47.7 /
// 59.0; mixed / 128 / 64: FP64 triangle 8192^2 x 16384 67.4 / 60.8 / 64, FP32
// 131.6 / 120.5 / 114, 4096 x 4100 x 8192 126 / 107 / 110, 3000^3 119 / 91 / 107.
// 32 x 32 when 64 x 64 leaves CUs with one workgroup or none: FP64 512^3 17.3
// against 9.2, 1024^3 39.3 / 38, 1536^3 42.5 / 42; FP32 512^3 23.3 / 14.2, 1024^3
// 64.4 / 64.9.  (With registers between memory and LDS, tiles as now: 8192^3
// 58.5, 4096^3 51.6, 1024^3 31.4, 512^3 12.8; FP32 133, 111, 47.7, 11.0.)
template <typename T>
static double round_us(int tile, int k)
{
  return tile == 128 ? 512 * 128 * 128 * (k + 150.0) / (sizeof(T) == 8 ? 35.25e6 : 68e6)
                     : 1280 * 64 * 64 * (k + 57.0) / (sizeof(T) == 8 ? 33e6 : 60e6);
}

template <typename T>
static int dma_tile(long t128, long t64, int k, bool may_mix, bool& mixed, double* us = nullptr)
{
  mixed = false;
  if (t64 < (sizeof(T) == 8 ? 512 : 256)) return 32;
  const double r128 = t128 / 512.0, r64 = t64 / 1280.0;
  const double w128 = std::floor(r128), w64 = std::floor(r64);
  const double f128 = r128 - w128, f64 = r64 - w64;
  double last = 0;
  if (w128 == 0) last = f128 <= 0.5 ? 0.62 : 1.06;
  else if (f128 > 0) {
    const double plain = std::min(1.12, 0.6 + 0.95 * f128), quarters = 0.1 + 1.2 * f128;
    mixed = may_mix && quarters < plain;
    last = mixed ? quarters : plain;
  }
  const double c128 = (w128 + last) * round_us<T>(128, k);
  const double c64 = (w64 + (f64 == 0 ? 0 : 0.5 + 0.5 * f64)) * round_us<T>(64, k);
  if (us) *us = std::min(c128, c64);
  return c128 < c64 ? 128 : 64;
}

template <typename T>
double gemm_tiles_us(int tile, long tiles, int k)
{
  const double r = tiles / (tile == 128 ? 512.0 : 1280.0), w = std::floor(r), f = r - w;
  double last = f == 0 ? 0 : 0.5 + 0.5 * f;
  if (tile == 128 && f > 0)
    last = w == 0 ? std::min(1.0, 0.62 + 0.95 * std::max(0.0, f - 0.5))
                  : std::min({1.12, 0.6 + 0.95 * f, 0.1 + 1.2 * f});
  return (w + last) * round_us<T>(tile, k);
}
template double gemm_tiles_us<double>(int, long, int);
template double gemm_tiles_us<float>(int, long, int);

// Whether the register-staged kernel is the faster one for aligned operands (us,
// it / direct to LDS).
// FP64: an inner dimension of less than two stages (4096^2 x 24 50.2 / 54.1, 1024^2
// x 8 8.9 / 9.6), or of a few where 32 x 32 tiles are more than one fill of the
// chip (160 x 7680 x 48 11.6 / 12.4, x 96 14.3 / 14.7).
// FP32: a remainder of a first or second stage where 64 x 64 tiles fit the chip at
// once (4096 x 512 x 48 12.5 / 14.4, 1024^2 x 16 9.7 / 11.5; 2048^2 x 16 23 / 16); and middling inner dimensions over
// many rounds, where two workgroups on a CU hide less of each other's loads than
// four, with both operands stored along their rows (12000^2 x 768 1909 / 2040) or
// with C's columns a multiple of 4 KB apart, which meet in the same memory channels
// (8192^2 x 768 881 / 985 and 914 with B along the inner dimension, 10240^2 1352 /
// 1387; 7936^2 866 / 842, 8192^2 x 512 641 / 619, x 1300 1417 / 1413).
template <typename T>
static bool registers_better(long t128, long t64, long t32, int k, bool ta, bool tb, long ldc)
{
  if (sizeof(T) == 8) return k < 32 || (k < 128 && t64 < 512 && t32 > 1024);
  const bool rows = !ta && tb, strided = ldc * 4 % 4096 == 0;
  if (k < 64) return k % 32 != 0 && t64 >= 256 && t128 < 160;
  return t128 >= 3072 && (rows || strided) && k >= 576 && k < (rows && strided ? 1536 : 1152);
}

template <typename T>
int gemm_tile_of(bool ta, bool tb, int m, int n, int k, long ldc, double* us)
{
  auto tiles = [&](int t) { return (long)((m + t - 1) / t) * ((n + t - 1) / t); };
  bool mixed;
  if (registers_better<T>(tiles(128), tiles(64), tiles(32), k, ta, tb, ldc)) return 0;
  return dma_tile<T>(tiles(128), tiles(64), k, true, mixed, us);
}
template int gemm_tile_of<double>(bool, bool, int, int, int, long, double*);
template int gemm_tile_of<float>(bool, bool, int, int, int, long, double*);

template <typename T>
void gemm(hipStream_t s, int transA, int transB, int m, int n, int k, T alpha, const T* A, long lda,
          const T* B, long ldb, T beta, T* C, long ldc, int tri, int batch, long sA, long sB, long sC, int kmode,
          int kpart, int tile)
{
  if (m <= 0 || n <= 0 || batch <= 0) return;
  if (tri != TRI_FULL)
    XK_CHECK(tri == TRI_LOWER ? m >= n : n >= m, "triangular gemm output must hold its whole diagonal");
  GemmParams<T> p;
  p.m = m; p.n = n; p.k = k; p.tri = tri; p.kmode = kmode; p.kpart = kpart;
  p.trap = tri != TRI_FULL && m != n;
  p.alpha = alpha; p.beta = beta;
  p.A = A; p.lda = lda; p.sA = sA;
  p.B = B; p.ldb = ldb; p.sB = sB;
  p.C = C; p.ldc = ldc; p.sC = sC;
  auto aligned = [](const void* q, long ld, long stride) {
    return ((uintptr_t)q % 16 == 0) && ((ld * (long)sizeof(T)) % 16 == 0) && ((stride * (long)sizeof(T)) % 16 == 0);
  };
  p.prio = gemm_is_priority_stream(s);
  p.vecA = aligned(A, lda, sA);
  p.vecB = aligned(B, ldb, sB);
  const bool ta = transA != NoTrans, tb = transB != NoTrans;
  auto tiles = [&](int t) {
    const long a = (m + t - 1) / t, b = (n + t - 1) / t;
    return (p.tri != TRI_FULL && !p.trap ? a * (a + 1) / 2 : a * b) * batch;
  };
  int bm = g_force_tile;
  // 32-bit offsets inside a tile
  const bool dma = p.vecA && p.vecB && lda < (1L << 21) && ldb < (1L << 21) &&
                   (bm || tile || !registers_better<T>(tiles(128), tiles(64), tiles(32), kpart ? kpart : k, ta, tb, ldc));
  if (dma) {
    bool mixed = false;
    if (bm == 0) {
      bm = dma_tile<T>(tiles(128), tiles(64), kpart ? kpart : k, batch == 1 && kmode == KRANGE_ALL, mixed);
      // tiles of unequal inner ranges fill the chip better when they are many:
      // 128 / 64, FP64 DTRMM 4000 x 1900 from the left 801 / 652 us, from the
      // right 1047 / 666, 8192 x 2000 2424 / 2338 and 2363 / 2455; FP32 4096^2 755
      // / 692 (in registers 756, 806, 2749, 2835 and 709)
      if (kmode != KRANGE_ALL && bm == 128) bm = 64;
      if (tile) bm = tile;
    }
    if (bm == 128 && mixed) {
      launch_mixed<T>(s, ta, tb, p, (int)(tiles(128) / 512 * 512), tiles(128));
      return;
    }
    if (bm == 128) launch_dma<T, 128, 2>(s, ta, tb, p, batch);
    else if (bm == 32) launch_dma<T, 32, 4>(s, ta, tb, p, batch);
    else launch_dma<T, 64, 2>(s, ta, tb, p, batch);
    return;
  }
  // also operands at odd offsets (row panels of an odd tile size): the tiles of
  // the register-staged kernel by the same reasons, FP64 55.8 against 47.1
  // TFLOP/s with 64 and 128 (more resident waves per CU), FP32 128 once they
  // fill the chip
  if (bm == 0) {
    bm = sizeof(T) == 8 || tiles(128) < 160 ? 64 : 128;
    if (sizeof(T) == 8 && tiles(64) < 512) bm = 32;
  }
  if constexpr (sizeof(T) == 8) {
    if (bm == 32) launch_shape<T, 32, 16>(s, ta, tb, p, batch);
    else launch_shape<T, 64, 16>(s, ta, tb, p, batch);
  } else {
    if (bm == 128) launch_shape<T, 128, 16>(s, ta, tb, p, batch);
    else launch_shape<T, 64, 16>(s, ta, tb, p, batch);
  }
}

template void gemm<double>(hipStream_t, int, int, int, int, int, double, const double*, long, const double*, long,
                           double, double*, long, int, int, long, long, long, int, int, int);
template void gemm<float>(hipStream_t, int, int, int, int, int, float, const float*, long, const float*, long,
                          float, float*, long, int, int, long, long, long, int, int, int);

}  // namespace xk
