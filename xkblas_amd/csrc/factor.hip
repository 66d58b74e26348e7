// factor.hip — latency-bound diagonal-block kernels for gfx950:
// Cholesky + inverse of blocks of order <= 128, triangular inverse, and small
// helpers (2-D copy, sums of partial products, int fill).
//
// The rows/columns of a leaf's last 16 x 16 tile beyond n are the identity.
// The Cholesky leaf writes the factor and its inverse in one launch.
#include "common.h"
#include "kernels.h"
#include <climits>
#include <utility>

namespace xk {

// sq = sqrt(p) and rs = 1 / sq for a finite pivot p > 0, without a division
// and without a branch: p = 2^(2h) p' with p' in [0.5, 2) (exact scaling by
// the exponent, denormal p included), Goldschmidt's iteration on p' from the
// hardware reciprocal square root, two Newton corrections of the root
// (correctly rounded) and one of the reciprocal (about 1 ulp), then
// sq = 2^h sqrt(p'), rs = 2^-h / sqrt(p').  For p <= 0, infinite or NaN the
// results are unspecified (the caller reports such a pivot from p itself).
__device__ __forceinline__ void sqrt_rcp(double p, double& sq, double& rs)
{
  const int h = __builtin_amdgcn_frexp_exp(p) >> 1;
  const double ps = __builtin_ldexp(p, -2 * h);
  const double r = __builtin_amdgcn_rsq(ps);
  double g = ps * r, hh = 0.5 * r;
  const double e = fma(-hh, g, 0.5);
  g = fma(g, e, g);
  hh = fma(hh, e, hh);
  g = fma(fma(-g, g, ps), hh, g);
  g = fma(fma(-g, g, ps), hh, g);
  double q = 2.0 * hh;
  q = fma(q, fma(-g, q, 1.0), q);
  sq = __builtin_ldexp(g, h);
  rs = __builtin_ldexp(q, -h);
}
__device__ __forceinline__ void sqrt_rcp(float p, float& sq, float& rs)
{
  sq = sqrtf(p);
  rs = 1.0f / sq;
}

// Workgroup barrier that orders LDS accesses only: global stores in flight
// are not waited for (nothing in the kernel reads them back).
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ---------------------------------------------------------------- tiles
// The leaves keep a block of order 16 NT in LDS as 16 x 16 tiles (lower
// triangle only, tile (i, k) at slot i (i + 1) / 2 + k), each 256 elements
// ordered so that element 64 r + l is what lane l holds in register r of an
// MFMA accumulator: row l % 16, column tile_col(l / 16, r).  The operands of
// X Y^T (v_mfma_*_16x16x4, Y issued first) take the same registers, the inner
// index running over the columns in the accumulator's order, so a product's
// result is the next one's operand without moving, and every tile access is
// 64 consecutive elements.
constexpr int LEAF = 128;
constexpr int TS = 256;  // elements of a tile

typedef double leaf_d4 __attribute__((ext_vector_type(4)));
typedef float leaf_f4 __attribute__((ext_vector_type(4)));
template <typename T> struct LeafV;
template <> struct LeafV<double> { typedef leaf_d4 type; };
template <> struct LeafV<float> { typedef leaf_f4 type; };

__device__ __forceinline__ leaf_d4 leaf_mfma(double a, double b, leaf_d4 c)
{
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ leaf_f4 leaf_mfma(float a, float b, leaf_f4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int tile_slot(int i, int k) { return ((i * (i + 1) >> 1) + k) * TS; }
template <typename T>
__device__ __forceinline__ int tile_col(int g, int r)
{
  return sizeof(T) == 8 ? g + 4 * r : 4 * g + r;
}
// position of column c (times 16) inside a tile
template <typename T>
__device__ __forceinline__ constexpr int col_pos(int c)
{
  return sizeof(T) == 8 ? c : (c >> 2) + 4 * (c & 3);
}

template <typename T>
__device__ __forceinline__ typename LeafV<T>::type tile_load(const T* t, int lane)
{
  return typename LeafV<T>::type{t[lane], t[lane + 64], t[lane + 128], t[lane + 192]};
}
template <typename T, typename V>
__device__ __forceinline__ void tile_store(T* t, int lane, const V& v)
{
#pragma unroll
  for (int r = 0; r < 4; ++r) t[lane + 64 * r] = v[r];
}
// the transpose of the tile at t as an operand
template <typename T>
__device__ __forceinline__ typename LeafV<T>::type tile_load_t(const T* t, int lane)
{
  typename LeafV<T>::type v;
  const int row = lane & 15, g = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = t[tile_col<T>(g, r) + 16 * col_pos<T>(row)];
  return v;
}
// acc + X Y^T
template <typename V>
__device__ __forceinline__ V tile_xyt(V acc, const V& x, const V& y)
{
#pragma unroll
  for (int s = 0; s < 4; ++s) acc = leaf_mfma(y[s], x[s], acc);
  return acc;
}

// value of lane J of this lane's row of 16 lanes
template <int J>
__device__ __forceinline__ double row_bcast(double x)
{
  const long y = __builtin_amdgcn_update_dpp(0L, __builtin_bit_cast(long, x), 0x150 + J, 0xf, 0xf, true);
  return __builtin_bit_cast(double, y);
}
template <int J>
__device__ __forceinline__ float row_bcast(float x)
{
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + J, 0xf, 0xf, true));
}

template <typename F, int... J>
__device__ __forceinline__ void for_each_index(F&& f, std::integer_sequence<int, J...>)
{
  (f(std::integral_constant<int, J>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void for_each(F&& f)
{
  for_each_index(f, std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ double frexp_mant(double p) { return __builtin_amdgcn_frexp_mant(p); }
__device__ __forceinline__ float frexp_mant(float p) { return __builtin_amdgcn_frexp_mantf(p); }
__device__ __forceinline__ int frexp_exp(double p) { return __builtin_amdgcn_frexp_exp(p); }
__device__ __forceinline__ int frexp_exp(float p) { return __builtin_amdgcn_frexp_expf(p); }
__device__ __forceinline__ double rcp_approx(double p) { return __builtin_amdgcn_rcp(p); }
__device__ __forceinline__ float rcp_approx(float p) { return __builtin_amdgcn_rcpf(p); }
__device__ __forceinline__ double scale2(double x, int h) { return __builtin_ldexp(x, h); }
__device__ __forceinline__ float scale2(float x, int h) { return __builtin_ldexpf(x, h); }

// d += (d of lane J of this lane's row of 16) * m, one instruction.  The
// hardware wants two wait states between a vector write and such a read of
// the same register and the compiler does not look into the statement: the
// callers keep other instructions between (volatile statements stay in order).
template <int J>
__device__ __forceinline__ void fmac_bcast(double& d, double m)
{
  asm volatile("v_fmac_f64_dpp %0, %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "+v"(d) : "v"(m), "n"(J));
}
template <int J>
__device__ __forceinline__ void fmac_bcast(float& d, float m)
{
  asm volatile("v_fmac_f32_dpp %0, %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "+v"(d) : "v"(m), "n"(J));
}

// x is computed here, between the statements before and after
template <typename T>
__device__ __forceinline__ void pin(T& x)
{
  asm volatile("" : "+v"(x));
}

// Cholesky factor and inverse of one 16 x 16 tile by one wave.  In: d[c] =
// A(i, c), the whole symmetric row i = lane % 16 (the four rows of 16 lanes
// hold the same data).  Out, below the diagonal: l[c] = L(i, c) sqrt(p_c) and
// d[c] = inv(L)(i, c) sqrt(p_i), p the pivots.  Returns this lane's pivot.
// Elimination without roots: W A = U with W unit lower triangular, the
// columns of W taking the place of the eliminated columns, so that each of
// the 16 steps is one reciprocal and 15 row updates from row j; the pivots'
// roots are left to the caller, who takes them once, for all 16 pivots at a
// time: L(i, j) = A_j(i, j) / sqrt(p_j), inv(L) = diag(1 / sqrt(p)) W.
// A step's chain is pivot (broadcast) -> mantissa -> reciprocal -> two
// corrections -> multiplier -> next pivot: 8 dependent instructions.  The
// updates of the step before stand between them, in this order (one wave,
// in-order issue; ordered by the compiler, a leaf of 128 took 39.6 us instead
// of 33.4 of then).
template <typename T>
__device__ __forceinline__ T factor16(T (&d)[16], T (&l)[16], int i)
{
  T m = T(0), piv = T(1);
  for_each<17>([&](auto jc) {
    constexpr int j = decltype(jc)::value;  // this step's pivot; the updates are those of pivot j - 1
    // updates UA .. UB - 1 of pivot j - 1, columns in order from j
    auto update = [&](auto from, auto to) {
      if constexpr (j > 0) {
        for_each<decltype(to)::value - decltype(from)::value>([&](auto q) {
          constexpr int c = (j + decltype(from)::value + decltype(q)::value) % 16;
          fmac_bcast<j - 1>(d[c], m);
        });
      }
    };
#define XK_UPD(a, b) update(std::integral_constant<int, a>{}, std::integral_constant<int, b>{})
    if constexpr (j == 16) {
      XK_UPD(0, 15);
      d[15] = m;
    } else {
      XK_UPD(0, 3);
      T p = row_bcast<j>(d[j]);
      pin(p);
      XK_UPD(3, 4);
      // -A(i, j) / p for the rows below, p = 2^h p' with p' in [0.5, 1) (no
      // overflow for a denormal p): r = 1 / p' to its hardware accuracy
      // (1 - e), the quotient corrected by 1 + e + e^2
      T ps = frexp_mant(p);
      pin(ps);
      int row = i;  // compared anew in each step: 32 lane masks do not fit the scalar registers
      pin(row);
      int h = -frexp_exp(p);
      T a = row > j ? -d[j] : T(0);
      pin(a);
      XK_UPD(4, 5);
      T r = rcp_approx(ps);
      pin(r);
      T q = scale2(a, h);
      pin(q);
      piv = row == j ? p : piv;
      XK_UPD(5, 8);
      T e = fma(-ps, r, T(1));
      pin(e);
      q *= r;
      pin(q);
      XK_UPD(8, 11);
      e = fma(e, e, e);
      pin(e);
      XK_UPD(11, 15);
      l[j] = d[j];
      if constexpr (j > 0) d[j - 1] = m;
      m = fma(q, e, q);
    }
#undef XK_UPD
  });
  return piv;
}

// Row i = lane % 16 of a lower triangular tile in l[]; y[c] = inv(L)(i, c).
// Rows up to j keep their value in step j (a product by zero would not: row j
// of a singular tile is infinite, and zero times that would reach the rows
// above, whose solutions are finite).
template <typename T>
__device__ __forceinline__ void invert16(const T (&l)[16], T (&y)[16], int i, T rdiag)
{
#pragma unroll
  for (int c = 0; c < 16; ++c) y[c] = i == c ? T(1) : T(0);
  for_each<16>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    // row j is final once scaled; rows below subtract L(i, j) times it
    const T m = i > j ? l[j] : T(0);
    for_each<j + 1>([&](auto cc) {
      constexpr int c = decltype(cc)::value;
      y[c] = i == j ? y[c] * rdiag : y[c];
      const T below = fma(-m, row_bcast<j>(y[c]), y[c]);
      y[c] = i > j ? below : y[c];
    });
  });
}

// The registers of tile operand (row i, columns tile_col(g, .)) out of a full row.
template <typename T>
__device__ __forceinline__ typename LeafV<T>::type row_to_tile(const T (&d)[16], int g)
{
  typename LeafV<T>::type v;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const T a = d[tile_col<T>(0, r)], b = d[tile_col<T>(1, r)], c = d[tile_col<T>(2, r)], e = d[tile_col<T>(3, r)];
    const T lo = g & 1 ? b : a, hi = g & 1 ? e : c;
    v[r] = g & 2 ? hi : lo;
  }
  return v;
}

// The lower triangle (as tiles) of a block of order n <= 16 NT: diagonal
// tiles whole when sym (mirrored), else zero above the diagonal; rows and
// columns beyond n are the identity.
template <typename T, int NT>
__device__ __forceinline__ void leaf_load(T* S, int uplo, int n, int nt, const T* A, long lda, bool sym, bool unit)
{
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ti = lane & 15, g = lane >> 4;
  // tiles of tile row / column `wave` so that all loads of a wave are in
  // flight together: tile (a, b) with a - b = q for q = 0 .. NT - 1, a = wave
  typename LeafV<T>::type v[NT];
#pragma unroll
  for (int b = 0; b < NT; ++b) {
    v[b] = typename LeafV<T>::type{0, 0, 0, 0};
    if (b > wave || wave >= nt) continue;
    const int row = wave * 16 + ti;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int col = b * 16 + tile_col<T>(g, r);
      T x = row == col ? T(1) : T(0);
      if (row < n && col < n) {
        const int hi = max(row, col), lo = min(row, col);
        if ((sym || col <= row) && !(unit && row == col)) x = uplo == Lower ? A[hi + (long)lo * lda] : A[lo + (long)hi * lda];
      }
      v[b][r] = x;
    }
  }
#pragma unroll
  for (int b = 0; b < NT; ++b)
    if (b <= wave && wave < nt) tile_store(S + tile_slot(wave, b), lane, v[b]);
}

// Cholesky factor and its inverse for one block of order <= 16 NT (NT = 4
// or 8), one workgroup of NT waves, all products on MFMA tiles.
// The chain of step k is wave 0's alone: factor and invert diagonal tile k in
// registers (factor16), form panel tile (k + 1, k) = A inv(L_kk)^T and update
// diagonal tile k + 1 with it, which is then ready for step k + 1.  Behind it
// the other waves form the rest of the panel and row k of the inverse,
// inv(L)(k, j) = inv(L_kk) S(k, j), update the remaining trailing tiles and the
// sums S(i, j) = -sum_t L(i, t) inv(L)(t, j) of the rows below, and write the
// results to memory.  S and the inverse are kept transposed, in the places of
// L, whose column k nothing reads after step k.
// An update's products are summed before they meet the tile: the diagonal is far
// larger than each, and 16 roundings a step at its size instead of one made the
// factor's error 1.8 times as large (order 128, G G^T + n I: |A - L L^T| 3.1e-16 of
// |A|, now 1.8e-16).  It costs half a microsecond; the sums of all steps kept apart
// from the tile (1.6e-16) cost 1.4 and three spilled registers.
// The waves meet in counters in LDS instead of barriers, so that wave 0 waits
// only for what its next step reads: diagonal tiles done (by wave 0), panel
// tiles and rows of the inverse done (all waves), updates of the two tiles that
// wave 0 takes next, waves done with the step (all but wave 0; their loads of A
// are step 0 of this count).  A count stands for a step only while no wave can
// add the next step's before all have added this one's: a wave that adds to one
// has waited for the step before to be complete in it.  The waves of a
// workgroup are resident together and none leaves before its last count, so
// every wait ends.
// Bound by latency: a step takes 6.7k cycles, 3.0k of them the 16 dependent
// pivots.  Order 128 takes 28 us (FP64); it took 33.4 with two barriers a
// step, the stores to memory on wave 0's way and the sums formed whole when
// their row came up, and two leaves of order 64 with scalar panels and the six
// launches that joined them took 130.
// LDS: 27.4 KB (FP64, NT = 4), 80.7 KB (NT = 8).
template <typename T, int NT>
__global__ __launch_bounds__(64 * NT) __attribute__((amdgpu_waves_per_eu(4)))
void potrf_leaf_kernel(int uplo, int n, T* A, long lda, long sA, T* Tinv, long ldinv, long sInv, int* info, int base,
                       int pair)
{
  typedef typename LeafV<T>::type V;
  constexpr int NW = NT - 1;  // waves beside wave 0
  __shared__ T S[NT * (NT + 1) / 2 * TS];
  __shared__ T LK[3 * TS], RT[3 * 32];  // factor16's l, the pivots' roots and their reciprocals, for the stores of L_kk
  __shared__ int done[4];
  enum { DIAG, PANEL, NEXT, TRAIL };
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ti = lane & 15, g = lane >> 4;
  const int nt = (n + 15) >> 4;
  A += (long)blockIdx.x * sA;
  if (Tinv) Tinv += (long)blockIdx.x * sInv;
  // entry (i, k) of a lower triangle, to the stored triangle
  auto put = [&](T* M, long ld, int i, int k, T v) {
    if (i < n && k < n) {
      if (uplo == Lower) M[i + (long)k * ld] = v;
      else M[k + (long)i * ld] = v;
    }
  };
  // One more of c is done.  The LDS executes a wave's operations in order, so
  // whoever sees the count sees this wave's writes before it: it is enough
  // that the compiler keeps the order, nothing is waited for.
  auto signal = [&](int c) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    if (lane == 0) __hip_atomic_fetch_add(&done[c], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  // until c has reached `count` and c2 `count2`
  auto wait2 = [&](int c, int count, int c2, int count2) {
    for (;;) {
      const int a = __hip_atomic_load(&done[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      const int b = __hip_atomic_load(&done[c2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (__builtin_amdgcn_readfirstlane(a) >= count && __builtin_amdgcn_readfirstlane(b) >= count2) break;
      __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  if (threadIdx.x < 4) done[threadIdx.x] = 0;
  lds_barrier();
  leaf_load<T, NT>(S, uplo, n, nt, A, lda, true, false);  // wave 0: tile (0, 0)
  if (wave == 0) {
    // the latency-bound step of the diagonal chain, which may share its CU
    // with update GEMM waves: its instructions issue first
    __builtin_amdgcn_s_setprio(3);
    int fail = INT_MAX;  // first order with a non-positive pivot
    for (int k = 0; k < nt; ++k) {
      const int c0 = k * 16;
      T* Dk = S + tile_slot(k, k);
      T d[16], l[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) d[c] = Dk[ti + 16 * col_pos<T>(c)];
      const T piv = factor16(d, l, ti);
      const unsigned long long bad = __ballot(!(piv > T(0)) && c0 + ti < n);
      if (bad && fail == INT_MAX) fail = c0 + __ffsll(bad) - 1;
      T sq, rs;
      sqrt_rcp(piv, sq, rs);
      V dk = row_to_tile(d, g);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = tile_col<T>(g, r);
        dk[r] = ti > col ? dk[r] * rs : (ti == col ? rs : T(0));
      }
      tile_store(Dk, lane, dk);
      signal(DIAG);
      const V lk = row_to_tile(l, g);
      // for the stores of L_kk
      auto keep = [&]() {
        tile_store(LK + k % 3 * TS, lane, lk);
        if (g < 2) RT[k % 3 * 32 + lane] = g ? rs : sq;
        signal(PANEL);
      };
      if (k + 1 == nt) {
        // nothing above waits for the other waves in this step: their part of
        // the step before has to be counted before this one's
        wait2(PANEL, k * NT, DIAG, 0);
        keep();
        break;
      }
      // tiles (k + 1, k) and (k + 1, k + 1), there with all updates before k
      T* P = S + tile_slot(k + 1, k);
      T* C = S + tile_slot(k + 1, k + 1);
      wait2(TRAIL, NW, NEXT, 2 * k);
      const V a = tile_load(P, lane), c = tile_load(C, lane);
      const V z = {0, 0, 0, 0};
      const V lp = tile_xyt(z, a, dk);
      tile_store(P, lane, lp);
      keep();
      tile_store(C, lane, c - tile_xyt(z, lp, lp));
    }
    // pair: orders 2i, 2i + 1 stand for order i of a complex block
    if (lane == 0 && fail != INT_MAX) atomicMin(info, pair ? (base + fail) / 2 + 1 : base + fail + 1);
    return;
  }
  signal(TRAIL);           // its tile row is loaded
  // Trailing tiles are counted from the last, column after column, rows
  // falling: those of step k are the first of one list for all steps, dealt to
  // waves 1 .. in turn.  A wave keeps its tiles in registers until the step
  // that takes them, tile (i, q) up to step lim - 1.
  constexpr int MT = (NT * (NT - 1) / 2 - 1 + NW - 1) / NW;
  V c[MT];
  int ci[MT], cq[MT], lim[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    int e = 0, r = wave - 1 + NW * m;
    while (r > e) r -= ++e;
    ci[m] = nt - 1 - r;
    cq[m] = nt - 1 - e;
    lim[m] = ci[m] == cq[m] ? cq[m] - 1 : cq[m];
  }
  const V zero = {0, 0, 0, 0};
  V s = zero;
  for (int k = 0; k < nt; ++k) {
    const int c0 = k * 16, h = nt - 1 - k;
    const int pi = k + 1 + wave;  // this wave's tile row of the panel (wave 0: k + 1)
    V lp = zero, z = zero;
    wait2(DIAG, k + 1, TRAIL, (k + 1) * NW);
    const V dk = tile_load(S + tile_slot(k, k), lane);
    // S(k - 1 + wave, k - 1), now that column k - 1 of L has been read
    if (Tinv && wave > 1 && k > 0 && k - 1 + wave < nt) tile_store(S + tile_slot(k - 1 + wave, k - 1), lane, s);
    if (pi < nt) {
      T* P = S + tile_slot(pi, k);
      lp = tile_xyt(zero, tile_load(P, lane), dk);
      tile_store(P, lane, lp);
    }
    // row k of the inverse, one tile a wave: column k - 1 is wave 1's
    const int j = wave == 1 ? k - 1 : wave - 2;
    const bool inv = Tinv && j >= 0 && (wave == 1 || j < k - 1);
    if (inv) {
      if (wave > 1) s = tile_load(S + tile_slot(k, j), lane);
      z = tile_xyt(zero, s, dk);
      tile_store(S + tile_slot(k, j), lane, z);
    }
    signal(PANEL);
    if (k == 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (lim[m] > 0) c[m] = tile_load(S + tile_slot(ci[m], cq[m]), lane);
    }
    wait2(PANEL, (k + 1) * NT, DIAG, 0);
    // trailing updates, those that wave 0 waits for first
#pragma unroll
    for (int m = MT - 1; m >= 0; --m)
      if (lim[m] > k) {
        const V x = tile_load(S + tile_slot(ci[m], k), lane), y = tile_load(S + tile_slot(cq[m], k), lane);
        c[m] -= tile_xyt(zero, x, y);
        if (lim[m] == k + 1) tile_store(S + tile_slot(ci[m], cq[m]), lane, c[m]);
        if (ci[m] == k + 2) signal(NEXT);
      }
    if (Tinv) {
      // S(i, j) -= L(i, k) inv(L)(k, j) for j < k < i, the waves with fewer
      // trailing tiles first; v / h by a multiplication
      const int rh = (int)(0x13161a202b408000ull >> (8 * h)) & 255;
      int v = wave - 1 - (h * (h + 1) / 2 - 1) % NW;
      for (v = v < 0 ? v + NW : v; v < k * h; v += NW) {
        const int jj = v * rh >> 7, i = k + 1 + v - jj * h;
        T* C = S + tile_slot(i, jj);
        const V x = tile_load(S + tile_slot(k, jj), lane), y = tile_load(S + tile_slot(i, k), lane);
        tile_store(C, lane, tile_xyt(tile_load(C, lane), x, -y));
      }
      // S(k + wave, k) = -L(k + wave, k) inv(L_kk)
      if (wave <= h)
        s = tile_xyt(zero, tile_load_t(S + tile_slot(k, k), lane), -tile_load(S + tile_slot(k + wave, k), lane));
    }
    // the last wave, without panel tiles, writes the diagonal tile and wave 0's panel tile
    const bool mine = wave == NW;
    V lk, l0;
    if (mine) {
      lk = tile_load(LK + k % 3 * TS, lane);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = tile_col<T>(g, r);
        const T root = RT[k % 3 * 32 + (ti > col ? 16 + col : ti)];
        lk[r] = ti > col ? lk[r] * root : root;
      }
      if (h) l0 = tile_load(S + tile_slot(k + 1, k), lane);
    }
    signal(TRAIL);
    // to memory: tile rows `row` .., columns col0 .., or their mirror image;
    // only the last tile row has orders beyond n
    auto put_tile = [&](T* M, long ld, int row, int col0, bool mirror, const V& t) {
      if (row + ti >= n) return;
      const bool down = (uplo == Lower) != mirror;
      T* q = M + (down ? row + ti + col0 * ld : (row + ti) * ld + col0);
      const long step = down ? ld : 1;
#pragma unroll
      for (int r = 0; r < 4; ++r) q[tile_col<T>(g, r) * step] = t[r];
    };
    if (pi < nt) {
      put_tile(A, lda, pi * 16, c0, false, lp);
      if (Tinv) put_tile(Tinv, ldinv, pi * 16, c0, true, zero);
    }
    if (mine && h) {
      put_tile(A, lda, c0 + 16, c0, false, l0);
      if (Tinv) put_tile(Tinv, ldinv, c0 + 16, c0, true, zero);
    }
    if (inv && h) put_tile(Tinv, ldinv, j * 16, c0, true, z);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int col = tile_col<T>(g, r);
      if (inv && !h) put(Tinv, ldinv, c0 + col, j * 16 + ti, z[r]);
      if (mine) {
        if (col <= ti) put(A, lda, c0 + ti, c0 + col, lk[r]);
        if (Tinv) put(Tinv, ldinv, c0 + ti, c0 + col, dk[r]);
      }
    }
  }
}

// Inverse of one triangular block of order <= 16 NT, one workgroup of NT
// waves: wave j inverts diagonal tile j (invert16), then forms block column j
// of the inverse downwards on MFMA tiles with its own tiles kept in
// registers: one barrier in all.  The longest column is 35 tile products.
template <typename T, int NT>
__global__ __launch_bounds__(64 * NT) void trtri_leaf_kernel(int uplo, int diag, int n, const T* A, long lda, long sA,
                                                             T* Tinv, long ldinv, long sInv)
{
  typedef typename LeafV<T>::type V;
  __shared__ T S[NT * (NT + 1) / 2 * TS];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ti = lane & 15, g = lane >> 4;
  const int nt = (n + 15) >> 4;
  A += (long)blockIdx.x * sA;
  Tinv += (long)blockIdx.x * sInv;
  leaf_load<T, NT>(S, uplo, n, nt, A, lda, false, diag == Unit);
  // inv(L)(i, k) to the stored triangle (inv(U) = inv(L)^T)
  auto put = [&](int i, int k, T v) {
    if (i < n && k < n) {
      if (uplo == Lower) Tinv[i + (long)k * ldinv] = v;
      else Tinv[k + (long)i * ldinv] = v;
    }
  };
  if (wave < nt) {
    T* D = S + tile_slot(wave, wave);  // loaded by this wave
    T l[16], y[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) l[c] = D[ti + 16 * col_pos<T>(c)];
    T own = T(1);
#pragma unroll
    for (int c = 0; c < 16; ++c) own = ti == c ? l[c] : own;
    invert16(l, y, ti, T(1) / own);
    const V d = row_to_tile(y, g);
    tile_store(D, lane, d);
#pragma unroll
    for (int r = 0; r < 4; ++r) put(wave * 16 + ti, wave * 16 + tile_col<T>(g, r), d[r]);
  }
  lds_barrier();
  if (wave >= nt) return;
  V zt[NT];  // zt[u] = inv(L)(wave + u, wave) transposed
  zt[0] = tile_load_t(S + tile_slot(wave, wave), lane);
#pragma unroll
  for (int v = 1; v < NT; ++v) {
    const int k = wave + v;
    if (k >= nt) break;
    V s = {0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < v; ++u) s = tile_xyt(s, zt[u], tile_load(S + tile_slot(k, wave + u), lane));
    const V z0 = {0, 0, 0, 0};
    zt[v] = tile_xyt(z0, s, -tile_load(S + tile_slot(k, k), lane));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = k * 16 + tile_col<T>(g, r), col = wave * 16 + ti;
      put(row, col, zt[v][r]);
      put(col, row, T(0));
    }
  }
}

template <typename T>
void potrf_leaf(hipStream_t s, int uplo, int n, T* A, long lda, long sA, T* Tinv, long ldinv, long sInv,
                int batch, int* info, int base, int pair)
{
  XK_CHECK(n >= 1 && n <= LEAF, "potrf leaf order must be in [1,128]");
  if (batch <= 0) return;
  if (n <= 64)
    hipLaunchKernelGGL((potrf_leaf_kernel<T, 4>), dim3(batch), dim3(256), 0, s, uplo, n, A, lda, sA, Tinv, ldinv,
                       sInv, info, base, pair);
  else
    hipLaunchKernelGGL((potrf_leaf_kernel<T, 8>), dim3(batch), dim3(512), 0, s, uplo, n, A, lda, sA, Tinv, ldinv,
                       sInv, info, base, pair);
  XK_HIP(hipGetLastError());
}

template <typename T>
void trtri_leaf(hipStream_t s, int uplo, int diag, int n, const T* A, long lda, long sA, T* Tinv, long ldinv,
                long sInv, int batch)
{
  XK_CHECK(n >= 1 && n <= LEAF, "trtri leaf order must be in [1,128]");
  if (batch <= 0) return;
  if (n <= 64)
    hipLaunchKernelGGL((trtri_leaf_kernel<T, 4>), dim3(batch), dim3(256), 0, s, uplo, diag, n, A, lda, sA, Tinv,
                       ldinv, sInv);
  else
    hipLaunchKernelGGL((trtri_leaf_kernel<T, 8>), dim3(batch), dim3(512), 0, s, uplo, diag, n, A, lda, sA, Tinv,
                       ldinv, sInv);
  XK_HIP(hipGetLastError());
}

// P <- P inv(L)^T in place (Upper: P^T <- P^T inv(L)^T with inv(L) = inv(U)^T):
// a workgroup of four waves takes 16 rows of P (columns, Upper), holds them in
// LDS as the eight 16 x 16 tiles of their 128 columns, and wave w forms
// column tiles w and 7 - w of the product (9 tile products each: inv(L) is
// triangular) with inv(L) read straight from L2 into the operand registers.
// Every workgroup has read its rows before it writes any, so P needs no copy.
// Bound by latency (one load of each operand, 36 dependent MFMAs): about 4 us
// at any m that fits the chip.
template <typename T>
__global__ __launch_bounds__(256) void trsm_panel_kernel(int uplo, int m, int n, T* __restrict__ P, long lda,
                                                         const T* __restrict__ Linv, long ldinv, int prio)
{
  typedef typename LeafV<T>::type V;
  constexpr int NT = LEAF / 16;
  __shared__ T S[NT * TS];
  if (prio) __builtin_amdgcn_s_setprio(3);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ti = lane & 15, g = lane >> 4;
  const int r0 = blockIdx.x * 16;
  // operand tiles (jn, kt) of inv(L): rows jn, inner index kt
  auto load_y = [&](int jn, V(&y)[NT]) {
    const int row = jn * 16 + ti;
#pragma unroll
    for (int kt = 0; kt < NT; ++kt) {
      if (kt > jn) break;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = kt * 16 + tile_col<T>(g, r);
        T v = T(0);
        if (k <= row && row < n) v = uplo == Lower ? Linv[row + (long)k * ldinv] : Linv[k + (long)row * ldinv];
        y[kt][r] = v;
      }
    }
  };
  V y[NT];
  load_y(wave, y);
  {
    T v[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      const int i = uplo == Lower ? tid & 15 : tid >> 4, k = q * 16 + (uplo == Lower ? tid >> 4 : tid & 15);
      v[q] = T(0);
      if (r0 + i < m && k < n) v[q] = uplo == Lower ? P[r0 + i + (long)k * lda] : P[k + (long)(r0 + i) * lda];
    }
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      const int i = uplo == Lower ? tid & 15 : tid >> 4, k = uplo == Lower ? tid >> 4 : tid & 15;
      S[q * TS + i + 16 * col_pos<T>(k)] = v[q];
    }
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int jn = h == 0 ? wave : NT - 1 - wave;
    if (jn * 16 >= n) continue;
    V acc = {0, 0, 0, 0};
    if (h == 1) load_y(jn, y);
#pragma unroll
    for (int kt = 0; kt < NT; ++kt) {
      if (kt > jn) break;
      const V x = tile_load(S + kt * TS, lane);
      // Upper: the transposed product, so that a lane's neighbours store neighbours
      acc = uplo == Lower ? tile_xyt(acc, x, y[kt]) : tile_xyt(acc, y[kt], x);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = r0 + (uplo == Lower ? ti : tile_col<T>(g, r)), k = jn * 16 + (uplo == Lower ? tile_col<T>(g, r) : ti);
      if (i < m && k < n) {
        if (uplo == Lower) P[i + (long)k * lda] = acc[r];
        else P[k + (long)i * lda] = acc[r];
      }
    }
  }
}

template <typename T>
void trsm_panel(hipStream_t s, int uplo, int m, int n, T* P, long lda, const T* Linv, long ldinv)
{
  XK_CHECK(n >= 1 && n <= LEAF, "panel solve: block order must be in [1,128]");
  if (m <= 0) return;
  hipLaunchKernelGGL((trsm_panel_kernel<T>), dim3((m + 15) / 16), dim3(256), 0, s, uplo, m, n, P, lda, Linv, ldinv,
                     gemm_is_priority_stream(s));
  XK_HIP(hipGetLastError());
}

template <typename T>
__global__ void copy2d_kernel(int m, int n, const T* X, long ldx, T* Y, long ldy)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (i < m && j < n) Y[i + (long)j * ldy] = X[i + (long)j * ldx];
}

template <typename T>
void copy2d(hipStream_t s, int m, int n, const T* X, long ldx, T* Y, long ldy)
{
  if (m <= 0 || n <= 0) return;
  XK_CHECK(n < 65536 * 16, "copy2d: too many columns");
  // one block column per matrix column, chunks of 256 rows
  for (int j0 = 0; j0 < n; j0 += 65535) {
    int nn = n - j0 < 65535 ? n - j0 : 65535;
    hipLaunchKernelGGL((copy2d_kernel<T>), dim3((m + 255) / 256, nn), dim3(256), 0, s, m, nn, X + (long)j0 * ldx,
                       ldx, Y + (long)j0 * ldy, ldy);
  }
  XK_HIP(hipGetLastError());
}

// C <- beta C + sum_p W_p (W_p: m x n, leading dimension m, p-th at p m n);
// beta == 0 never reads C.
template <typename T>
__global__ void splitk_reduce_kernel(int m, int n, int parts, const T* __restrict__ W, T beta, T* __restrict__ C,
                                     long ldc, int tri)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int j = blockIdx.y;
  if (i >= m || j >= n || (tri == TRI_LOWER && i < j) || (tri == TRI_UPPER && i > j)) return;
  const long mn = (long)m * n, e = i + (long)j * m;
  T v = W[e];
  for (int p = 1; p < parts; ++p) v += W[p * mn + e];
  T* c = C + i + (long)j * ldc;
  *c = beta != T(0) ? beta * *c + v : v;
}

template <typename T>
void splitk_reduce(hipStream_t s, int m, int n, int parts, const T* W, T beta, T* C, long ldc, int tri)
{
  if (m <= 0 || n <= 0) return;
  XK_CHECK(n <= 65535, "splitk_reduce: too many columns");
  hipLaunchKernelGGL((splitk_reduce_kernel<T>), dim3((m + 255) / 256, n), dim3(256), 0, s, m, n, parts, W, beta, C,
                     ldc, tri);
  XK_HIP(hipGetLastError());
}

__global__ void fill_int_kernel(int* p, int n, int v)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void fill_int(hipStream_t s, int* p, int n, int v)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(fill_int_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, n, v);
  XK_HIP(hipGetLastError());
}

#define XK_INST(T)                                                                                           \
  template void trsm_panel<T>(hipStream_t, int, int, int, T*, long, const T*, long);                           \
  template void potrf_leaf<T>(hipStream_t, int, int, T*, long, long, T*, long, long, int, int*, int, int);         \
  template void trtri_leaf<T>(hipStream_t, int, int, int, const T*, long, long, T*, long, long, int);         \
  template void copy2d<T>(hipStream_t, int, int, const T*, long, T*, long);                                    \
  template void splitk_reduce<T>(hipStream_t, int, int, int, const T*, T, T*, long, int);
XK_INST(double)
XK_INST(float)
#undef XK_INST

}  // namespace xk
