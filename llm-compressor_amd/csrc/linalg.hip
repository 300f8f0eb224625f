// fp32 linear algebra for the GPTQ solve on gfx950: MFMA GEMM, blocked
// Cholesky and triangular inverse.
//
// The reference (modifiers/gptq/gptq_quantize.py:181-188) damps H, then runs
// cholesky -> cholesky_inverse -> cholesky(upper) to obtain the upper
// Cholesky factor U of H^-1.  With J the exchange matrix, F = J H J = L L^T
// gives H = R R^T for the upper-triangular R = J L J, so H^-1 = R^-T R^-1
// and U = R^-1 = J L^-1 J (the factor is unique for positive diagonals).
// That is one potrf and one trtri (2 d^3 / 3 flops instead of 4 d^3 / 3),
// with identical mathematics and fp32 rounding of the same order.
//
//   prepare:  F[a][b] = (H[p(d-1-a)][p(d-1-b)] / n), dead-column and
//             damping rules on the diagonal (lower triangle of F only)
//   potrf:    per 128-column panel: diagonal block Cholesky + its inverse
//             (one workgroup, LDS resident), panel solve as a GEMM with the
//             block inverse, trailing update as a lower-only MFMA GEMM
//   trtri:    recursive doubling inv([[A,0],[B,C]]) = [[A^-1,0],[-C^-1 B A^-1, C^-1]]
//             on top of the diagonal-block inverses, as batched GEMMs
//   flip:     hinv[a][b] = X[d-1-a][d-1-b] for a <= b, 0 below
#include "linalg.h"

#pragma clang fp contract(off)

namespace mi355q {
namespace {

// ---------------------------------------------------------------- GEMM
// x if keep else +0.0, as a bit mask: a select on a loaded value can be
// turned back into a branch around the load, which serialises the loads
__device__ __forceinline__ float keep_if(float x, bool keep) {
  return __uint_as_float(__float_as_uint(x) & (keep ? 0xffffffffu : 0u));
}

constexpr int GBM = 128, GBN = 128, GBK = 32, GNT = 256;
constexpr int LA = GBK + 1;     // LDS row stride for [m][k] tiles
constexpr int LBN = GBN + 32;   // LDS row stride for [k][n] tiles

// AT: A is stored transposed, [K x M] row-major (lda): A[m][k] = A_mem[k][m]
// (the Hessian X^T X of token-major X); it is staged like a non-transposed B.
template <bool BT, bool AT = false>
__global__ __launch_bounds__(GNT, 2) void gemm_f32_kernel(GemmArgs g) {
  __shared__ float lds_a[2][AT ? GBK * LBN : GBM * LA];
  __shared__ float lds_b[2][BT ? GBN * LA : GBK * LBN];

  const int64_t m0 = (int64_t)blockIdx.y * GBM, n0 = (int64_t)blockIdx.x * GBN;
  if (g.lower_only && m0 + GBM - 1 < n0) return;
  if (g.upper_only && m0 > n0 + GBN - 1) return;
  if (g.only_if && *g.only_if == 0) return;
  const int64_t bz = blockIdx.z;
  const int64_t b1 = g.inner > 0 ? bz % g.inner : bz, b2 = g.inner > 0 ? bz / g.inner : 0;
  const float* A = g.A + b1 * g.strideA + b2 * g.strideA2;
  const float* B = g.B + b1 * g.strideB + b2 * g.strideB2;
  float* C = g.C + b1 * g.strideC + b2 * g.strideC2;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  f32x16_t acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;

  f32x4_t ra[4], rb[4];
  // Branch-free loads: out-of-range elements read a clamped in-range address
  // and are zeroed when the tile is stored to LDS (after the MFMAs of the
  // current stage), so the loads issue back to back and are not waited for
  // before the MFMAs.
  const bool vec_a = ((reinterpret_cast<uintptr_t>(A) & 15) == 0) && ((g.lda & 3) == 0) && ((g.K & 3) == 0);
  const bool vec_bk = ((reinterpret_cast<uintptr_t>(B) & 15) == 0) && ((g.ldb & 3) == 0) && ((g.K & 3) == 0);
  const bool vec_bn = ((reinterpret_cast<uintptr_t>(B) & 15) == 0) && ((g.ldb & 3) == 0) && ((g.N & 3) == 0);
  // A / B^T tiles: 128 rows x 32 k -> 1024 float4 (4 per thread)
  auto load_mk = [&](const float* P, int64_t ld, bool vec, int64_t rows_lim, int64_t r0, int64_t k0,
                     f32x4_t* r) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int idx = v * GNT + tid;
      const int64_t gr = r0 + (idx >> 3), gk = k0 + 4 * (idx & 7);
      const int64_t grc = gr < rows_lim ? gr : rows_lim - 1;
      if (vec) {
        const int64_t gkc = gk < g.K ? gk : g.K - 4;
        r[v] = *reinterpret_cast<const f32x4_t*>(P + grc * ld + gkc);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) r[v][e] = P[grc * ld + (gk + e < g.K ? gk + e : g.K - 1)];
      }
    }
  };
  auto store_mk = [&](float* L, const f32x4_t* r, int64_t rows_lim, int64_t r0, int64_t k0) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int idx = v * GNT + tid;
      const int row = idx >> 3, quad = idx & 7;
      const bool rok = r0 + row < rows_lim;
#pragma unroll
      for (int e = 0; e < 4; ++e) L[row * LA + 4 * quad + e] = keep_if(r[v][e], rok && k0 + 4 * quad + e < g.K);
    }
  };
  // [k][n] tiles (B not transposed, or A transposed): 32 k x 128 columns
  // c0.. of P (ld, `cols` columns) -> 1024 float4
  const bool vec_am = AT && ((reinterpret_cast<uintptr_t>(A) & 15) == 0) && ((g.lda & 3) == 0) && ((g.M & 3) == 0);
  auto load_kn_of = [&](const float* P, int64_t ld, bool vec, int64_t cols, int64_t c0, int64_t k0, f32x4_t* r) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int idx = v * GNT + tid;
      const int64_t gk = k0 + (idx >> 5), gn = c0 + 4 * (idx & 31);
      const int64_t gkc = gk < g.K ? gk : g.K - 1;
      if (vec) {
        const int64_t gnc = gn < cols ? gn : cols - 4;
        r[v] = *reinterpret_cast<const f32x4_t*>(P + gkc * ld + gnc);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) r[v][e] = P[gkc * ld + (gn + e < cols ? gn + e : cols - 1)];
      }
    }
  };
  auto store_kn_of = [&](float* L, const f32x4_t* r, int64_t cols, int64_t c0, int64_t k0) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int idx = v * GNT + tid;
      const int krow = idx >> 5, quad = idx & 31;
      const bool kok = k0 + krow < g.K;
      f32x4_t x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = keep_if(r[v][e], kok && c0 + 4 * quad + e < cols);
      *reinterpret_cast<f32x4_t*>(L + krow * LBN + 4 * quad) = x;
    }
  };
  auto load_kn = [&](int64_t k0, f32x4_t* r) { load_kn_of(B, g.ldb, vec_bn, g.N, n0, k0, r); };
  auto store_kn = [&](float* L, const f32x4_t* r, int64_t k0) { store_kn_of(L, r, g.N, n0, k0); };
  auto load_a = [&](int64_t k0, f32x4_t* r) {
    if (AT) load_kn_of(A, g.lda, vec_am, g.M, m0, k0, r); else load_mk(A, g.lda, vec_a, g.M, m0, k0, r);
  };
  auto store_a = [&](float* L, const f32x4_t* r, int64_t k0) {
    if (AT) store_kn_of(L, r, g.M, m0, k0); else store_mk(L, r, g.M, m0, k0);
  };

  // K range of this tile: all of K, or where a triangular operand can be nonzero
  const int64_t kbeg = g.b_lower ? (n0 / GBK) * GBK : 0;
  const int64_t kend = g.a_lower ? (m0 + GBM < g.K ? m0 + GBM : g.K) : g.K;
  const int64_t nst = kend > kbeg ? (kend - kbeg + GBK - 1) / GBK : 0;
  if (nst > 0) {
    load_a(kbeg, ra);
    if (BT) load_mk(B, g.ldb, vec_bk, g.N, n0, kbeg, rb); else load_kn(kbeg, rb);
    store_a(lds_a[0], ra, kbeg);
    if (BT) store_mk(lds_b[0], rb, g.N, n0, kbeg); else store_kn(lds_b[0], rb, kbeg);
  }
  __syncthreads();
  for (int64_t st = 0; st < nst; ++st) {
    const int buf = st & 1;
    const bool more = st + 1 < nst;
    const int64_t kn = kbeg + (st + 1) * GBK;
    if (more) {
      load_a(kn, ra);
      if (BT) load_mk(B, g.ldb, vec_bk, g.N, n0, kn, rb); else load_kn(kn, rb);
    }
    const float* la = lds_a[buf];
    const float* lb = lds_b[buf];
#pragma unroll
    for (int kk = 0; kk < GBK / 2; ++kk) {
      const int k = 2 * kk + (lane >> 5);
      float fa[2], fb[2];
#pragma unroll
      for (int bm = 0; bm < 2; ++bm) {
        const int m = wm * 64 + bm * 32 + (lane & 31);
        fa[bm] = AT ? la[k * LBN + m] : la[m * LA + k];
      }
#pragma unroll
      for (int bn = 0; bn < 2; ++bn) {
        const int n = wn * 64 + bn * 32 + (lane & 31);
        fb[bn] = BT ? lb[n * LA + k] : lb[k * LBN + n];
      }
#pragma unroll
      for (int bm = 0; bm < 2; ++bm)
#pragma unroll
        for (int bn = 0; bn < 2; ++bn)
          acc[bm][bn] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[bm], fb[bn], acc[bm][bn], 0, 0, 0);
    }
    if (more) {
      store_a(lds_a[buf ^ 1], ra, kn);
      if (BT) store_mk(lds_b[buf ^ 1], rb, g.N, n0, kn); else store_kn(lds_b[buf ^ 1], rb, kn);
    }
    __syncthreads();
  }

  // C is read (clamped, all loads in flight together) before any store
  float cv[64];
  if (g.beta != 0.f) {
#pragma unroll
    for (int bm = 0; bm < 2; ++bm)
#pragma unroll
      for (int bn = 0; bn < 2; ++bn)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t gm = m0 + wm * 64 + bm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          const int64_t gn = n0 + wn * 64 + bn * 32 + (lane & 31);
          cv[(bm * 2 + bn) * 16 + r] = C[(gm < g.M ? gm : g.M - 1) * g.ldc + (gn < g.N ? gn : g.N - 1)];
        }
  }
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t gm = m0 + wm * 64 + bm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const int64_t gn = n0 + wn * 64 + bn * 32 + (lane & 31);
        if (gm < g.M && gn < g.N && (!g.lower_only || gm >= gn) && (!g.upper_only || gm <= gn)) {
          const float prod = g.alpha * acc[bm][bn][r];
          C[gm * g.ldc + gn] = g.beta == 0.f ? prod : g.beta * cv[(bm * 2 + bn) * 16 + r] + prod;
        }
      }
}

// ---------------------------------------------------------------- K <= 128 GEMM
// The solve's panel GEMMs all have K = 128 (one panel of columns): the
// Cholesky panel solve and trailing update, and GPTQ's lazy update.  A
// workgroup keeps its 128-row tile of A (all of K) in LDS and walks the
// column tiles n = blockIdx.x, blockIdx.x + gridDim.x, ...; the next B tile
// and the current C tile are fetched into registers while the MFMAs of the
// current tile run, so every load after the first overlaps compute.
constexpr int KT = 128;          // tile edge and largest K
constexpr int KLA = KT + 1;      // LDS stride of [row][k] tiles (odd: 32 consecutive rows hit 32 banks)

// Whole tiles only: K == 128, M and N multiples of 128, 16-byte aligned rows
// (other shapes take the general kernel).  Every address is a wave-uniform
// tile base plus a 32-bit lane offset, with no clamping, so the loads issue
// back to back from few registers.
template <bool BT>
__global__ __launch_bounds__(GNT, 1) void gemm_k128_kernel(GemmArgs g) {
  __shared__ float la[KT * KLA];
  __shared__ float lb[BT ? KT * KLA : KT * LBN];
  {
    const int64_t bz = blockIdx.z;
    const int64_t b1 = g.inner > 0 ? bz % g.inner : bz, b2 = g.inner > 0 ? bz / g.inner : 0;
    g.A += b1 * g.strideA + b2 * g.strideA2;
    g.B += b1 * g.strideB + b2 * g.strideB2;
    g.C += b1 * g.strideC + b2 * g.strideC2;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t m0 = (int64_t)blockIdx.y * KT;
  const int64_t ntiles = g.N / KT;
  int64_t nt = blockIdx.x;
  if (nt >= ntiles || (g.lower_only && nt * KT > m0)) return;

  // [row][k] tiles: float4 v covers row 8 v + tid / 32, k 4 (tid % 32)
  // lane offsets in bytes (32-bit: uniform base + lane offset addressing)
  const uint32_t off_a = (uint32_t)((tid >> 5) * g.lda + 4 * (tid & 31)) * 4u;
  const uint32_t off_b = (uint32_t)((tid >> 5) * g.ldb + 4 * (tid & 31)) * 4u;
  const uint32_t off_c = (uint32_t)((wm * 64 + 4 * (lane >> 5)) * g.ldc + wn * 64 + (lane & 31)) * 4u;
  auto at = [](const float* base, uint32_t off) {
    return reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + off);
  };
  auto load_rows = [&](const float* base, int64_t ld, uint32_t off, f32x4_t* r) {
#pragma unroll
    for (int v = 0; v < 16; ++v) r[v] = *reinterpret_cast<const f32x4_t*>(at(base + 8 * v * ld, off));
  };
  auto store_rk = [&](float* L, const f32x4_t* r) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int row = 8 * v + (tid >> 5), k4 = 4 * (tid & 31);
#pragma unroll
      for (int e = 0; e < 4; ++e) L[row * KLA + k4 + e] = r[v][e];
    }
  };
  auto store_kn = [&](const f32x4_t* r) {
#pragma unroll
    for (int v = 0; v < 16; ++v)
      *reinterpret_cast<f32x4_t*>(lb + (8 * v + (tid >> 5)) * LBN + 4 * (tid & 31)) = r[v];
  };
  auto b_tile = [&](int64_t t) { return BT ? g.B + t * KT * g.ldb : g.B + t * KT; };

  f32x4_t rv[16];
  load_rows(g.A + m0 * g.lda, g.lda, off_a, rv);
  store_rk(la, rv);
  load_rows(b_tile(nt), g.ldb, off_b, rv);
  if (BT) store_rk(lb, rv); else store_kn(rv);
  __syncthreads();

  for (;;) {
    const int64_t n0 = nt * KT;
    const int64_t nn = nt + gridDim.x;
    const bool more = nn < ntiles && !(g.lower_only && nn * KT > m0);
    if (more) load_rows(b_tile(nn), g.ldb, off_b, rv);
    float* cbase = g.C + m0 * g.ldc + n0;
    float cv[64];
    if (g.beta != 0.f) {
#pragma unroll
      for (int bm = 0; bm < 2; ++bm)
#pragma unroll
        for (int bn = 0; bn < 2; ++bn)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            cv[(bm * 2 + bn) * 16 + r] = *at(cbase + (bm * 32 + 8 * (r >> 2) + (r & 3)) * g.ldc + bn * 32, off_c);
    }
    f32x16_t acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
    // operands of step kk + 1 are read while the MFMAs of step kk run
    // (explicit double buffer + scheduling groups: the default schedule
    // waits for each step's LDS reads right before its MFMAs)
    {
      const float* pa = la + (wm * 64 + (lane & 31)) * KLA + (lane >> 5);
      const float* pb = BT ? lb + (wn * 64 + (lane & 31)) * KLA + (lane >> 5)
                           : lb + (lane >> 5) * LBN + wn * 64 + (lane & 31);
      auto rd = [&](int kk, float* fa, float* fb) __attribute__((always_inline)) {
        fa[0] = pa[2 * kk];
        fa[1] = pa[32 * KLA + 2 * kk];
        fb[0] = BT ? pb[2 * kk] : pb[2 * kk * LBN];
        fb[1] = BT ? pb[32 * KLA + 2 * kk] : pb[2 * kk * LBN + 32];
      };
      float f[2][4];
      rd(0, f[0], f[0] + 2);
#pragma unroll 8
      for (int kk = 0; kk < KT / 2; ++kk) {
        float* cur = f[kk & 1];
        float* nxt = f[(kk + 1) & 1];
        if (kk + 1 < KT / 2) rd(kk + 1, nxt, nxt + 2);
#pragma unroll
        for (int bm = 0; bm < 2; ++bm)
#pragma unroll
          for (int bn = 0; bn < 2; ++bn)
            acc[bm][bn] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[bm], cur[2 + bn], acc[bm][bn], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA of step kk
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one read of step kk + 1
        }
      }
    }
    // Only the diagonal tile of a lower-only product straddles gm >= gn; the
    // stores of every other tile are emitted without a test (a test on a
    // value the compiler cannot see is uniform put each of the 64 stores in
    // a branch of its own, behind exec-mask updates).
    const bool diag = g.lower_only && n0 == m0;
    auto put = [&](auto masked) __attribute__((always_inline)) {
#pragma unroll
      for (int bm = 0; bm < 2; ++bm)
#pragma unroll
        for (int bn = 0; bn < 2; ++bn)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int tm = wm * 64 + bm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            const int tn = wn * 64 + bn * 32 + (lane & 31);
            const float prod = g.alpha * acc[bm][bn][r];
            const float out = g.beta == 0.f ? prod : g.beta * cv[(bm * 2 + bn) * 16 + r] + prod;
            if (!decltype(masked)::value || tm >= tn)
              *const_cast<float*>(at(cbase + (bm * 32 + 8 * (r >> 2) + (r & 3)) * g.ldc + bn * 32, off_c)) = out;
          }
    };
    if (diag) put(std::true_type{}); else put(std::false_type{});
    if (!more) break;
    __syncthreads();  // every wave is done reading lb
    if (BT) store_rk(lb, rv); else store_kn(rv);
    __syncthreads();
    nt = nn;
  }
}

// Skinny K = 128 products (few 128 x 128 tiles: the Cholesky panel solves
// and updates at d = 4096 have N = 128 and at most 31 row tiles) leave most
// CUs idle on the big-tile kernel, and each of its tiles is a long MFMA
// chain.  This variant computes one 64 x 64 tile per workgroup (each wave a
// 32 x 32 quadrant, K = 128 as 64 MFMA steps on two accumulators), so the
// same product spreads over four times as many CUs with a quarter of the
// chain per wave.  Whole tiles only: M and N multiples of 64, 16-byte
// aligned rows.  Both operands sit in LDS as [row][k] (B transposed on the
// way in when it arrives as [k][n]): 66 KB, two workgroups per CU.
constexpr int ST = 64;           // tile edge

template <bool BT>
__global__ __launch_bounds__(GNT, 2) void gemm_k128_small_kernel(GemmArgs g) {
  __shared__ float la[ST * KLA];
  __shared__ float lb[ST * KLA];
  {
    const int64_t bz = blockIdx.z;
    const int64_t b1 = g.inner > 0 ? bz % g.inner : bz, b2 = g.inner > 0 ? bz / g.inner : 0;
    g.A += b1 * g.strideA + b2 * g.strideA2;
    g.B += b1 * g.strideB + b2 * g.strideB2;
    g.C += b1 * g.strideC + b2 * g.strideC2;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t m0 = (int64_t)blockIdx.y * ST, n0 = (int64_t)blockIdx.x * ST;
  if (g.lower_only && n0 > m0) return;

  // A (and B^T) tiles [row][k]: float4 v covers row 8 v + tid / 32, k 4 (tid % 32);
  // B tiles [k][n]: float4 v covers k 16 v + tid / 16, n 4 (tid % 16)
  auto at = [](const float* base, uint32_t off) {
    return reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + off);
  };
  f32x4_t ra[8], rb[8];
  {
    const uint32_t off_a = (uint32_t)((tid >> 5) * g.lda + 4 * (tid & 31)) * 4u;
    const float* pa = g.A + m0 * g.lda;
#pragma unroll
    for (int v = 0; v < 8; ++v) ra[v] = *reinterpret_cast<const f32x4_t*>(at(pa + 8 * v * g.lda, off_a));
    if (BT) {
      const uint32_t off_b = (uint32_t)((tid >> 5) * g.ldb + 4 * (tid & 31)) * 4u;
      const float* pb = g.B + n0 * g.ldb;
#pragma unroll
      for (int v = 0; v < 8; ++v) rb[v] = *reinterpret_cast<const f32x4_t*>(at(pb + 8 * v * g.ldb, off_b));
    } else {
      const uint32_t off_b = (uint32_t)((tid >> 4) * g.ldb + 4 * (tid & 15)) * 4u;
      const float* pb = g.B + n0;
#pragma unroll
      for (int v = 0; v < 8; ++v) rb[v] = *reinterpret_cast<const f32x4_t*>(at(pb + 16 * v * g.ldb, off_b));
    }
  }
  // C quadrant of this wave, fetched while the tiles are staged
  const uint32_t off_c = (uint32_t)((wm * 32 + 4 * (lane >> 5)) * g.ldc + wn * 32 + (lane & 31)) * 4u;
  float* cbase = g.C + m0 * g.ldc + n0;
  float cv[16];
  if (g.beta != 0.f) {
#pragma unroll
    for (int r = 0; r < 16; ++r) cv[r] = *at(cbase + (8 * (r >> 2) + (r & 3)) * g.ldc, off_c);
  }
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    const int row = 8 * v + (tid >> 5), k4 = 4 * (tid & 31);
#pragma unroll
    for (int e = 0; e < 4; ++e) la[row * KLA + k4 + e] = ra[v][e];
  }
  if (BT) {
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const int row = 8 * v + (tid >> 5), k4 = 4 * (tid & 31);
#pragma unroll
      for (int e = 0; e < 4; ++e) lb[row * KLA + k4 + e] = rb[v][e];
    }
  } else {
    // [k][n] float4 -> [n][k]: lanes of a wave hit banks 4 (n / 4) + k % 4, all distinct
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const int k = 16 * v + (tid >> 4), n4 = 4 * (tid & 15);
#pragma unroll
      for (int e = 0; e < 4; ++e) lb[(n4 + e) * KLA + k] = rb[v][e];
    }
  }
  __syncthreads();

  f32x16_t acc0, acc1;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc0[r] = acc1[r] = 0.f;
  const float* pa = la + (wm * 32 + (lane & 31)) * KLA + (lane >> 5);
  const float* pb = lb + (wn * 32 + (lane & 31)) * KLA + (lane >> 5);
#pragma unroll
  for (int kk = 0; kk < KT / 2; kk += 2) {
    const float a0 = pa[2 * kk], a1 = pa[2 * kk + 2];
    const float b0 = pb[2 * kk], b1 = pb[2 * kk + 2];
    acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, acc0, 0, 0, 0);
    acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, acc1, 0, 0, 0);
  }
  const bool diag = g.lower_only && n0 == m0;  // only the diagonal tile straddles gm >= gn
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int tm = wm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
    const int tn = wn * 32 + (lane & 31);
    const float prod = g.alpha * (acc0[r] + acc1[r]);
    const float out = g.beta == 0.f ? prod : g.beta * cv[r] + prod;
    if (!diag || tm >= tn) *const_cast<float*>(at(cbase + (8 * (r >> 2) + (r & 3)) * g.ldc, off_c)) = out;
  }
}

// In-place K = N = 128 products C = alpha A B^T with C the rows of A (the
// Cholesky panel solve F[r, k0:k0+128] <- F[r, k0:k0+128] linv^T).  Each
// workgroup owns whole rows of C - 32 x 128 tiles, all of N - and has read
// all of a tile's A rows before any of its waves writes, so no workgroup reads
// what another one overwrites.  (Two 64-column tiles per row tile would let
// one workgroup overwrite rows its neighbour had not read yet, which happens
// whenever the two do not run at the same time.)  Four waves, each a 32 x 32
// quadrant.  B goes through LDS once into registers (a lane's 64 values), and
// the workgroup walks its matrix's row tiles, the next tile's loads in flight
// under this one's 64 MFMAs (4096 cycles, 1.9 us): with a workgroup per tile,
// which loaded and staged B's 64 KB each time, that took longer than the
// products.  The 15 solves of 64 matrices of order 2048 take 458 us, 663 before.
constexpr int RT = 32;           // rows per tile

__global__ __launch_bounds__(GNT, 1) void gemm_k128_rows_kernel(GemmArgs g) {
  __shared__ float la[2][RT * KLA];
  __shared__ float lb[KT * KLA];
  {
    const int64_t bz = blockIdx.z;
    const int64_t b1 = g.inner > 0 ? bz % g.inner : bz, b2 = g.inner > 0 ? bz / g.inner : 0;
    g.A += b1 * g.strideA + b2 * g.strideA2;
    g.B += b1 * g.strideB + b2 * g.strideB2;
    g.C += b1 * g.strideC + b2 * g.strideC2;
  }
  const int tid = threadIdx.x, lane = tid & 63, wn = tid >> 6;
  const int64_t ntiles = g.M / RT;
  auto at = [](const float* base, uint32_t off) {
    return reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + off);
  };
  // float4 v of a [row][k] tile covers row 8 v + tid / 32, k 4 (tid % 32)
  const int row = tid >> 5, k4 = 4 * (tid & 31);
  const uint32_t off_a = (uint32_t)(row * g.lda + k4) * 4u;
  f32x4_t ra[RT / 8];
  auto load_a = [&](int64_t t) {
    const float* p = g.A + t * RT * g.lda;
#pragma unroll
    for (int v = 0; v < RT / 8; ++v) ra[v] = *reinterpret_cast<const f32x4_t*>(at(p + 8 * v * g.lda, off_a));
  };
  auto store_a = [&](float* l) {
#pragma unroll
    for (int v = 0; v < RT / 8; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) l[(8 * v + row) * KLA + k4 + e] = ra[v][e];
  };
  load_a(blockIdx.y);
  {
    f32x4_t rb[KT / 8];
    const uint32_t off_b = (uint32_t)(row * g.ldb + k4) * 4u;
#pragma unroll
    for (int v = 0; v < KT / 8; ++v) rb[v] = *reinterpret_cast<const f32x4_t*>(at(g.B + 8 * v * g.ldb, off_b));
    store_a(la[0]);
#pragma unroll
    for (int v = 0; v < KT / 8; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) lb[(8 * v + row) * KLA + k4 + e] = rb[v][e];
  }
  const int64_t step = gridDim.y;
  int64_t t = blockIdx.y;
  if (t + step < ntiles) load_a(t + step);
  __syncthreads();   // every A row of a tile is read before any C row of it is written
  const float* pb = lb + (wn * 32 + (lane & 31)) * KLA + (lane >> 5);
  float bv[KT / 2];
#pragma unroll
  for (int kk = 0; kk < KT / 2; ++kk) bv[kk] = pb[2 * kk];
  const uint32_t off_c = (uint32_t)(4 * (lane >> 5) * g.ldc + wn * 32 + (lane & 31)) * 4u;
  for (int buf = 0;; buf ^= 1, t += step) {
    float* cbase = g.C + t * RT * g.ldc;
    float cv[16];
    if (g.beta != 0.f) {
#pragma unroll
      for (int r = 0; r < 16; ++r) cv[r] = *at(cbase + (8 * (r >> 2) + (r & 3)) * g.ldc, off_c);
    }
    f32x16_t acc0, acc1;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc0[r] = acc1[r] = 0.f;
    const float* pa = la[buf] + (lane & 31) * KLA + (lane >> 5);
#pragma unroll
    for (int kk = 0; kk < KT / 2; kk += 2) {
      acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(pa[2 * kk], bv[kk], acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(pa[2 * kk + 2], bv[kk + 1], acc1, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float prod = g.alpha * (acc0[r] + acc1[r]);
      const float out = g.beta == 0.f ? prod : g.beta * cv[r] + prod;
      *const_cast<float*>(at(cbase + (8 * (r >> 2) + (r & 3)) * g.ldc, off_c)) = out;
    }
    if (t + step >= ntiles) break;
    store_a(la[buf ^ 1]);
    if (t + 2 * step < ntiles) load_a(t + 2 * step);
    __syncthreads();
  }
}

// ---------------------------------------------------------------- large-K GEMM
// The solve's products with K >= 256 (GPTQ mid- and super-block lazy
// updates, the Cholesky chain's rank-512 trailing updates, the triangular
// inverse's doubling products): C = beta C + alpha A op(B) on fp32 MFMA
// 32x32x2, tiles of TM x TN on WGM x WGN waves, K in stages of 32.
constexpr int LKK = 32;          // K per stage
// The same products with the operand tiles streamed global -> LDS by the
// gfx950 LDS-DMA load (global_load_lds_dwordx4: no registers, no VALU)
// through a ring of NS stages, so NS - 1 stages of loads are in flight while
// one is multiplied (one stage ahead, with register staging, does not cover
// the memory latency when a CU runs a single workgroup).  Each wave DMA instruction fills 1 KB of LDS
// with 16-byte chunks in lane order; the lanes pick which global chunk lands
// where, which gives the swizzles:
//   [row][k] tiles (A, B^T): 128-byte rows (32 floats), the chunk of k-quad c
//     stored at position c ^ ((row >> 1) & 7), so the 16-byte operand reads of
//     16 consecutive rows fall on 16 distinct bank quads;
//   [k][n] tiles (B): TN * 4-byte rows, the chunk of n-quad c stored at
//     c ^ (8 ((k >> 2) & 1)), so rows k and k + 4 (the two lane halves of one
//     MFMA) read disjoint banks.
// Elements past M, N or K (K, and N for [k][n] tiles, multiples of 4) are
// fetched from a zero chunk.  The K order inside each group of 8 is permuted
// so that one 16-byte LDS read gives a lane its [row][k] operand for four
// MFMAs: MFMA s of group q contracts k = 8q + s (lanes 0-31) with
// k = 8q + 4 + s (lanes 32-63).
typedef __attribute__((address_space(3))) void lds_void_t;
__device__ __attribute__((aligned(16))) const float kZeroF4[4] = {0.f, 0.f, 0.f, 0.f};

__device__ __forceinline__ void dma16(const void* gaddr, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gaddr), "s"(lds_addr) : "memory", "m0");
}

template <int TM, int TN, int WGM, int WGN, bool BT, int NS>
__global__ __launch_bounds__(64 * WGM * WGN, 1) void gemm_dma_kernel(GemmArgs g) {
  constexpr int NW = WGM * WGN;
  constexpr int WTM = TM / WGM, WTN = TN / WGN;      // wave tile
  constexpr int MB = WTM / 32, NB2 = WTN / 32;
  constexpr int NACC = MB * NB2 == 1 ? 2 : MB * NB2;
  constexpr int ABYTES = TM * 128;                    // TM rows x 32 floats
  constexpr int BBYTES = BT ? TN * 128 : LKK * TN * 4;
  constexpr int SBYTES = ABYTES + BBYTES;
  constexpr int DA = ABYTES / 1024 / NW, DB = BBYTES / 1024 / NW;   // DMA instructions per wave and stage
  static_assert(DA * NW * 1024 == ABYTES && DB * NW * 1024 == BBYTES, "tile / wave split");
  constexpr int BROW = TN * 4;                        // bytes per [k][n] row
  constexpr int BRPI = 1024 / BROW;                   // [k][n] rows per DMA instruction
  constexpr int BCH = TN / 4;                         // 16-byte chunks per [k][n] row
  __shared__ __attribute__((aligned(1024))) char lds[NS * SBYTES];
  {
    const int64_t bz = blockIdx.z;
    const int64_t b1 = g.inner > 0 ? bz % g.inner : bz, b2 = g.inner > 0 ? bz / g.inner : 0;
    g.A += b1 * g.strideA + b2 * g.strideA2;
    g.B += b1 * g.strideB + b2 * g.strideB2;
    g.C += b1 * g.strideC + b2 * g.strideC2;
  }
  // tile of this workgroup (1-D grid over mt x nt tiles).  With a triangular
  // operand the tiles with the longest K range are dispatched first (tiles
  // of one n column for a lower B, of one m row from the bottom for a lower
  // A); otherwise each XCD (workgroups are dispatched round-robin over the
  // 8) takes a contiguous m-major run of tiles, which share A rows and B
  // columns in its L2.
  const int64_t mt = (g.M + TM - 1) / TM, ntl = (g.N + TN - 1) / TN, ntot = mt * ntl;
  int64_t tm_i, tn_i;
  {
    const int64_t b = blockIdx.x;
    if (g.b_lower) {
      tn_i = b / mt; tm_i = b % mt;
    } else if (g.a_lower) {
      tm_i = mt - 1 - b / ntl; tn_i = b % ntl;
    } else {
      // (lower-only products keep the round-robin order: the tiles above the
      // diagonal exit at once, so contiguous runs would load XCDs unevenly)
      const int64_t t = ntot % 8 == 0 && !g.lower_only ? (b % 8) * (ntot / 8) + b / 8 : b;
      tm_i = t / ntl; tn_i = t % ntl;
    }
  }
  const int64_t m0 = tm_i * TM, n0 = tn_i * TN;
  if (g.lower_only && m0 + TM - 1 < n0) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  const int64_t kbeg = g.b_lower ? (n0 / LKK) * LKK : 0;
  const int64_t kend = g.a_lower ? (m0 + TM < g.K ? m0 + TM : g.K) : g.K;
  const int64_t nst = kend > kbeg ? (kend - kbeg + LKK - 1) / LKK : 0;

  // DMA sources of this lane: instruction j of the wave covers [row][k] rows
  // 8 u .. 8 u + 7 (u = wave DA + j) or [k][n] rows BRPI u ..
  const float* a_src[DA];
  int a_ck[DA];
  bool a_ok[DA];
#pragma unroll
  for (int j = 0; j < DA; ++j) {
    const int r = 8 * (wave * DA + j) + (lane >> 3);
    a_ck[j] = (lane & 7) ^ ((r >> 1) & 7);
    a_ok[j] = m0 + r < g.M;
    a_src[j] = g.A + (a_ok[j] ? m0 + r : 0) * g.lda + 4 * a_ck[j];
  }
  const float* b_src[DB];
  int b_ck[DB], b_kr[DB];
  bool b_ok[DB];
#pragma unroll
  for (int j = 0; j < DB; ++j) {
    if (BT) {
      const int r = 8 * (wave * DB + j) + (lane >> 3);
      b_ck[j] = (lane & 7) ^ ((r >> 1) & 7);
      b_kr[j] = 0;
      b_ok[j] = n0 + r < g.N;
      b_src[j] = g.B + (b_ok[j] ? n0 + r : 0) * g.ldb + 4 * b_ck[j];
    } else {
      const int kr = BRPI * (wave * DB + j) + lane / BCH;
      const int ck = (lane % BCH) ^ (8 * ((kr >> 2) & 1));
      b_ck[j] = ck;
      b_kr[j] = kr;
      b_ok[j] = n0 + 4 * ck < g.N;
      b_src[j] = g.B + kr * g.ldb + n0 + (b_ok[j] ? 4 * ck : 0);
    }
  }
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((lds_void_t*)lds);
  // DMA instruction i (A first, then B) of stage `stage` (clamped to the last
  // one, so every wave issues the same count) into ring slot stage % NS
  auto issue = [&](int64_t stage, int i) __attribute__((always_inline)) {
    const int64_t sc = stage < nst ? stage : nst - 1;
    const int64_t k0 = kbeg + sc * LKK;
    const uint32_t slot = lds0 + (uint32_t)((stage % NS) * SBYTES);
    if (i < DA) {
      const bool ok = a_ok[i] && k0 + 4 * a_ck[i] < g.K;
      dma16(ok ? (const void*)(a_src[i] + k0) : (const void*)kZeroF4, slot + (uint32_t)((wave * DA + i) * 1024));
    } else {
      const int j = i - DA;
      if (BT) {
        const bool ok = b_ok[j] && k0 + 4 * b_ck[j] < g.K;
        dma16(ok ? (const void*)(b_src[j] + k0) : (const void*)kZeroF4,
              slot + ABYTES + (uint32_t)((wave * DB + j) * 1024));
      } else {
        const bool ok = b_ok[j] && k0 + b_kr[j] < g.K;
        dma16(ok ? (const void*)(b_src[j] + k0 * g.ldb) : (const void*)kZeroF4,
              slot + ABYTES + (uint32_t)((wave * DB + j) * 1024));
      }
    }
  };

  f32x16_t acc[NACC];
#pragma unroll
  for (int a = 0; a < NACC; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[a][r] = 0.f;

  const int half = lane >> 5, l32 = lane & 31;
  const int xr = (l32 >> 1) & 7;                       // row swizzle of this lane's [row][k] rows
  const int a_row = (wm * WTM + l32) * 128;            // + bm * 32 * 128
  const int bt_row = (wn * WTN + l32) * 128;
  // [k][n] read offset of column block bn (its 8 chunks form an aligned block of 8)
  int bk_lane[NB2];
#pragma unroll
  for (int bn = 0; bn < NB2; ++bn)
    bk_lane[bn] = 4 * half * BROW + (((wn * WTN + bn * 32 + l32) >> 2) ^ (8 * half)) * 16 + (l32 & 3) * 4;
  struct Frag { f32x4_t a[MB], b[NB2]; };
  auto read_group = [&](const char* sl, int q, Frag& f) __attribute__((always_inline)) {
    const int ch = ((2 * q + half) ^ xr) * 16;
#pragma unroll
    for (int bm = 0; bm < MB; ++bm) f.a[bm] = *reinterpret_cast<const f32x4_t*>(sl + a_row + bm * 32 * 128 + ch);
#pragma unroll
    for (int bn = 0; bn < NB2; ++bn) {
      if (BT) {
        f.b[bn] = *reinterpret_cast<const f32x4_t*>(sl + ABYTES + bt_row + bn * 32 * 128 + ch);
      } else {
        // column block bn: 32 columns = 8 chunks, XOR by 8 keeps them a block
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2)
          f.b[bn][s2] = *reinterpret_cast<const float*>(sl + ABYTES + bk_lane[bn] + (8 * q + s2) * BROW);
      }
    }
  };
  auto mma_group = [&](const Frag& f) __attribute__((always_inline)) {
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
      for (int bm = 0; bm < MB; ++bm)
#pragma unroll
        for (int bn = 0; bn < NB2; ++bn) {
          const int ai = MB * NB2 == 1 ? (s2 & 1) : bm * NB2 + bn;
          acc[ai] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[bm][s2], f.b[bn][s2], acc[ai], 0, 0, 0);
        }
  };

  constexpr int ND = DA + DB;
  if (nst > 0) {
#pragma unroll
    for (int p = 0; p < NS - 1; ++p)
#pragma unroll
      for (int i = 0; i < ND; ++i) issue(p, i);
    for (int64_t st = 0; st < nst; ++st) {
      // this wave's DMAs of stage st are done (those of the NS - 2 later
      // stages may be in flight) and its LDS reads of stage st - 1 have
      // returned; the barrier makes every wave's DMAs visible and frees the
      // slot of stage st - 1, which takes stage st + NS - 1
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * ND) : "memory");
      const char* sl = lds + (st % NS) * SBYTES;
      Frag f0, f1;
      read_group(sl, 0, f0);
      read_group(sl, 1, f1);
#pragma unroll
      for (int i = 0; i < ND / 2; ++i) issue(st + NS - 1, i);
      mma_group(f0);
      read_group(sl, 2, f0);
      mma_group(f1);
#pragma unroll
      for (int i = ND / 2; i < ND; ++i) issue(st + NS - 1, i);
      read_group(sl, 3, f1);
      mma_group(f0);
      mma_group(f1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  constexpr int NBLK = MB * NB2;
  float cv[NBLK * 16];
  auto gm_of = [&](int bm, int r) { return m0 + wm * WTM + bm * 32 + 8 * (r >> 2) + 4 * half + (r & 3); };
  auto gn_of = [&](int bn) { return n0 + wn * WTN + bn * 32 + l32; };
  if (g.beta != 0.f) {
#pragma unroll
    for (int bm = 0; bm < MB; ++bm)
#pragma unroll
      for (int bn = 0; bn < NB2; ++bn)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t gm = gm_of(bm, r), gn = gn_of(bn);
          cv[(bm * NB2 + bn) * 16 + r] = g.C[(gm < g.M ? gm : g.M - 1) * g.ldc + (gn < g.N ? gn : g.N - 1)];
        }
  }
  // A tile inside C and (lower-only products) wholly on or below the
  // diagonal stores every element without a test; the per-element tests of
  // edge and diagonal tiles put each store in a branch of its own.
  const bool whole = m0 + TM <= g.M && n0 + TN <= g.N && (!g.lower_only || m0 >= n0 + TN - 1);
  auto put = [&](auto masked) __attribute__((always_inline)) {
#pragma unroll
    for (int bm = 0; bm < MB; ++bm)
#pragma unroll
      for (int bn = 0; bn < NB2; ++bn)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t gm = gm_of(bm, r), gn = gn_of(bn);
          if (!decltype(masked)::value || (gm < g.M && gn < g.N && (!g.lower_only || gm >= gn))) {
            const float sum = NBLK == 1 ? acc[0][r] + acc[1][r] : acc[bm * NB2 + bn][r];
            const float prod = g.alpha * sum;
            g.C[gm * g.ldc + gn] = g.beta == 0.f ? prod : g.beta * cv[(bm * NB2 + bn) * 16 + r] + prod;
          }
        }
  };
  if (whole) put(std::false_type{}); else put(std::true_type{});
}

// fp32-accurate products on the bf16 MFMA ("x6"): every fp32 operand value
// v is split exactly into three bf16 parts, v = h + m + l (h = bf16(v),
// m = bf16(v - h), l = v - h - m, which has at most 8 significant bits and
// is exact in bf16; the subtractions are exact in fp32), and a 16-deep slice
// of A B is summed as the six products h h', h m', m h', h l', m m', l h'
// on v_mfma_f32_32x32x16_bf16 (exact products, fp32 accumulation).  The
// three dropped products are below 2^-24 of |a| |b| each, about the rounding
// of one fp32 product; the sum is rounded in the MFMA's fp32 accumulator, as
// on the fp32 MFMA.  Six bf16 MFMAs (192 cycles) replace the eight fp32
// MFMAs (512 cycles) of a 16-deep slice.  (Operands beyond 3.39e38, where
// bf16 rounding overflows, do not occur in the solve's products.)
//
// A split takes 44 VALU instructions per eight values: a wave that splits its
// own operands, as many as its MFMAs take, spends as long on it.  So a
// workgroup splits each value of its tile once: the threads load the fp32
// values of a 32-deep stage into registers, split them and write the three
// parts to LDS in 16-byte chunks of 8 k, ordered [part][k / 8][row], which
// every wave reads as its MFMA operands.  How splits and MFMAs come to overlap
// differs by tile:
//   256 x 128  eight waves, two stages of parts: of the two waves on a SIMD one
//              splits the next stage while the other multiplies this one
//   128 x 128  four waves, one stage of parts; two workgroups on a CU, out of
//              step by themselves
//   64 x 128   four waves with a CU mostly to themselves: two stages, loads two
//              stages ahead, each wave's splits scheduled between its MFMAs
// Lazy updates of 4096 rows, K = 1024, against each wave splitting its own: N =
// 3072 184 -> 131 us, N = 2048 103 -> 83 us; 14336 x 3072 663 -> 441 us; 64
// products of 768 x 1536, K = 512, 514 -> 402 us; 256 x 3072 36 -> 30 us.  The
// sums are the same bits: the same products in the same order.

// two fp32 values to a packed bf16 pair (one v_cvt_pk_bf16_f32, round to
// nearest even), first value in the low half
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
  typedef float f32x2v __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v){a, b}, bf16x2v));
}
// the exact three-part split of a pair: 11 VALU instructions (the bf16
// halves read back as fp32 by a shift and a mask)
__device__ __forceinline__ void split_x6_pair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pk_bf16(a, b);
  const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
  m = pk_bf16(ra, rb);
  const float sa = ra - __uint_as_float(m << 16), sb = rb - __uint_as_float(m & 0xffff0000u);
  l = pk_bf16(sa, sb);
}
__device__ __forceinline__ void split_x6(const f32x4_t& lo4, const f32x4_t& hi4, bf16x8_t* o) {
  uint32_t h[4], m[4], l[4];
  split_x6_pair(lo4[0], lo4[1], h[0], m[0], l[0]);
  split_x6_pair(lo4[2], lo4[3], h[1], m[1], l[1]);
  split_x6_pair(hi4[0], hi4[1], h[2], m[2], l[2]);
  split_x6_pair(hi4[2], hi4[3], h[3], m[3], l[3]);
  o[0] = __builtin_bit_cast(bf16x8_t, (u32x4_t){h[0], h[1], h[2], h[3]});
  o[1] = __builtin_bit_cast(bf16x8_t, (u32x4_t){m[0], m[1], m[2], m[3]});
  o[2] = __builtin_bit_cast(bf16x8_t, (u32x4_t){l[0], l[1], l[2], l[3]});
}

template <int TM, int TN, int WGM, int WGN, bool BT>
__global__ __launch_bounds__(64 * WGM * WGN, 2) void gemm_x6_kernel(GemmArgs g) {
  constexpr int NTH = 64 * WGM * WGN;
  constexpr bool HALVES = NTH == 512, DEEP = TM == 64, DB = HALVES || DEEP;   // DB: two stages of parts
  constexpr int WTM = TM / WGM, WTN = TN / WGN;       // wave tile
  constexpr int MB = WTM / 32, NB2 = WTN / 32;
  constexpr int UA = TM * 4 / NTH, UB = TN * 4 / NTH; // 8-value units of a thread and stage
  static_assert(UA * NTH == TM * 4 && UB * NTH == TN * 4, "tile / thread split");
  // bytes from one 8-deep chunk of all rows to the next: the 32 on top keep the
  // four chunks of a row, written by neighbouring lanes, on different banks
  constexpr int ASTR = TM * 16 + 32, BSTR = TN * 16 + 32;
  constexpr int APL = 4 * ASTR, BPL = 4 * BSTR, BOFF = 3 * APL, STAGE = 3 * (APL + BPL);
  __shared__ __attribute__((aligned(1024))) char lds[(DB ? 2 : 1) * STAGE];
  {
    const int64_t bz = blockIdx.z;
    const int64_t b1 = g.inner > 0 ? bz % g.inner : bz, b2 = g.inner > 0 ? bz / g.inner : 0;
    g.A += b1 * g.strideA + b2 * g.strideA2;
    g.B += b1 * g.strideB + b2 * g.strideB2;
    g.C += b1 * g.strideC + b2 * g.strideC2;
  }
  // tile of this workgroup: as gemm_dma_kernel
  const int64_t mt = (g.M + TM - 1) / TM, ntl = (g.N + TN - 1) / TN, ntot = mt * ntl;
  int64_t tm_i, tn_i;
  {
    const int64_t b = blockIdx.x;
    if (g.b_lower) {
      tn_i = b / mt; tm_i = b % mt;
    } else if (g.a_lower) {
      tm_i = mt - 1 - b / ntl; tn_i = b % ntl;
    } else {
      const int64_t t = ntot % 8 == 0 && !g.lower_only ? (b % 8) * (ntot / 8) + b / 8 : b;
      tm_i = t / ntl; tn_i = t % ntl;
    }
  }
  const int64_t m0 = tm_i * TM, n0 = tn_i * TN;
  if (g.lower_only && m0 + TM - 1 < n0) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  const int64_t kbeg = g.b_lower ? (n0 / LKK) * LKK : 0;
  const int64_t kend = g.a_lower ? (m0 + TM < g.K ? m0 + TM : g.K) : g.K;
  const int64_t nst = kend > kbeg ? (kend - kbeg + LKK - 1) / LKK : 0;

  // This thread's units.  [row][k] operands: row idx / 4, chunk idx % 4 (a row's
  // 128 bytes go to four lanes); [k][n]: column idx % TN, chunk idx / TN.  A
  // chunk is the 8 k a lane gives an MFMA, two runs of four from k_of on and 8
  // further.  Rows past the end repeat the last one: their results are not
  // stored.
  auto k_of = [](int kc) __attribute__((always_inline)) { return 16 * (kc >> 1) + 4 * (kc & 1); };
  uint32_t a_off[UA], b_off[UB];
  int a_lds[UA], b_lds[UB], a_k[UA], b_k[UB];
  const uint32_t b_row = (uint32_t)g.ldb * 4;
#pragma unroll
  for (int u = 0; u < UA; ++u) {
    const int idx = u * NTH + tid, row = idx >> 2, kc = idx & 3;
    const int64_t rc = m0 + row < g.M ? row : g.M - 1 - m0;
    a_off[u] = (uint32_t)(rc * g.lda * 4) + 4 * k_of(kc);
    a_lds[u] = kc * ASTR + row * 16;
    a_k[u] = k_of(kc);
  }
#pragma unroll
  for (int u = 0; u < UB; ++u) {
    const int idx = u * NTH + tid;
    const int row = BT ? idx >> 2 : idx % TN, kc = BT ? idx & 3 : idx / TN;
    const int64_t rc = n0 + row < g.N ? row : g.N - 1 - n0;
    b_off[u] = BT ? (uint32_t)(rc * g.ldb * 4) + 4 * k_of(kc) : (uint32_t)(rc * 4) + k_of(kc) * b_row;
    b_lds[u] = BOFF + kc * BSTR + row * 16;
    b_k[u] = k_of(kc);
  }
  const float* a_base = g.A + m0 * g.lda;
  const float* b_base = BT ? g.B + n0 * g.ldb : g.B + n0;
  struct Regs { f32x4_t a[UA][2], b[UB][2]; };
  auto at = [](const float* p, uint32_t off) __attribute__((always_inline)) {
    return reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + off);
  };
  // The 32 k from k0 on.  A last stage past K (a multiple of 4) reads the
  // stage's first k in place of those past it, which the split then clears.
  auto load = [&](Regs& r, int64_t k0) __attribute__((always_inline)) {
    const int lim = (int)(g.K - k0 < LKK ? g.K - k0 : LKK);
    const float* b_k0 = BT ? b_base + k0 : b_base + k0 * g.ldb;
#pragma unroll
    for (int u = 0; u < UA; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bool ok = a_k[u] + 8 * h < lim;
        r.a[u][h] = *reinterpret_cast<const f32x4_t*>(at(a_base + k0, ok ? a_off[u] + 32 * h : a_off[u] - 4 * a_k[u]));
      }
#pragma unroll
    for (int u = 0; u < UB; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bool ok = b_k[u] + 8 * h < lim;
        if (BT) {
          r.b[u][h] =
              *reinterpret_cast<const f32x4_t*>(at(b_k0, ok ? b_off[u] + 32 * h : b_off[u] - 4 * b_k[u]));
        } else {
          const uint32_t off = ok ? b_off[u] : b_off[u] - b_k[u] * b_row;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            r.b[u][h][e] = *at(b_k0, off + (uint32_t)(8 * h + e < lim ? 8 * h + e : lim - 1) * b_row);
        }
      }
  };
  auto clear_tail = [&](Regs& r, int64_t k0) __attribute__((always_inline)) {
    if (k0 + LKK > g.K) {
      const int lim = (int)(g.K - k0);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int u = 0; u < UA; ++u) r.a[u][h][e] = keep_if(r.a[u][h][e], a_k[u] + 8 * h < lim);
#pragma unroll
          for (int u = 0; u < UB; ++u) r.b[u][h][e] = keep_if(r.b[u][h][e], b_k[u] + 8 * h < lim);
        }
    }
  };
  auto split_only = [&](Regs& r, char* sl) __attribute__((always_inline)) {
    bf16x8_t o[3];
#pragma unroll
    for (int u = 0; u < UA; ++u) {
      split_x6(r.a[u][0], r.a[u][1], o);
#pragma unroll
      for (int t = 0; t < 3; ++t) *reinterpret_cast<bf16x8_t*>(sl + t * APL + a_lds[u]) = o[t];
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      split_x6(r.b[u][0], r.b[u][1], o);
#pragma unroll
      for (int t = 0; t < 3; ++t) *reinterpret_cast<bf16x8_t*>(sl + t * BPL + b_lds[u]) = o[t];
    }
  };

  auto split_store = [&](Regs& r, int64_t k0, char* sl) __attribute__((always_inline)) {
    clear_tail(r, k0);
    split_only(r, sl);
  };

  f32x16_t acc[MB * NB2];
#pragma unroll
  for (int a = 0; a < MB * NB2; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[a][r] = 0.f;
  const int half = lane >> 5, l32 = lane & 31;
  const int a_rd = half * ASTR + (wm * WTM + l32) * 16, b_rd = BOFF + half * BSTR + (wn * WTN + l32) * 16;
  // the six products of a stage's two 16-deep slices, term-major so that
  // consecutive MFMAs update different accumulators
  auto multiply = [&](const char* sl) __attribute__((always_inline)) {
    constexpr int TA[6] = {1, 2, 0, 1, 0, 0}, TB[6] = {1, 0, 2, 0, 1, 0};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8_t fa[MB][3], fb[NB2][3];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
#pragma unroll
        for (int bm = 0; bm < MB; ++bm)
          fa[bm][t] = *reinterpret_cast<const bf16x8_t*>(sl + t * APL + 2 * s * ASTR + a_rd + bm * 512);
#pragma unroll
        for (int bn = 0; bn < NB2; ++bn)
          fb[bn][t] = *reinterpret_cast<const bf16x8_t*>(sl + t * BPL + 2 * s * BSTR + b_rd + bn * 512);
      }
#pragma unroll
      for (int t = 0; t < 6; ++t)
#pragma unroll
        for (int bm = 0; bm < MB; ++bm)
#pragma unroll
          for (int bn = 0; bn < NB2; ++bn)
            acc[bm * NB2 + bn] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[bm][TA[t]], fb[bn][TB[t]], acc[bm * NB2 + bn], 0, 0, 0);
    }
  };
  // LDS reads and writes done, every wave here (the loads into registers may
  // be in flight)
  auto sync = []() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  if (nst > 0) {
    Regs r0;
    load(r0, kbeg);
    if constexpr (HALVES) {
      split_store(r0, kbeg, lds);
      if (nst > 1) load(r0, kbeg + LKK);
      sync();
      // each half of the waves alternates between the two, the second half
      // beginning with the split; both meet once a stage
      const bool split_first = wave >= 4;
      bool skip = split_first;
      for (int64_t m = 0, n = 0;;) {
        if (!skip) {
          multiply(lds + (m & 1) * STAGE);
          ++m;
          if (split_first) {
            sync();
            if (m == nst) break;
          }
        }
        skip = false;
        if (n + 1 < nst) {
          split_store(r0, kbeg + (n + 1) * LKK, lds + ((n + 1) & 1) * STAGE);
          if (n + 2 < nst) load(r0, kbeg + (n + 2) * LKK);
        }
        ++n;
        if (!split_first) {
          sync();
          if (n == nst) break;
        }
      }
    } else if constexpr (DEEP) {
      // a workgroup or two on a CU: the loads two stages ahead, in two sets of
      // registers, and one barrier a stage.  Past the last stage that one is
      // loaded and split again, unread: without branches around them the older
      // set's loads can be waited for while the newer's stay in flight.
      Regs r1;
      auto k_at = [&](int64_t st) __attribute__((always_inline)) { return kbeg + (st < nst ? st : nst - 1) * LKK; };
      load(r1, k_at(1));
      split_store(r0, kbeg, lds);
      load(r0, k_at(2));
      sync();
      auto stage = [&](Regs& r, int64_t st, int buf) __attribute__((always_inline)) {
        clear_tail(r, k_at(st + 1));
        multiply(lds + buf * STAGE);
        split_only(r, lds + (buf ^ 1) * STAGE);
        load(r, k_at(st + 3));
        // all LDS reads, then an MFMA (32 cycles) and the VALU instructions that
        // go beside it, in turn
        __builtin_amdgcn_sched_group_barrier(0x100, 6 * (MB + NB2), 0);
#pragma unroll
        for (int i = 0; i < 12 * MB * NB2; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, (44 * (UA + UB) + 30) / (12 * MB * NB2), 0);
        }
        sync();
      };
      for (int64_t st = 0; st < nst; st += 2) {
        stage(r1, st, 0);
        if (st + 1 < nst) stage(r0, st + 1, 1);
      }
    } else {
      for (int64_t st = 0; st < nst; ++st) {
        split_store(r0, kbeg + st * LKK, lds);
        if (st + 1 < nst) load(r0, kbeg + (st + 1) * LKK);
        sync();
        multiply(lds);
        sync();
      }
    }
  }

  constexpr int NBLK = MB * NB2;
  float cv[NBLK * 16];
  auto gm_of = [&](int bm, int r) { return m0 + wm * WTM + bm * 32 + 8 * (r >> 2) + 4 * half + (r & 3); };
  auto gn_of = [&](int bn) { return n0 + wn * WTN + bn * 32 + l32; };
  if (g.beta != 0.f) {
#pragma unroll
    for (int bm = 0; bm < MB; ++bm)
#pragma unroll
      for (int bn = 0; bn < NB2; ++bn)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t gm = gm_of(bm, r), gn = gn_of(bn);
          cv[(bm * NB2 + bn) * 16 + r] = g.C[(gm < g.M ? gm : g.M - 1) * g.ldc + (gn < g.N ? gn : g.N - 1)];
        }
  }
  // (masked stores at C's edges and the diagonal only: as gemm_dma_kernel)
  const bool whole = m0 + TM <= g.M && n0 + TN <= g.N && (!g.lower_only || m0 >= n0 + TN - 1);
  auto put = [&](auto masked) __attribute__((always_inline)) {
#pragma unroll
    for (int bm = 0; bm < MB; ++bm)
#pragma unroll
      for (int bn = 0; bn < NB2; ++bn)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t gm = gm_of(bm, r), gn = gn_of(bn);
          if (!decltype(masked)::value || (gm < g.M && gn < g.N && (!g.lower_only || gm >= gn))) {
            const float prod = g.alpha * acc[bm * NB2 + bn][r];
            g.C[gm * g.ldc + gn] = g.beta == 0.f ? prod : g.beta * cv[(bm * NB2 + bn) * 16 + r] + prod;
          }
        }
  };
  if (whole) put(std::false_type{}); else put(std::true_type{});
}

// Global-memory pointers of the dataflow factorisation's task functions
// carry their address space: through generic pointers every access becomes
// a flat instruction, which also counts against the LDS counter, so waiting
// for an LDS read would wait for the tile fetches in flight.
typedef __attribute__((address_space(1))) float gfloat;
typedef __attribute__((address_space(1))) int32_t gint;
__device__ __forceinline__ void store4(float* p, const f32x4_t& v) { *reinterpret_cast<f32x4_t*>(p) = v; }
__device__ __forceinline__ void store4(gfloat* p, const f32x4_t& v) {
  *reinterpret_cast<__attribute__((address_space(1))) f32x4_t*>(p) = v;
}

// ---------------------------------------------------------------- Cholesky pieces
constexpr int NB = 128;        // panel width
constexpr int SB = 32;         // register-resident sub-block of the diagonal kernel
constexpr int PNT = 256;       // threads of the diagonal-block kernel (4 waves)
constexpr int LP = NB + 1;     // LDS row stride
constexpr int LT = 2 * SB + 1; // LDS row stride of the product scratch

// 16 x 16 fp32 MFMA tile, operands in LDS: acc += sign * sum_{k in [kb, ke)}
// A[m][k] op(B)[k][n], A row-major (lda), B row-major [k][n] (ldb) or, if bt,
// [n][k].  kb and ke are multiples of 16.  acc[q] is row 4 (lane / 16) + q,
// column lane % 16; the A operand of lane l is row l % 16, k offset l / 16.
// The K ranges follow the triangles: with a lower-triangular operand only
// the k that can be nonzero are visited.
__device__ __forceinline__ void mfma16_tile(f32x4_t& acc, const float* A, int lda, const float* B, int ldb,
                                            bool bt, int kb, int ke, int lane, float sign) {
  const int r = lane & 15, kq = lane >> 4;
#pragma unroll 2
  for (int k0 = kb; k0 < ke; k0 += 16) {
    float av[4], bv[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = k0 + 4 * s + kq;
      av[s] = sign * A[r * lda + k];
      bv[s] = bt ? B[r * ldb + k] : B[k * ldb + r];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s], bv[s], acc, 0, 0, 0);
  }
}

__device__ __forceinline__ f32x4_t tile16_load(const float* C, int ldc, int lane) {
  f32x4_t acc;
#pragma unroll
  for (int q = 0; q < 4; ++q) acc[q] = C[(4 * (lane >> 4) + q) * ldc + (lane & 15)];
  return acc;
}
__device__ __forceinline__ void tile16_store(const f32x4_t& acc, float* C, int ldc, int lane) {
#pragma unroll
  for (int q = 0; q < 4; ++q) C[(4 * (lane >> 4) + q) * ldc + (lane & 15)] = acc[q];
}
__device__ __forceinline__ f32x4_t zero4() {
  f32x4_t z;
  z[0] = z[1] = z[2] = z[3] = 0.f;
  return z;
}

// Inverse X = L^-1 of the lower Cholesky factor of an NB x NB diagonal
// block.  L itself is not written back: the blocked Cholesky only consumes
// L^-1 (panel solves and the triangular inverse) and the off-diagonal
// panels.
//
// The block is processed in 32-wide steps.  Wave 0 factors the 32 x 32
// diagonal sub-block in registers and inverts it on the way; all four waves
// apply the sub-block inverse to the panel below, and the trailing lower
// triangle is updated with fp32 MFMA (16 x 16 tiles), the next diagonal
// sub-block first so that its factorisation overlaps the rest.  The block
// inverse is assembled from the four sub-block inverses by two doubling
// steps, inv([[A,0],[B,C]]) = [[A^-1,0],[-C^-1 B A^-1, C^-1]], partly under
// the last factorisations.
//
// On entry `a` (NB x NB, row
// stride LP, LDS) holds the lower triangle of the block with zeros above,
// visible to the whole workgroup; on exit the rows of L^-1 (zeros above the
// diagonal) are in `out` (row stride ldo) and in `x` (LDS, row stride LP;
// x's strictly upper 32 x 32 sub-blocks are never written).  `t` and `cb`
// are scratch (3 SB LT and 2 SB floats, 16-byte aligned).  Every thread of
// the PNT-thread workgroup calls it.
template <typename OutPtr>
__device__ __forceinline__ void potf2_inv_lds(float* a, float* x, float* t, float* cb, OutPtr out, int64_t ldo,
                                              int32_t* status) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // pivot check, off the dependency chain: every pivot positive and finite
  // (denormals included), tested on the bits of the wave-uniform pivot with
  // integer compares, which run on the scalar unit beside the column updates
  int pd_ok = 1;

  // Factor + invert the 32 x 32 diagonal sub-block at o (wave 0 only).
  // Lanes 0..31 hold the rows of the sub-block (row role), lanes 32..63 the
  // columns of its inverse (column role): v = row li of A, or column li of
  // X = L^-1, initially e_li.  Right-looking Cholesky and the inverse's row
  // elimination (X[j][:] /= L[j][j]; X[i][:] -= L[i][j] X[j][:], i > j)
  // advance together, and with col = A[:, j] before scaling both take the
  // same form:
  //   m = v[j] / piv;  v[k] -= m col[k] (k > j);  v[j] /= L[j][j]
  // Column j reaches every lane through one LDS write and broadcast reads (a
  // wave's LDS operations complete in program order, so no barrier is
  // needed).  Entries above the diagonal are updated too and never used,
  // which keeps every update unpredicated.
  //
  // The column loop is latency-bound (one wave, 128 sequential steps per
  // block), so its dependency chain is kept short: rl = 1 / L[j][j] straight
  // from the hardware reciprocal square root (within 1 ulp), and the column
  // is scaled by the reciprocal, as LAPACK's potf2 scales it (dscal by
  // 1 / ajj).  The values on the chain from one step to the next, the pivot
  // col[j] and col[j + 1], col[j + 2] (the updates of the next two columns,
  // made first), are taken from their lanes with v_readlane; the rest of the
  // column goes through LDS, written and read a step ahead of its use, so
  // the LDS round trip stays off the chain.
  auto factor = [&](int o) __attribute__((always_inline)) {
    const int li = lane & 31;
    const bool row_role = lane < SB;
    float v[SB];
#pragma unroll
    for (int c = 0; c < SB; ++c) v[c] = row_role ? a[(o + li) * LP + o + c] : ((c == li) ? 1.f : 0.f);
    // every lane stores (column-role lanes into a scratch slot): no
    // divergent branch around the LDS write that the reads could sink into.
    // Only col[j + 3 .. SB - 1] is read from LDS, exactly those elements (a
    // loaded element that is never used frees its register while the load
    // may still be in flight, and the register's next use would wait for it)
    float col[SB];
    auto read_col = [&](int j, float* c) __attribute__((always_inline)) {
      int k = j;
      if (k & 1) {
        c[k] = cb[k];
        ++k;
      }
      if ((k & 3) == 2) {
        const f32x2_t w = *reinterpret_cast<const f32x2_t*>(cb + k);
        c[k] = w[0];
        c[k + 1] = w[1];
        k += 2;
      }
#pragma unroll
      for (; k < SB; k += 4) {
        const f32x4_t w = *reinterpret_cast<const f32x4_t*>(cb + k);
        c[k] = w[0];
        c[k + 1] = w[1];
        c[k + 2] = w[2];
        c[k + 3] = w[3];
      }
    };
    // lane l's x (l a constant below SB: a row-role lane)
    auto from_lane = [](float x, int l) __attribute__((always_inline)) {
      return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));
    };
    // chain values of step j: piv = col[j], c1 = col[j + 1], c2 = col[j + 2]
    float piv = from_lane(v[0], 0), c1 = from_lane(v[0], 1), c2 = from_lane(v[0], 2);
    cb[lane] = v[0];
    read_col(3, col);
#pragma unroll
    for (int j = 0; j < SB; ++j) {
      {
        const int pb = __builtin_bit_cast(int, piv);
        pd_ok &= (pb > 0) & (pb < 0x7f800000);
      }
      const float rl = __builtin_amdgcn_rsqf(piv);
      const float sj = v[j] * rl;
      const float m = sj * rl;
      // software pipeline: the next two columns are updated first, the
      // next step's chain values read from their lanes and the next column
      // written and read back, then this step's other updates
      float ncol[SB], npiv = 0.f, nc1 = 0.f, nc2 = 0.f;
      if (j + 1 < SB) {
        v[j + 1] = fmaf(-m, c1, v[j + 1]);
        if (j + 2 < SB) v[j + 2] = fmaf(-m, c2, v[j + 2]);
        npiv = from_lane(v[j + 1], j + 1);
        if (j + 2 < SB) nc1 = from_lane(v[j + 1], j + 2);
        if (j + 3 < SB) nc2 = from_lane(v[j + 1], j + 3);
        if (j + 4 < SB) {
          cb[lane] = v[j + 1];
          read_col(j + 4, ncol);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int k = j + 3; k < SB; ++k) v[k] = fmaf(-m, col[k], v[k]);
      v[j] = sj;
      // (keeps the next step's chain from being scheduled into these updates)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = j + 4; k < SB; ++k) col[k] = ncol[k];
      piv = npiv;
      c1 = nc1;
      c2 = nc2;
    }
    // column li of the sub-block inverse, zeros above the diagonal included
    if (!row_role) {
#pragma unroll
      for (int i = 0; i < SB; ++i) x[(o + i) * LP + o + li] = v[i];
    }
  };
  // trailing tile tt (16 x 16, lower triangle of the region below / right of
  // sub-block o, enumerated row by row): A[ti][tj] -= P_ti P_tj^T
  auto trailing_tile = [&](int o, int tt) __attribute__((always_inline)) {
    const int rb = o + SB;
    int ti = 0, rem = tt;
    while (rem > ti) { rem -= ti + 1; ++ti; }
    const int tj = rem;
    float* cp = a + (rb + 16 * ti) * LP + rb + 16 * tj;
    f32x4_t acc = tile16_load(cp, LP, lane);
    mfma16_tile(acc, a + (rb + 16 * ti) * LP + o, LP, a + (rb + 16 * tj) * LP + o, LP, true, 0, SB, lane, -1.f);
    tile16_store(acc, cp, LP, lane);
  };
  // one wave: X[c0][a0] = -X[c0][c0] L[c0][a0] X[a0][a0] for the 32-wide pair
  // (a0, c0 = a0 + 32), through T (32 x 32 at tp); the wave's own LDS writes
  // and reads stay in program order
  auto pair_one_wave = [&](int a0, float* tp) __attribute__((always_inline)) {
    const int c0 = a0 + SB;
#pragma unroll
    for (int tr = 0; tr < 2; ++tr) {
      const float* A = a + (c0 + 16 * tr) * LP + a0;
      f32x4_t acc0 = zero4(), acc1 = zero4();
      mfma16_tile(acc0, A, LP, x + a0 * LP + a0, LP, false, 0, SB, lane, 1.f);
      mfma16_tile(acc1, A, LP, x + a0 * LP + a0 + 16, LP, false, 16, SB, lane, 1.f);
      tile16_store(acc0, tp + 16 * tr * LT, LT, lane);
      tile16_store(acc1, tp + 16 * tr * LT + 16, LT, lane);
    }
#pragma unroll
    for (int tc = 0; tc < 2; ++tc) {
      f32x4_t acc0 = zero4(), acc1 = zero4();
      mfma16_tile(acc0, x + c0 * LP + c0, LP, tp + 16 * tc, LT, false, 0, 16, lane, -1.f);
      mfma16_tile(acc1, x + (c0 + 16) * LP + c0, LP, tp + 16 * tc, LT, false, 0, SB, lane, -1.f);
      tile16_store(acc0, x + c0 * LP + a0 + 16 * tc, LP, lane);
      tile16_store(acc1, x + (c0 + 16) * LP + a0 + 16 * tc, LP, lane);
    }
  };
  // level-2 first product, row strip r: T2[16 r..][0:64] = L[64 + 16 r..][0:64] X[0:64][0:64]
  auto level2_strip = [&](int r) __attribute__((always_inline)) {
    const float* A = a + (2 * SB + 16 * r) * LP;
#pragma unroll
    for (int tc = 0; tc < 4; ++tc) {
      f32x4_t acc = zero4();
      mfma16_tile(acc, A, LP, x + 16 * tc, LP, false, 16 * tc, 2 * SB, lane, 1.f);
      tile16_store(acc, t + 16 * r * LT + 16 * tc, LT, lane);
    }
  };

  // rows r0 .. r0 + 63 of L^-1 to linv, zeros above the diagonal, by `nthr`
  // threads (thread index q): float4 v covers row r0 + v nthr / 32 + q / 32,
  // columns 4 (q % 32) .. + 3
  auto store_rows = [&](int r0, int q, int nthr) __attribute__((always_inline)) {
    const int j = 4 * (q & 31);
    for (int i = r0 + (q >> 5); i < r0 + 2 * SB; i += nthr / 32) {
      f32x4_t o4;
#pragma unroll
      for (int c = 0; c < 4; ++c) o4[c] = (j + c <= i) ? x[i * LP + j + c] : 0.f;
      store4(out + i * ldo + j, o4);
    }
  };

  // Lookahead: after the panel of sub-block kb, the three 16 x 16 trailing
  // tiles that form the next diagonal sub-block are updated first; then
  // wave 0 factors sub-block kb + 1 while waves 1..3 finish the trailing
  // update of kb and the inverse products whose inputs are complete (the
  // pair (0, 1) during factor 2, the first level-2 product during factor 3).
  if (wave == 0) factor(0);
  __syncthreads();
#pragma unroll 1
  for (int kb = 0; kb < NB / SB; ++kb) {
    const int o = kb * SB;
    // panel below the sub-block: P = A_panel Xd^T in place, 16 rows per unit
    // (both column tiles of a unit in one wave, read before written);
    // Xd^T is upper triangular, so column tile c needs k < 16 (c + 1)
    const int R = NB - o - SB;
    for (int u = wave; u < R / 16; u += PNT / 64) {
      float* ap = a + (o + SB + 16 * u) * LP + o;
      f32x4_t acc0 = zero4(), acc1 = zero4();
      mfma16_tile(acc0, ap, LP, x + o * LP + o, LP, true, 0, 16, lane, 1.f);
      mfma16_tile(acc1, ap, LP, x + (o + 16) * LP + o, LP, true, 0, 32, lane, 1.f);
      tile16_store(acc0, ap, LP, lane);
      tile16_store(acc1, ap + 16, LP, lane);
    }
    __syncthreads();
    if (kb + 1 == NB / SB) break;
    // the next diagonal sub-block: trailing tiles 0, 1, 2
    if (wave < 3) trailing_tile(o, wave);
    __syncthreads();
    const int nt = R / 16, ntt = nt * (nt + 1) / 2;
    if (wave == 0) {
      factor(o + SB);
    } else if (kb == 1 && wave == 3) {
      pair_one_wave(0, t + 2 * SB * LT - SB * LT);  // T of pair (0, 1) in rows 32..63 of t
    } else {
      const int nw = kb == 1 ? 2 : 3;             // waves 1..nw share the remaining tiles
      for (int tt = 3 + (wave - 1); tt < ntt; tt += nw) trailing_tile(o, tt);
      if (kb == 2) {
        // first level-2 product, row strips 0..3 over waves 1..3; waves 2
        // and 3 then store rows 0..63 of L^-1, final since the pair (0, 1)
        level2_strip(wave - 1);
        if (wave == 1) level2_strip(3);
        else store_rows(0, tid - 128, 128);
      }
    }
    __syncthreads();
  }
  if (wave == 0 && lane == 0 && status && !pd_ok) *status = MI355Q_NOT_POSITIVE_DEFINITE;

  // pair (2, 3): T_1 = L[96:128][64:96] X[64:96][64:96]; X[96:128][64:96] = -X[96:128][96:128] T_1
  {
    const int tr = wave >> 1, tc = wave & 1;
    f32x4_t acc = zero4();
    mfma16_tile(acc, a + (3 * SB + 16 * tr) * LP + 2 * SB, LP, x + 2 * SB * LP + 2 * SB + 16 * tc, LP, false,
                16 * tc, SB, lane, 1.f);
    tile16_store(acc, t + (2 * SB + 16 * tr) * LT + 16 * tc, LT, lane);
  }
  __syncthreads();
  {
    const int tr = wave >> 1, tc = wave & 1;
    f32x4_t acc = zero4();
    mfma16_tile(acc, x + (3 * SB + 16 * tr) * LP + 3 * SB, LP, t + 2 * SB * LT + 16 * tc, LT, false, 0,
                16 * (tr + 1), lane, -1.f);
    tile16_store(acc, x + (3 * SB + 16 * tr) * LP + 2 * SB + 16 * tc, LP, lane);
  }
  __syncthreads();
  // X[64:128][0:64] = -X[64:128][64:128] T2, one 16-column strip per wave:
  // row tile tr needs k < 16 (tr + 1); the B values of a k step are shared
  // by the row tiles and the four accumulators interleave
  {
    const int r = lane & 15, kq = lane >> 4;
    f32x4_t acc[4];
#pragma unroll
    for (int tr = 0; tr < 4; ++tr) acc[tr] = zero4();
#pragma unroll
    for (int k4 = 0; k4 < 16; ++k4) {
      const int k = 4 * k4 + kq;
      const float bv = t[k * LT + 16 * wave + r];
#pragma unroll
      for (int tr = k4 / 4; tr < 4; ++tr) {
        const float av = -x[(2 * SB + 16 * tr + r) * LP + 2 * SB + k];
        acc[tr] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv, acc[tr], 0, 0, 0);
      }
    }
#pragma unroll
    for (int tr = 0; tr < 4; ++tr) tile16_store(acc[tr], x + (2 * SB + 16 * tr) * LP + 16 * wave, LP, lane);
  }
  __syncthreads();

  // rows 64..127 of L^-1 (rows 0..63 went out during the last factorisation)
  store_rows(2 * SB, tid, PNT);
}

// The diagonal block at (k0, k0) of F into linv (NB x NB, zeros above the
// diagonal).  nb <= NB is the block size; rows / columns beyond nb are
// padded with the identity so the whole NB block factors uniformly.
__global__ __launch_bounds__(PNT) void potf2_inv_kernel(const float* F, int64_t ldf, int64_t k0, int nb,
                                                        float* linv, int32_t* status, int64_t wsf) {
  __shared__ float a[NB * LP];
  __shared__ float x[NB * LP];
  // product scratch: rows 0..63 the first level-2 product (and, earlier, the
  // pair (0, 1) in rows 32..63), rows 64..95 the pair (2, 3)
  __shared__ __attribute__((aligned(16))) float t[3 * SB * LT];
  __shared__ __attribute__((aligned(16))) float cb[2 * SB];  // column broadcast of the factorisation
  const int tid = threadIdx.x;
  // matrix blockIdx.x of a batch: workspaces wsf floats apart
  F += (int64_t)blockIdx.x * wsf;
  linv += (int64_t)blockIdx.x * wsf;
  status += blockIdx.x;

  // load the lower triangle (zeros above): thread tid covers columns
  // 4 (tid % 32) .. + 3 of rows 8 v + tid / 32
  if (nb == NB && (ldf & 3) == 0) {
    const int i0 = tid >> 5, j = 4 * (tid & 31);
    const float* src = F + (k0 + i0) * ldf + k0 + j;
    f32x4_t lv[NB * NB / (4 * PNT)];
#pragma unroll
    for (int v = 0; v < NB * NB / (4 * PNT); ++v) lv[v] = *reinterpret_cast<const f32x4_t*>(src + 8 * v * ldf);
#pragma unroll
    for (int v = 0; v < NB * NB / (4 * PNT); ++v) {
      const int i = 8 * v + i0;
#pragma unroll
      for (int c = 0; c < 4; ++c) a[i * LP + j + c] = (j + c <= i) ? lv[v][c] : 0.f;
    }
  } else {
    // ragged block: addresses clamped into the block, identity padding
    float lv[NB * NB / PNT];
#pragma unroll
    for (int v = 0; v < NB * NB / PNT; ++v) {
      const int e = v * PNT + tid;
      const int i = min(e / NB, nb - 1), j = min(e % NB, nb - 1);
      lv[v] = F[(k0 + i) * ldf + (k0 + j)];
    }
#pragma unroll
    for (int v = 0; v < NB * NB / PNT; ++v) {
      const int e = v * PNT + tid;
      const int i = e / NB, j = e % NB;
      a[i * LP + j] = (i < nb && j < nb && j <= i) ? lv[v] : ((i == j) ? 1.f : 0.f);
    }
  }
  __syncthreads();
  potf2_inv_lds(a, x, t, cb, linv, NB, status);
}

// ---------------------------------------------------------------- dataflow Cholesky + inverse
// For d a multiple of NB, one persistent launch does the work of the blocked
// chain and of the doubling inverse: it factors F = L L^T in NB x NB tiles
// and builds X = L^-1 alongside, with no launch boundary between dependent
// steps (each costs about 4 us on gfx950, and the chain is a sequence of
// small dependent steps).  For tile (i, j), i >= j, of matrix b:
//   chain (one workgroup per matrix: the critical path), j = 0, 1, ...:
//     wait for the diagonal tile A_jj fully updated, factor and invert it
//     into X_jj = L_jj^-1;
//   S(c, s), s = 0..3 (helpers, one per 32-row strip of tile row c + 1):
//     accumulate strip s of A_{c+1,c} and of the diagonal tile's lower
//     blocks A_{c+1,c+1}[s][0..s] over k < c, then (once X_cc is out) its
//     rows of L_{c+1,c} = A_{c+1,c} X_cc^T, then (once the strips above are
//     out) A_{c+1,c+1}[s][0..s] -= L_{c+1,c}[s] L_{c+1,c}[0..s]^T.  Four
//     workgroups share the chain's step between two factorisations;
//   H(i, c), i >= c + 2 (helpers): A_ic -= sum_{k < c} L_ik L_ck^T, then
//     L_ic = A_ic X_cc^T;
//   V(c, j) (helpers): X_cj = -X_cc sum_{k=j}^{c-1} L_ck X_kj.
// hinv = J X J is written by the tasks themselves (V its tile and the zero
// tile mirrored below the diagonal, S(c, 0) the diagonal tile of X_cc once
// its own work is done, the chain the last one), so no flip pass follows.
// Helpers take tasks from one counter in an order where every input comes
// earlier - level 0: H(2.., 0); level c >= 1: S(c-1, 0..3), H(c+2.., c),
// V(c, 0..c-1); the chain's step c counted right after S(c-1, 3) - so the
// earliest unfinished task always has its inputs: the launch needs no
// co-residency beyond one helper next to the chains.  A tile is published by
// a release store of its flag after its data; consumers poll with relaxed
// loads and acquire once.  Every wait is bounded: past `timeout` wall-clock
// ticks the waiter marks its matrix MI355Q_TIMEOUT and raises the abort word,
// after which every wait returns at once and all workgroups drain.
//
// Flags (int32, per matrix in its workspace): lf[i T + j] = 1 when tile
// (i, j) of F holds L_ij (i > j) or X_jj is in X (i == j); xf[i T + j] = 1
// when X_ij (i > j) is in X; st[4 c + s] = 1 when strip s of L_{c+1,c} is
// out; nd[c] counts the strips of A_{c+1,c+1} fully updated, which the chain
// waits for itself; nl[c] counts the strips done with both, the last of which
// sets L_{c+1,c}'s lf (for H tasks and later S, which need it only after the
// chain's next factorisation).  Matrix 0's area then holds the
// task counter and the abort word.  diag_damp_kernel clears them.
constexpr int DSM = 2 * NB * LP + 3 * SB * LT + 2 * SB;  // LDS floats (157 KB: one workgroup per CU)

constexpr int DLB = NB + 32;                             // LDS row stride of [k][n] tiles
constexpr int DAG_LF_FINAL = 1;
// flags per matrix: lf, xf (T^2 each), st (4 T), nl, nd (T each), then counter and abort word
__host__ __device__ constexpr int64_t dag_nflags(int64_t T) { return 2 * T * T + 6 * T + 2; }

struct DagParams {
  float* F;          // workspaces, wsf floats apart
  float* X;
  int32_t* flags;    // DAG_NFLAGS(T) flags per matrix (wsf apart); matrix 0's end with the counter and abort word
  int32_t* status;   // [batch]
  int64_t d, wsf;
  int T, batch, ntasks;
  uint64_t timeout;  // wall-clock ticks per wait
  // hinv = J X J (upper), written by the tasks that produce X's tiles
  float* hinv;
  int64_t shinv;
};

// thread tid's share of a 128 x 128 global tile: float4 v at row 8 v + tid / 32, columns 4 (tid % 32)
__device__ __forceinline__ void dag_fetch(const gfloat* g, int64_t ld, f32x4_t (&v)[16]) {
  typedef __attribute__((address_space(1))) const f32x4_t gf4;
  const int tid = threadIdx.x;
  const gfloat* p = g + (tid >> 5) * ld + 4 * (tid & 31);
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = *reinterpret_cast<gf4*>(p + 8 * i * ld);
}
// ... into LDS as [r][k] (row stride LP)
__device__ __forceinline__ void dag_put_rk(const f32x4_t (&v)[16], float* l) {
  const int tid = threadIdx.x, r0 = tid >> 5, c = 4 * (tid & 31);
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) l[(8 * i + r0) * LP + c + e] = v[i][e];
}
// ... into LDS as [k][n] (row stride DLB)
__device__ __forceinline__ void dag_put_kn(const f32x4_t (&v)[16], float* l) {
  const int tid = threadIdx.x, r0 = tid >> 5, c = 4 * (tid & 31);
#pragma unroll
  for (int i = 0; i < 16; ++i) *reinterpret_cast<f32x4_t*>(l + (8 * i + r0) * DLB + c) = v[i];
}

// 128 x 128 accumulator over four waves: wave (wm, wn) holds the 64 x 64
// quadrant (wm, wn) as 2 x 2 fp32 32x32 MFMA tiles; element r of tile
// (bm, bn) is row 64 wm + 32 bm + 8 (r / 4) + 4 (lane / 32) + r % 4, column
// 64 wn + 32 bn + lane % 32.
struct DagAcc {
  f32x16_t t[2][2];
};
template <typename Fn>
__device__ __forceinline__ void dag_each(Fn&& fn) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 1, wn = wave & 1;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        fn(bm, bn, r, wm * 64 + bm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), wn * 64 + bn * 32 + (lane & 31));
}
__device__ __forceinline__ void dag_zero(DagAcc& acc) {
  dag_each([&](int bm, int bn, int r, int, int) { acc.t[bm][bn][r] = 0.f; });
}
__device__ __forceinline__ void dag_load_acc(DagAcc& acc, const gfloat* g, int64_t ld) {
  dag_each([&](int bm, int bn, int r, int row, int col) { acc.t[bm][bn][r] = g[row * ld + col]; });
}
__device__ __forceinline__ void dag_store_acc(const DagAcc& acc, gfloat* g, int64_t ld) {
  dag_each([&](int bm, int bn, int r, int row, int col) { g[row * ld + col] = acc.t[bm][bn][r]; });
}

// acc += sign * A op(B): A in LDS as [r][k] (stride LP); B as [k][n]
// (stride DLB) if BKN, else as [n][k] (stride LP); K = 128.  Operands of
// step kk + 1 are read while the MFMAs of step kk run.
template <bool BKN>
__device__ __forceinline__ void dag_mma(DagAcc& acc, const float* la, const float* lb, float sign) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 1, wn = wave & 1;
  const float* pa = la + (wm * 64 + (lane & 31)) * LP + (lane >> 5);
  const float* pb = BKN ? lb + (lane >> 5) * DLB + wn * 64 + (lane & 31) : lb + (wn * 64 + (lane & 31)) * LP + (lane >> 5);
  for (int c = 0; c < NB / 32; ++c) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int k2 = 32 * c + 2 * q;
      const float a0 = sign * pa[k2], a1 = sign * pa[32 * LP + k2];
      const float b0 = BKN ? pb[k2 * DLB] : pb[k2], b1 = BKN ? pb[k2 * DLB + 32] : pb[32 * LP + k2];
      acc.t[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, acc.t[0][0], 0, 0, 0);
      acc.t[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b1, acc.t[0][1], 0, 0, 0);
      acc.t[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b0, acc.t[1][0], 0, 0, 0);
      acc.t[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, acc.t[1][1], 0, 0, 0);
    }
  }
}

// The chain's two products, shaped by the triangles.  Sub-diagonal solve
// L = A X^T with X lower triangular: out[r][n] = sum_{k < 32 (n / 32 + 1)}
// A[r][k] X[n][k]; wave (wm, wn) holds row blocks 2 wm, 2 wm + 1 and column
// blocks 3 - wn, wn (K = 128 + 32 or 96 + 64: equal work per wave).
template <typename Fn>
__device__ __forceinline__ void dag_each_tri(Fn&& fn) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 1, wn = wave & 1;
#pragma unroll
  for (int bm = 0; bm < 2; ++bm)
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        fn(bm, bn, r, wm * 64 + bm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3),
           32 * (bn == 0 ? 3 - wn : wn) + (lane & 31));
}
__device__ __forceinline__ void dag_mma_tri(DagAcc& acc, const float* la, const float* x) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 1, wn = wave & 1;
  const int ca = 3 - wn, cbk = wn;
  const float* pa = la + (wm * 64 + (lane & 31)) * LP + (lane >> 5);
  const float* pba = x + (32 * ca + (lane & 31)) * LP + (lane >> 5);
  const float* pbb = x + (32 * cbk + (lane & 31)) * LP + (lane >> 5);
  // K in chunks of 32 (16 MFMA steps): both column blocks while the
  // shorter one lasts, then the longer one alone.  The operands of step
  // k + 1 are read while the MFMAs of step k run (one read after each MFMA).
  float f[2][4];
  auto rd = [&](int k2, float* g) __attribute__((always_inline)) {
    g[0] = pa[k2];
    g[1] = pa[32 * LP + k2];
    g[2] = pba[k2];
    g[3] = pbb[k2];
  };
  rd(0, f[0]);
  for (int c = 0; c <= cbk; ++c) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const float* cur = f[q & 1];
      float* nxt = f[(q + 1) & 1];
      rd(32 * c + 2 * q + 2, nxt);  // (past the short block: read, unused)
      acc.t[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[0], cur[2], acc.t[0][0], 0, 0, 0);
      acc.t[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[0], cur[3], acc.t[0][1], 0, 0, 0);
      acc.t[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[1], cur[2], acc.t[1][0], 0, 0, 0);
      acc.t[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[1], cur[3], acc.t[1][1], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    }
  }
  for (int c = cbk + 1; c <= ca; ++c) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const float* cur = f[q & 1];
      float* nxt = f[(q + 1) & 1];
      if (c < ca || q < 15) {
        const int k2 = 32 * c + 2 * q + 2;
        nxt[0] = pa[k2];
        nxt[1] = pa[32 * LP + k2];
        nxt[2] = pba[k2];
      }
      acc.t[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[0], cur[2], acc.t[0][0], 0, 0, 0);
      acc.t[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[1], cur[2], acc.t[1][0], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
  }
}

// Every wave's stores have reached the L2 (their acknowledgements count down
// vmcnt): one release by thread 0 then writes all of them back.  (A release
// fence in every wave before it is a second write-back in line.  The chain of
// d = 4096 is 31 steps of four such hand-overs each, so what stands between
// them counts: with one write-back each, the strips' flags polled side by
// side and the diagonal tile's count read by the chain itself, the launch
// takes 1190 us, 1360 before; 17 of the 37 us of a step are the diagonal
// tile's factorisation.)
__device__ __forceinline__ void dag_stores_done() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}
// Publish: every wave's stores complete and written back, then the flag.
__device__ __forceinline__ void dag_publish(gint* flag, int v) {
  dag_stores_done();
  if (threadIdx.x == 0) __hip_atomic_store(flag, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

// One LDS allocation shared by the task functions below (157 KB: one
// workgroup per CU); separate functions keep the chain's register
// allocation apart from the helpers'.
__shared__ __attribute__((aligned(16))) float dag_smem[DSM];
__shared__ int dag_word;

// Wait until the n flags from `flag` on are all >= v; false when the wait was
// abandoned (time-out or abort).  Thread 0 polls them side by side; the
// workgroup leaves together.
__device__ __forceinline__ bool dag_wait(const gint* flag, int v, const DagParams& p, int b, int n = 1) {
  if (threadIdx.x == 0) {
    gint* abort_word = (gint*)p.flags + dag_nflags(p.T) - 1;
    int ok = 1;
    auto low = [&]() __attribute__((always_inline)) {
      int f[3];
#pragma unroll
      for (int q = 0; q < 3; ++q)
        f[q] = __hip_atomic_load(flag + (q < n ? q : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return min(f[0], min(f[1], f[2]));
    };
    auto one = [&]() __attribute__((always_inline)) {
      return __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto reached = [&]() __attribute__((always_inline)) { return (n > 1 ? low() : one()) >= v; };
    if (!reached()) {
      const uint64_t t0 = wall_clock64();
      for (;;) {
        __builtin_amdgcn_s_sleep(1);
        if (reached()) break;
        if (__hip_atomic_load(abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
          p.status[b] = MI355Q_TIMEOUT;  // this matrix's results are incomplete too
          ok = 0;
          break;
        }
        if (wall_clock64() - t0 > p.timeout) {
          p.status[b] = MI355Q_TIMEOUT;
          __hip_atomic_store(abort_word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ok = 0;
          break;
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    dag_word = ok;
  }
  __syncthreads();
  const bool ok = dag_word != 0;
  __syncthreads();
  return ok;
}

__device__ __forceinline__ gfloat* dag_tile(float* base, const DagParams& p, int b, int i, int j) {
  return (gfloat*)base + (int64_t)b * p.wsf + (int64_t)i * NB * p.d + (int64_t)j * NB;
}
__device__ __forceinline__ gint* dag_lf(const DagParams& p, int b) { return (gint*)p.flags + (int64_t)b * p.wsf; }

// F[a][c] of matrix b as the preparation kernel wrote it (read once, by the
// task that owns the tile).  (Reading H itself instead, with the flip, the
// scaling and the diagonal rules in the tasks, measured slower than the
// preparation kernel: 1.448 against 1.438 ms at d = 4096, 6.07 against 5.86
// at 8192.)
__device__ __forceinline__ float dag_orig(const DagParams& p, int b, int64_t a, int64_t c) {
  return ((const gfloat*)p.F)[(int64_t)b * p.wsf + a * p.d + c];
}

// X tile (i, j) of matrix b into hinv = J X J: element (r, c) of the tile
// goes to hinv[d-1-(128 i + r)][d-1-(128 j + c)]
__device__ __forceinline__ gfloat* dag_hinv_at(const DagParams& p, int b, int i, int j, int r, int c) {
  return (gfloat*)p.hinv + (int64_t)b * p.shinv + (p.d - 1 - ((int64_t)i * NB + r)) * p.d +
         (p.d - 1 - ((int64_t)j * NB + c));
}
// hinv's diagonal tile T-1-j from X_jj in LDS (row stride LP, only its lower
// triangle read): reversed in both directions, zeros below the diagonal
__device__ __forceinline__ void dag_hinv_diag(const DagParams& p, int b, int j, const float* x) {
  for (int e = threadIdx.x; e < NB * NB; e += PNT) {
    const int r = e >> 7, cc = e & (NB - 1);
    *dag_hinv_at(p, b, j, j, r, cc) = cc <= r ? x[r * LP + cc] : 0.f;
  }
}
// zeros over hinv tile (i, j) (the lower half of J X J: tile (T-1-j', T-1-i') of X's mirror)
__device__ __forceinline__ void dag_hinv_zero_tile(const DagParams& p, int b, int ti, int tj) {
  typedef __attribute__((address_space(1))) f32x4_t gf4;
  const int tid = threadIdx.x;
  gfloat* base = (gfloat*)p.hinv + (int64_t)b * p.shinv + (int64_t)ti * NB * p.d + (int64_t)tj * NB;
  const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 16; ++i) *reinterpret_cast<gf4*>(base + (8 * i + (tid >> 5)) * p.d + 4 * (tid & 31)) = z;
}

// The chain of matrix b: factor and invert each diagonal tile once it is
// fully updated.
__device__ __noinline__ void dag_chain(DagParams p, int b) {
  const int T = p.T;
  const int64_t d = p.d;
  gint* lf = dag_lf(p, b);
  const gint* nd = lf + 2 * T * T + 5 * T;
  float* a = dag_smem;
  float* x = dag_smem + NB * LP;
  float* t = dag_smem + 2 * NB * LP;
  float* cb = t + 3 * SB * LT;
  f32x4_t v[16];
  for (int j = 0; j < T; ++j) {
    const int r0 = threadIdx.x >> 5, c = 4 * (threadIdx.x & 31);
    // (the first diagonal tile has no update: as prepared)
    if (j >= 1 && !dag_wait(nd + j - 1, 4, p, b)) return;
    dag_fetch(dag_tile(p.F, p, b, j, j), d, v);
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) a[(8 * i + r0) * LP + c + e] = (c + e <= 8 * i + r0) ? v[i][e] : 0.f;
    __syncthreads();
    potf2_inv_lds(a, x, t, cb, dag_tile(p.X, p, b, j, j), d, p.status + b);
    dag_publish(lf + j * T + j, DAG_LF_FINAL);
    if (j == T - 1) dag_hinv_diag(p, b, j, x);  // (strip task S(j, 0) writes the others)
  }
}

// Strip accumulators: wave w holds the 32 x 32 block (strip rows, column
// block w) of A_{c+1,c} (and of the diagonal tile for w <= s), each as two
// MFMA chains (even and odd k) summed at the end.
template <typename Fn>
__device__ __forceinline__ void dag_each_strip(Fn&& fn) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < 16; ++r) fn(r, 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), lane & 31);
}

// One strip-row operand and one or two [n][k] operands from LDS (stride LP),
// k in [0, 2 kk_end): acc0/acc1 += A B0^T, acc2/acc3 += A B1^T (if two).
template <bool TWO>
__device__ __forceinline__ void dag_mma_strip(f32x16_t& s0, f32x16_t& s1, f32x16_t& d0, f32x16_t& d1, const float* pa,
                                              const float* pb0, const float* pb1, int kk_end, float sign) {
  for (int c = 0; c < kk_end; c += 16) {
#pragma unroll
    for (int q = 0; q < 16; q += 2) {
      const int k2 = 2 * (c + q);
      const float a0 = sign * pa[k2], a1 = sign * pa[k2 + 2];
      const float b0 = pb0[k2], b1 = pb0[k2 + 2];
      s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, s1, 0, 0, 0);
      if (TWO) {
        const float e0 = pb1[k2], e1 = pb1[k2 + 2];
        d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, e0, d0, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, e1, d1, 0, 0, 0);
      }
    }
  }
}

__device__ __forceinline__ void dag_fetch_rows(const gfloat* g, int64_t ld, int rows, f32x4_t (&v)[16]) {
  typedef __attribute__((address_space(1))) const f32x4_t gf4;
  const int tid = threadIdx.x;
  const gfloat* p = g + (tid >> 5) * ld + 4 * (tid & 31);
#pragma unroll
  for (int i = 0; i < 16; ++i)
    if (8 * i < rows) v[i] = *reinterpret_cast<gf4*>(p + 8 * i * ld);
}
__device__ __forceinline__ void dag_put_rows(const f32x4_t (&v)[16], int rows, float* l) {
  const int tid = threadIdx.x, r0 = tid >> 5, c = 4 * (tid & 31);
#pragma unroll
  for (int i = 0; i < 16; ++i)
    if (8 * i < rows)
#pragma unroll
      for (int e = 0; e < 4; ++e) l[(8 * i + r0) * LP + c + e] = v[i][e];
}

// S(c, s): strip s (rows 32 s ..) of tile row c + 1.
__device__ __noinline__ void dag_task_s(DagParams p, int b, int c, int s) {
  const int T = p.T;
  const int64_t d = p.d;
  gint* lf = dag_lf(p, b);
  gint* st = lf + 2 * T * T;
  gint* nl = st + 4 * T;
  gint* nd = nl + T;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r0 = 32 * s, r1 = 32 * (s + 1);
  const bool dw = w <= s;  // this wave has a block of the diagonal strip
  float* la = dag_smem;              // rows 0 .. r1 of L_{c+1,k} (the strip's own among them)
  float* lb = dag_smem + NB * LP;    // L_{c,k}, then X_cc
  gfloat* sub = dag_tile(p.F, p, b, c + 1, c) + (int64_t)r0 * d + 32 * w;
  gfloat* dia = dag_tile(p.F, p, b, c + 1, c + 1) + (int64_t)r0 * d + 32 * w;
  f32x16_t s0, s1, d0, d1;
  const int64_t ra = (int64_t)(c + 1) * NB + r0;  // first row of the strip in F
  dag_each_strip([&](int r, int row, int col) {
    s0[r] = dag_orig(p, b, ra + row, (int64_t)c * NB + 32 * w + col);
    s1[r] = 0.f;
    d0[r] = dw ? dag_orig(p, b, ra + row, (int64_t)(c + 1) * NB + 32 * w + col) : 0.f;
    d1[r] = 0.f;
  });
  const float* pa = la + (r0 + (lane & 31)) * LP + (lane >> 5);
  const float* pbs = lb + (32 * w + (lane & 31)) * LP + (lane >> 5);
  const float* pbd = la + (32 * w + (lane & 31)) * LP + (lane >> 5);
  f32x4_t va[16], vb[16];
  auto ready = [&](int k) {
    return dag_wait(lf + (c + 1) * T + k, DAG_LF_FINAL, p, b) && dag_wait(lf + c * T + k, DAG_LF_FINAL, p, b);
  };
  if (c > 0) {
    if (!ready(0)) return;
    dag_fetch_rows(dag_tile(p.F, p, b, c + 1, 0), d, r1, va);
    dag_fetch(dag_tile(p.F, p, b, c, 0), d, vb);
  }
  for (int k = 0; k < c; ++k) {
    dag_put_rows(va, r1, la);
    dag_put_rk(vb, lb);
    __syncthreads();
    if (k + 1 < c) {
      if (!ready(k + 1)) return;
      dag_fetch_rows(dag_tile(p.F, p, b, c + 1, k + 1), d, r1, va);
      dag_fetch(dag_tile(p.F, p, b, c, k + 1), d, vb);
    }
    if (dw)
      dag_mma_strip<true>(s0, s1, d0, d1, pa, pbs, pbd, NB / 2, -1.f);
    else
      dag_mma_strip<false>(s0, s1, d0, d1, pa, pbs, pbd, NB / 2, -1.f);
    __syncthreads();
  }
  // L_{c+1,c}[s] = A_{c+1,c}[s] X_cc^T (X_cc lower: column block w needs k < 32 (w + 1))
  if (!dag_wait(lf + c * T + c, DAG_LF_FINAL, p, b)) return;
  dag_fetch(dag_tile(p.X, p, b, c, c), d, vb);
  dag_put_rk(vb, lb);
  dag_each_strip([&](int r, int row, int col) { la[row * LP + 32 * w + col] = s0[r] + s1[r]; });
  __syncthreads();
  {
    f32x16_t l0, l1, u0, u1;
#pragma unroll
    for (int r = 0; r < 16; ++r) l0[r] = l1[r] = u0[r] = u1[r] = 0.f;
    dag_mma_strip<false>(l0, l1, u0, u1, la + (lane & 31) * LP + (lane >> 5), pbs, pbs, 16 * (w + 1), 1.f);
    dag_each_strip([&](int r, int row, int col) { s0[r] = l0[r] + l1[r]; });
  }
  dag_each_strip([&](int r, int row, int col) { sub[row * d + col] = s0[r]; });
  dag_publish(st + 4 * c + s, 1);
  // A_{c+1,c+1}[s][0..s] -= L[s] L[0..s]^T
  if (s > 0 && !dag_wait(st + 4 * c, 1, p, b, s)) return;
  // (this workgroup read its strip's rows of A_{c+1,c} before storing them
  // as L: drop any cached copy before reading them back)
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  dag_fetch_rows(dag_tile(p.F, p, b, c + 1, c), d, r1, va);
  dag_put_rows(va, r1, la);
  __syncthreads();
  if (dw) {
    dag_mma_strip<false>(d0, d1, s0, s1, pa, pbd, pbd, NB / 2, -1.f);
    dag_each_strip([&](int r, int row, int col) { dia[row * d + col] = d0[r] + d1[r]; });
  }
  dag_stores_done();
  if (threadIdx.x == 0) {
    __hip_atomic_fetch_add(nd + c, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    // off the chain's path from here: L_{c+1,c} complete with its last strip
    if (__hip_atomic_fetch_add(nl + c, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == 3)
      __hip_atomic_store(lf + (c + 1) * T + c, DAG_LF_FINAL, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
  }
  // hinv's diagonal tile for X_cc, still in lb
  if (s == 0) dag_hinv_diag(p, b, c, lb);
}

// H(i, c), i >= c + 2: A_ic -= sum_{k < c} L_ik L_ck^T, then L_ic = A_ic
// X_cc^T.  The tiles of step k + 1 are fetched while step k's MFMAs run.
__device__ __noinline__ void dag_task_h(DagParams p, int b, int i, int c) {
  const int T = p.T;
  const int64_t d = p.d;
  gint* lf = dag_lf(p, b);
  float* la = dag_smem;
  float* lb = dag_smem + NB * LP;
  f32x4_t va[16], vb[16];
  DagAcc acc;
  gfloat* out = dag_tile(p.F, p, b, i, c);
  dag_each([&](int bm, int bn, int r, int row, int col) {
    acc.t[bm][bn][r] = dag_orig(p, b, (int64_t)i * NB + row, (int64_t)c * NB + col);
  });
  auto ready = [&](int k) {
    return dag_wait(lf + i * T + k, DAG_LF_FINAL, p, b) && dag_wait(lf + c * T + k, DAG_LF_FINAL, p, b);
  };
  if (c > 0) {
    if (!ready(0)) return;
    dag_fetch(dag_tile(p.F, p, b, i, 0), d, va);
    dag_fetch(dag_tile(p.F, p, b, c, 0), d, vb);
  }
  for (int k = 0; k < c; ++k) {
    dag_put_rk(va, la);
    dag_put_rk(vb, lb);
    __syncthreads();
    if (k + 1 < c) {
      if (!ready(k + 1)) return;
      dag_fetch(dag_tile(p.F, p, b, i, k + 1), d, va);
      dag_fetch(dag_tile(p.F, p, b, c, k + 1), d, vb);
    }
    dag_mma<false>(acc, la, lb, -1.f);
    __syncthreads();
  }
  if (!dag_wait(lf + c * T + c, DAG_LF_FINAL, p, b)) return;
  dag_fetch(dag_tile(p.X, p, b, c, c), d, vb);
  dag_put_rk(vb, lb);
  dag_each([&](int bm, int bn, int r, int row, int col) { la[row * LP + col] = acc.t[bm][bn][r]; });
  __syncthreads();
  dag_zero(acc);
  dag_mma_tri(acc, la, lb);
  dag_each_tri([&](int bm, int bn, int r, int row, int col) { out[row * d + col] = acc.t[bm][bn][r]; });
  dag_publish(lf + i * T + c, DAG_LF_FINAL);
}

// V(c, j): X_cj = -X_cc sum_{k=j}^{c-1} L_ck X_kj (fetches of step k + 1
// under step k's MFMAs).
__device__ __noinline__ void dag_task_v(DagParams p, int b, int c, int j) {
  const int T = p.T;
  const int64_t d = p.d;
  gint* lf = dag_lf(p, b);
  gint* xf = lf + T * T;
  float* la = dag_smem;
  float* lb = dag_smem + NB * LP;
  f32x4_t va[16], vb[16];
  DagAcc acc;
  dag_zero(acc);
  auto ready = [&](int k) {
    return dag_wait(lf + c * T + k, DAG_LF_FINAL, p, b) &&
           (k == j ? dag_wait(lf + j * T + j, DAG_LF_FINAL, p, b) : dag_wait(xf + k * T + j, 1, p, b));
  };
  if (!ready(j)) return;
  dag_fetch(dag_tile(p.F, p, b, c, j), d, va);
  dag_fetch(dag_tile(p.X, p, b, j, j), d, vb);
  for (int k = j; k < c; ++k) {
    dag_put_rk(va, la);
    dag_put_kn(vb, lb);
    __syncthreads();
    if (k + 1 < c) {
      if (!ready(k + 1)) return;
      dag_fetch(dag_tile(p.F, p, b, c, k + 1), d, va);
      dag_fetch(dag_tile(p.X, p, b, k + 1, j), d, vb);
    }
    dag_mma<true>(acc, la, lb, 1.f);
    __syncthreads();
  }
  if (!dag_wait(lf + c * T + c, DAG_LF_FINAL, p, b)) return;
  dag_fetch(dag_tile(p.X, p, b, c, c), d, va);
  dag_put_rk(va, la);
  dag_each([&](int bm, int bn, int r, int row, int col) { lb[row * DLB + col] = acc.t[bm][bn][r]; });
  __syncthreads();
  dag_zero(acc);
  dag_mma<true>(acc, la, lb, -1.f);
  dag_store_acc(acc, dag_tile(p.X, p, b, c, j), d);
  dag_each([&](int bm, int bn, int r, int row, int col) { *dag_hinv_at(p, b, c, j, row, col) = acc.t[bm][bn][r]; });
  dag_hinv_zero_tile(p, b, T - 1 - j, T - 1 - c);
  dag_publish(xf + c * T + j, 1);
}

// task index -> kind (0 chain, 1 H, 2 V, 3 S), matrix b, (i, j).  Order:
// chains 0..B-1, then per level c = 0, 1, ... the matrices 0..B-1 in turn,
// each with level 0: H(2.., 0) (T - 2 tasks); level c >= 1: S(c-1, 0..3),
// H(c+2.., c), V(c, 0..c-1) (T + 2 tasks, T + 3 on the last level).
__device__ __forceinline__ void dag_decode(int idx, int T, int B, int& kind, int& b, int& i, int& j) {
  if (idx < B) {
    kind = 0;
    b = idx;
    i = j = 0;
    return;
  }
  int r = idx - B;
  if (r < B * (T - 2)) {
    kind = 1;
    b = r / (T - 2);
    i = 2 + r % (T - 2);
    j = 0;
    return;
  }
  r -= B * (T - 2);
  int c, nc;
  if (r < B * (T + 2) * (T - 2)) {
    c = 1 + r / (B * (T + 2));
    r %= B * (T + 2);
    nc = T + 2;
  } else {
    r -= B * (T + 2) * (T - 2);
    c = T - 1;
    nc = T + 3;
  }
  b = r / nc;
  int u = r % nc;
  if (u < 4) {
    kind = 3;
    i = c - 1;
    j = u;
    return;
  }
  u -= 4;
  const int nh = T - c - 2 > 0 ? T - c - 2 : 0;
  if (u < nh) {
    kind = 1;
    i = c + 2 + u;
    j = c;
  } else {
    kind = 2;
    i = c;
    j = u - nh;
  }
}

__global__ __launch_bounds__(PNT, 1) void chol_dag_kernel(DagParams p) {
  int32_t* ctl = p.flags + dag_nflags(p.T) - 2;
  for (;;) {
    if (threadIdx.x == 0) {
      const bool aborted = __hip_atomic_load(ctl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
      dag_word = aborted ? p.ntasks : __hip_atomic_fetch_add(ctl, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    const int task = dag_word;
    __syncthreads();
    if (task >= p.ntasks) break;
    int kind, b, i, j;
    dag_decode(task, p.T, p.batch, kind, b, i, j);
    if (kind == 0)
      dag_chain(p, b);
    else if (kind == 1)
      dag_task_h(p, b, i, j);
    else if (kind == 2)
      dag_task_v(p, b, i, j);
    else
      dag_task_s(p, b, i, j);
  }
}

// diag'[j] = H[p(j)][p(j)] / n with 0 -> 1 (dead), damp = percdamp * mean(diag')
// (one workgroup per matrix of a batch)
// (also clears the matrix's nflags dataflow flags, flags + bm wsf, when set)
__global__ __launch_bounds__(1024) void diag_damp_kernel(const float* H, int64_t ldh, int64_t sh, int64_t d,
                                                         const int32_t* perm, int64_t sp, const float* ns_arr,
                                                         float ns0, float percdamp, int32_t* dead,
                                                         float* damp_out, int64_t wsf, int32_t* status,
                                                         int32_t* flags, int nflags) {
  __shared__ float part[1024 / 64];
  const int64_t bm = blockIdx.x;
  if (flags)
    for (int e = threadIdx.x; e < nflags; e += 1024) flags[bm * wsf + e] = 0;
  H += bm * sh;
  if (perm) perm += bm * sp;
  if (dead) dead += bm * d;
  damp_out += bm * wsf;
  if (status) status += bm;
  const float num_samples = ns_arr ? ns_arr[bm] : ns0;
  float s = 0.f;
  for (int64_t j = threadIdx.x; j < d; j += 1024) {
    const int64_t pj = perm ? perm[j] : j;
    float v = H[pj * ldh + pj] / num_samples;
    const bool dd = v == 0.f;
    if (dead) dead[j] = dd ? 1 : 0;
    s += dd ? 1.f : v;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.f;
    for (int w = 0; w < 1024 / 64; ++w) t += part[w];
    damp_out[0] = percdamp * (t / (float)d);
    if (status) *status = 0;
  }
}

// F (lower) = flip(permute(H / n)) with dead / damping rules on the diagonal.
__global__ void prepare_flip_kernel(const float* H, int64_t ldh, int64_t sh, int64_t d, const int32_t* perm,
                                    int64_t sp, const float* ns_arr, float ns0, const float* damp, float* F,
                                    int64_t wsf, int vec) {
  const int64_t bm = blockIdx.z;
  H += bm * sh;
  if (perm) perm += bm * sp;
  damp += bm * wsf;
  F += bm * wsf;
  const float num_samples = ns_arr ? ns_arr[bm] : ns0;
  const int64_t a = (int64_t)blockIdx.y * 16 + threadIdx.y;
  if (vec) {
    // (no permutation, d, ldh and the batch stride multiples of 4, H 16-byte
    // aligned: checked on the host, which sizes the grid for it) four columns
    // per thread: F[a][b4 + e] = H[d-1-a][d-1-b4-e], one 16-byte load of H's
    // row read backwards and one 16-byte store (zeros above the diagonal,
    // which nothing reads: four 4-byte stores per thread ran at 2.4 TB/s)
    const int64_t b4 = ((int64_t)blockIdx.x * 64 + threadIdx.x) * 4;
    if (a >= d || b4 > a) return;
    const int64_t ia = d - 1 - a;
    const f32x4_t h = *reinterpret_cast<const f32x4_t*>(H + ia * ldh + d - 4 - b4);
    f32x4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t b = b4 + e;
      float v = h[3 - e] / num_samples;
      if (a == b) {
        if (v == 0.f) v = 1.f;
        v = v + damp[0];
      }
      o[e] = b <= a ? v : 0.f;
    }
    *reinterpret_cast<f32x4_t*>(F + a * d + b4) = o;
    return;
  }
  const int64_t b = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (a >= d || b > a) return;
  const int64_t ia = d - 1 - a, ib = d - 1 - b;
  const int64_t pa = perm ? perm[ia] : ia, pb = perm ? perm[ib] : ib;
  const int64_t r = pa < pb ? pa : pb, c = pa < pb ? pb : pa;
  float v = H[r * ldh + c] / num_samples;
  if (a == b) {
    if (v == 0.f) v = 1.f;
    v = v + damp[0];
  }
  F[a * d + b] = v;
}

// hinv[a][b] = X[d-1-a][d-1-b] (a <= b), zero below the diagonal.
__global__ void flip_out_kernel(const float* X, int64_t d, float* hinv, int64_t wsf, int64_t shinv, int vec) {
  X += (int64_t)blockIdx.z * wsf;
  hinv += (int64_t)blockIdx.z * shinv;
  const int64_t a = (int64_t)blockIdx.y * 16 + threadIdx.y;
  if (vec) {
    // (d and shinv multiples of 4, hinv 16-byte aligned: checked on the host)
    // four columns per thread: one 16-byte load of X's row read backwards,
    // one 16-byte store (the load is skipped where all four are below)
    const int64_t b4 = ((int64_t)blockIdx.x * 64 + threadIdx.x) * 4;
    if (a >= d || b4 >= d) return;
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
    if (b4 + 3 >= a) {
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(X + (d - 1 - a) * d + d - 4 - b4);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (a <= b4 + e) ? x[3 - e] : 0.f;
    }
    *reinterpret_cast<f32x4_t*>(hinv + a * d + b4) = o;
    return;
  }
  const int64_t b = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (a >= d || b >= d) return;
  hinv[a * d + b] = (a <= b) ? X[(d - 1 - a) * d + (d - 1 - b)] : 0.f;
}

// dst[r][c] = src[r][c] for r < rows, c < cols (cols % 4 == 0, 16-byte
// aligned rows): a strided panel into a compact buffer (matrix blockIdx.y
// at src + y wsf, dst + y wsf)
__global__ void copy_panel_kernel(const float* src, int64_t lds_, float* dst, int64_t ldd, int64_t rows,
                                  int64_t cols, int64_t wsf) {
  src += (int64_t)blockIdx.y * wsf;
  dst += (int64_t)blockIdx.y * wsf;
  const int64_t q = cols / 4, n = rows * q;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / q, c = 4 * (i % q);
    *reinterpret_cast<f32x4_t*>(dst + r * ldd + c) = *reinterpret_cast<const f32x4_t*>(src + r * lds_ + c);
  }
}

// Place diagonal-block inverses into X.
__global__ void place_diag_inv_kernel(const float* linv, int64_t d, float* X, int64_t wsf) {
  linv += (int64_t)blockIdx.y * wsf;
  X += (int64_t)blockIdx.y * wsf;
  const int blk = blockIdx.x;
  const int64_t k0 = (int64_t)blk * NB;
  for (int e = threadIdx.x; e < NB * NB; e += blockDim.x) {
    const int i = e / NB, j = e % NB;
    if (k0 + i < d && k0 + j < d) X[(k0 + i) * d + (k0 + j)] = linv[(int64_t)blk * NB * NB + e];
    // zeros in the block right of it: the 256-row tiles of a lower-triangular
    // operand read that far above the diagonal
    if (k0 + i < d && k0 + NB + j < d) X[(k0 + i) * d + (k0 + NB + j)] = 0.f;
  }
}

// hinv of matrix b = identity where status[b] != 0 (blockIdx.y = b); every
// thread reads the flag, so a positive-definite matrix costs one load
__global__ void identity_on_failure_kernel(float* hinv, int64_t d, int64_t stride, const int32_t* status) {
  const int64_t b = blockIdx.y;
  if (status[b] == 0) return;
  float* h = hinv + b * stride;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < d * d; i += (int64_t)gridDim.x * blockDim.x)
    h[i] = (i / d == i % d) ? 1.f : 0.f;
}

inline size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct HinvLayout {
  size_t F, X, T, linv, damp, flags, total;
};

HinvLayout hinv_layout(int64_t d) {
  HinvLayout L{};
  size_t off = 0;
  const int64_t nblk = (d + NB - 1) / NB;
  L.F = off; off = align256(off + (size_t)d * d * sizeof(float));
  L.X = off; off = align256(off + (size_t)d * d * sizeof(float));
  L.T = off; off = align256(off + (size_t)(d * ((d + 1) / 2 + NB)) * sizeof(float));
  L.linv = off; off = align256(off + (size_t)nblk * NB * NB * sizeof(float));
  L.damp = off; off = align256(off + 64);
  // dataflow factorisation: 2 T^2 tile flags, then (matrix 0) the task counter and abort word
  L.flags = off; off = align256(off + (size_t)dag_nflags(nblk) * sizeof(int32_t));
  L.total = off;
  return L;
}

}  // namespace

// Compute units of the current device (256 on an MI355X).
int64_t gemm_cus() {
  int dev = 0, ncu = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) !=
      hipSuccess || ncu <= 0)
    return 256;
  return ncu;
}

// The x6 products, unless MI355Q_GEMM_X6=0 (every product then on the fp32 MFMA).
bool x6_enabled() {
  static const bool on = [] {
    const char* e = getenv("MI355Q_GEMM_X6");
    return !(e && e[0] == '0');
  }();
  return on;
}

int gemm_f32(const GemmArgs& g, bool b_trans, int batch, hipStream_t stream) {
  if (g.M <= 0 || g.N <= 0 || batch <= 0) return MI355Q_OK;
  if (g.in_place) {
    // one workgroup per row tile: the whole-row K = 128 kernel, else the
    // general kernel (N <= GBN: a single column tile)
    MQ_CHECK_ARG(b_trans && !g.a_trans && !g.upper_only && !g.lower_only && !g.a_lower && !g.b_lower &&
                     g.N <= GBN && batch <= 65535,
                 "gemm: an in-place product takes B transposed, N <= %d and no triangular options", GBN);
    const bool strides16 = g.strideA % 4 == 0 && g.strideB % 4 == 0 && g.strideA2 % 4 == 0 && g.strideB2 % 4 == 0;
    if (g.K == KT && g.N == KT && g.M % RT == 0 && g.M / RT <= 65535 && g.lda % 4 == 0 && g.ldb % 4 == 0 &&
        aligned16(g.A) && aligned16(g.B) && (batch == 1 || strides16) && (g.lda * 7 + KT) < (1 << 29) &&
        (g.ldb * 7 + KT) < (1 << 29) && (g.ldc * 31 + KT) < (1 << 29)) {
      // one workgroup per CU, the matrices' row tiles shared out among them
      const int64_t per = (gemm_cus() + batch - 1) / batch;
      hipLaunchKernelGGL(gemm_k128_rows_kernel, dim3(1, (unsigned)(g.M / RT < per ? g.M / RT : per), (unsigned)batch),
                         dim3(GNT), 0, stream, g);
    } else {
      hipLaunchKernelGGL((gemm_f32_kernel<true, false>), dim3(1, (unsigned)((g.M + GBM - 1) / GBM), (unsigned)batch),
                         dim3(GNT), 0, stream, g);
    }
    MQ_LAUNCH_CHECK();
    return MI355Q_OK;
  }
  if (g.a_trans || g.upper_only) {   // the general kernel only
    MQ_CHECK_ARG(batch <= 65535 && !g.a_lower && !g.b_lower && !g.lower_only,
                 "gemm: transposed-A / upper-only products take no triangular options");
    dim3 grid((unsigned)((g.N + GBN - 1) / GBN), (unsigned)((g.M + GBM - 1) / GBM), (unsigned)batch);
    if (!g.a_trans && b_trans)
      hipLaunchKernelGGL((gemm_f32_kernel<true, false>), grid, dim3(GNT), 0, stream, g);
    else if (!g.a_trans)
      hipLaunchKernelGGL((gemm_f32_kernel<false, false>), grid, dim3(GNT), 0, stream, g);
    else if (b_trans)
      hipLaunchKernelGGL((gemm_f32_kernel<true, true>), grid, dim3(GNT), 0, stream, g);
    else
      hipLaunchKernelGGL((gemm_f32_kernel<false, true>), grid, dim3(GNT), 0, stream, g);
    MQ_LAUNCH_CHECK();
    return MI355Q_OK;
  }
  // K >= 256: the LDS-DMA kernel with a two-stage ring (two or three
  // workgroups per CU).  Tile shapes as measured best on the solve's
  // products: plain products 128 x 128 on eight waves when one product
  // fills the CUs at least once (117 TFLOP/s on 4096 x 3072 x 1024, against
  // 98 for 64 x 128), else 64 x 128 (also for batches: the MoE experts' solves
  // ran 6 % slower on the larger tile); 64 x 64 with a triangular operand;
  // lower-only products 64 x 64 up to 4096 rows (the rank-512 Cholesky
  // updates of 512 .. 3584 rows: within 5 % of the best of six shapes at
  // every size), 128 x 64 above, and for batches above 2048 rows in total.
  const bool v16 = g.K % 4 == 0 && g.lda % 4 == 0 && g.ldb % 4 == 0 && aligned16(g.A) && aligned16(g.B) &&
                   (b_trans || g.N % 4 == 0) && g.strideA % 4 == 0 && g.strideB % 4 == 0 && g.strideA2 % 4 == 0 &&
                   g.strideB2 % 4 == 0;
  if ((g.K >= 256 || (g.K >= 128 && g.x6 == 2)) && v16 && batch <= 65535 &&
      ((g.M + 63) / 64) * ((g.N + 63) / 64) < (1ll << 31) && g.x6 && x6_enabled() &&
      g.lda < (1 << 20) && g.ldb < (1 << 20)) {   // 32-bit offsets within a tile
    // fp32-accurate bf16 products
#define MQ_X6(TM, TN, WM, WN)                                                                                  \
  do {                                                                                                         \
    dim3 grid((unsigned)(((g.N + TN - 1) / TN) * ((g.M + TM - 1) / TM)), 1, (unsigned)batch);                  \
    if (b_trans)                                                                                               \
      hipLaunchKernelGGL((gemm_x6_kernel<TM, TN, WM, WN, true>), grid, dim3(64 * WM * WN), 0, stream, g);      \
    else                                                                                                       \
      hipLaunchKernelGGL((gemm_x6_kernel<TM, TN, WM, WN, false>), grid, dim3(64 * WM * WN), 0, stream, g);     \
  } while (0)
    // Which tile, by how many of them a CU gets (those of a lower-only product
    // above the diagonal exit at once, so half count).  4096 rows, K = 1024, by
    // N, in us (256 x 128 | 128 x 128 | 64 x 128):
    //   N = 1024   79 |  68 |  59   one 128 x 128 tile a CU has nothing beside it
    //   N = 2048   83 |  92 | 114   one round of wide tiles, full
    //   N = 3072  159 | 131 | 173   two rounds of wide tiles, the second half empty
    // and 64 products of 768 x 1536, K = 512, 446 | 402 | 565: over many rounds
    // the clock sinks to what the chip's power allows (1.5 GHz over 0.8 ms), and
    // the tiles two to a CU, whose rounds do not all end at once, come out
    // ahead.  192 .. 204 TFLOP/s are 1150 .. 1230 on the bf16 MFMA, the rate of
    // a large library product here.  Triangular operands: a wide tile's K range
    // is the coarser one.
    const int64_t cus = gemm_cus(), half = g.lower_only ? 2 : 1;
    const int64_t t256 = ((g.M + 255) / 256) * ((g.N + 127) / 128) * batch / half;
    const int64_t t128 = ((g.M + 127) / 128) * ((g.N + 127) / 128) * batch / half;
    if (!g.a_lower && !g.b_lower && t256 <= cus && 10 * t256 >= 7 * cus)
      MQ_X6(256, 128, 4, 2);
    else if (2 * t128 >= 3 * cus)
      MQ_X6(128, 128, 2, 2);
    else
      MQ_X6(64, 128, 2, 2);
#undef MQ_X6
    MQ_LAUNCH_CHECK();
    return MI355Q_OK;
  }
  if (g.K >= 256 && v16 && batch <= 65535 && ((g.M + 63) / 64) * ((g.N + 63) / 64) < (1ll << 31)) {
#define MQ_DMA(TM, TN, WM, WN)                                                                             \
  do {                                                                                                     \
    dim3 grid((unsigned)(((g.N + TN - 1) / TN) * ((g.M + TM - 1) / TM)), 1, (unsigned)batch);              \
    if (b_trans)                                                                                           \
      hipLaunchKernelGGL((gemm_dma_kernel<TM, TN, WM, WN, true, 2>), grid, dim3(64 * WM * WN), 0, stream, g); \
    else                                                                                                   \
      hipLaunchKernelGGL((gemm_dma_kernel<TM, TN, WM, WN, false, 2>), grid, dim3(64 * WM * WN), 0, stream, g); \
  } while (0)
    if (g.a_lower || g.b_lower) {
      MQ_DMA(64, 64, 2, 2);        // uneven K ranges: small tiles, the longest dispatched first
    } else if (!g.lower_only) {
      if (batch == 1 && ((g.M + 127) / 128) * ((g.N + 127) / 128) >= 256)
        MQ_DMA(128, 128, 2, 4);
      else
        MQ_DMA(64, 128, 2, 2);
    } else if (g.M * batch > (batch > 1 ? 2048 : 4096)) {
      MQ_DMA(128, 64, 2, 2);
    } else {
      MQ_DMA(64, 64, 2, 2);
    }
#undef MQ_DMA
    MQ_LAUNCH_CHECK();
    return MI355Q_OK;
  }
  // large-K lower-only products: K = 128 slices on the whole-tile kernel
  if (g.lower_only && g.K > KT && g.K % KT == 0 && g.M % KT == 0 && g.N % KT == 0) {
    GemmArgs s = g;
    s.K = KT;
    for (int64_t k0 = 0; k0 < g.K; k0 += KT) {
      s.A = g.A + k0;
      s.B = b_trans ? g.B + k0 : g.B + k0 * g.ldb;
      s.beta = k0 == 0 ? g.beta : 1.f;
      const int rc = gemm_f32(s, b_trans, batch, stream);
      if (rc) return rc;
    }
    return MI355Q_OK;
  }
  MQ_CHECK_ARG(batch <= 65535, "gemm: batch too large");
  // whole-tile K = 128 products (every batch member 16-byte aligned)
  const bool strides16 = g.strideA % 4 == 0 && g.strideB % 4 == 0 && g.strideA2 % 4 == 0 && g.strideB2 % 4 == 0;
  const bool k128 = !g.a_lower && !g.b_lower && g.K == KT && g.M % KT == 0 && g.N % KT == 0 && g.lda % 4 == 0 && g.ldb % 4 == 0 &&
                    aligned16(g.A) && aligned16(g.B) && (batch == 1 || strides16) &&
                    (g.lda * 7 + KT) < (1 << 29) && (g.ldb * 7 + KT) < (1 << 29) && (g.ldc * 127 + KT) < (1 << 29);
  // the same products in 64 x 64 tiles when 128 x 128 tiles would leave
  // most CUs idle (fewer than two tiles per CU)
  const bool k128s = !g.a_lower && !g.b_lower && g.K == KT && g.M % ST == 0 && g.N % ST == 0 && g.lda % 4 == 0 &&
                     g.ldb % 4 == 0 && aligned16(g.A) && aligned16(g.B) && (batch == 1 || strides16) &&
                     (g.lda * 63 + KT) < (1 << 29) && (g.ldb * 127 + KT) < (1 << 29) && (g.ldc * 63 + ST) < (1 << 29) &&
                     g.M / ST <= 65535 && g.N / ST <= 65535;
  const int64_t big_tiles = (g.M / KT) * (g.N / KT) * batch / (g.lower_only ? 2 : 1);
  if (k128s && (!k128 || big_tiles < 512)) {
    dim3 grid((unsigned)(g.N / ST), (unsigned)(g.M / ST), (unsigned)batch);
    if (b_trans)
      hipLaunchKernelGGL(gemm_k128_small_kernel<true>, grid, dim3(GNT), 0, stream, g);
    else
      hipLaunchKernelGGL(gemm_k128_small_kernel<false>, grid, dim3(GNT), 0, stream, g);
    MQ_LAUNCH_CHECK();
    return MI355Q_OK;
  }
  if (k128) {
    // one workgroup per CU: spread the column tiles so ~256 workgroups run
    const int64_t mt = g.M / KT, ntl = g.N / KT;
    int64_t p = (256 + mt * batch - 1) / (mt * batch);
    if (p > ntl) p = ntl;
    if (p < 1) p = 1;
    dim3 grid((unsigned)p, (unsigned)mt, (unsigned)batch);
    if (b_trans)
      hipLaunchKernelGGL(gemm_k128_kernel<true>, grid, dim3(GNT), 0, stream, g);
    else
      hipLaunchKernelGGL(gemm_k128_kernel<false>, grid, dim3(GNT), 0, stream, g);
    MQ_LAUNCH_CHECK();
    return MI355Q_OK;
  }
  dim3 grid((unsigned)((g.N + GBN - 1) / GBN), (unsigned)((g.M + GBM - 1) / GBM), (unsigned)batch);
  if (b_trans)
    hipLaunchKernelGGL(gemm_f32_kernel<true>, grid, dim3(GNT), 0, stream, g);
  else
    hipLaunchKernelGGL(gemm_f32_kernel<false>, grid, dim3(GNT), 0, stream, g);
  MQ_LAUNCH_CHECK();
  return MI355Q_OK;
}

int syrk_f32_upper(const float* x, int64_t n, int64_t d, int64_t ldx, float* h, int64_t ldh, float alpha,
                   float beta, hipStream_t stream, const int* only_if) {
  GemmArgs g{};
  g.only_if = only_if;
  g.A = x; g.lda = ldx; g.a_trans = 1;
  g.B = x; g.ldb = ldx;
  g.C = h; g.ldc = ldh;
  g.M = d; g.N = d; g.K = n;
  g.alpha = alpha; g.beta = beta; g.upper_only = 1;
  return gemm_f32(g, false, 1, stream);
}

}  // namespace mi355q

using namespace mi355q;

extern "C" size_t mi355q_gptq_hinv_workspace_size(int64_t d) { return d > 0 ? hinv_layout(d).total : 0; }

namespace mi355q {
namespace {

// The dataflow factorisation takes orders that are multiples of NB with at
// least 4 and at most 64 blocks, in batches of at most 8 (measured on
// MI355X: 4096 1.45 ms against the blocked chain's 1.85, 8192 5.9 against
// 6.4, but 14336 27.7 against 23.9 - the helpers' single-workgroup tile
// products lose to the chain's large GEMMs - and 2048 x 16 2.55 against
// 2.20: one chain workgroup per matrix).  MI355Q_HINV_DAG=0 in the
// environment turns it off.
bool dag_eligible(int64_t d, int64_t batch) {
  if (d % NB != 0 || d / NB < 4 || d / NB > 64 || batch > 8) return false;
  const char* e = getenv("MI355Q_HINV_DAG");
  return !(e && e[0] == '0');
}

// The hinv pipeline for `batch` matrices of order d: matrix b reads
// H + b sh (and perm + b sp), writes hinv + b shinv, dead + b d, status[b],
// and uses workspace bytes [b L.total, (b + 1) L.total).
int hinv_impl(const float* h_dev, int64_t ldh, int64_t sh, int64_t d, int64_t batch, const int32_t* perm_dev,
              int64_t sp, const float* ns_dev, float ns0, float percdamp, float* hinv_dev, int64_t shinv,
              int32_t* dead_dev, int32_t* status_dev, char* ws, hipStream_t st) {
  const HinvLayout L = hinv_layout(d);
  const int64_t wsf = (int64_t)(L.total / sizeof(float));
  float* F = reinterpret_cast<float*>(ws + L.F);
  float* X = reinterpret_cast<float*>(ws + L.X);
  float* T = reinterpret_cast<float*>(ws + L.T);
  const int64_t tfloats = (int64_t)((L.linv - L.T) / sizeof(float));
  float* linv = reinterpret_cast<float*>(ws + L.linv);
  float* damp = reinterpret_cast<float*>(ws + L.damp);
  const unsigned nb_ = (unsigned)batch;
  const int64_t nblk = (d + NB - 1) / NB;
  const bool dag = dag_eligible(d, batch);
  int32_t* flags = reinterpret_cast<int32_t*>(ws + L.flags);

  hipLaunchKernelGGL(diag_damp_kernel, dim3(nb_), dim3(1024), 0, st, h_dev, ldh, sh, d, perm_dev, sp, ns_dev, ns0,
                     percdamp, dead_dev, damp, wsf, status_dev, dag ? flags : nullptr, (int)dag_nflags(nblk));
  MQ_LAUNCH_CHECK();
  // 64 x 16 threads; the vectorised paths take four columns per thread, so a
  // block row covers 256 columns instead of 64
  const bool vin = !perm_dev && (d & 3) == 0 && (ldh & 3) == 0 && (nb_ == 1 || (sh & 3) == 0) && aligned16(h_dev) &&
                   aligned16(F);
  const bool vout = (d & 3) == 0 && (nb_ == 1 || (shinv & 3) == 0) && aligned16(hinv_dev);
  auto grid_for = [&](bool vec) {
    const int64_t cpb = vec ? 256 : 64;
    return dim3((unsigned)((d + cpb - 1) / cpb), (unsigned)((d + 15) / 16), nb_);
  };
  const dim3 fb(64, 16);
  hipLaunchKernelGGL(prepare_flip_kernel, grid_for(vin), fb, 0, st, h_dev, ldh, sh, d, perm_dev, sp, ns_dev, ns0,
                     damp, F, wsf, vin ? 1 : 0);
  MQ_LAUNCH_CHECK();
  if (dag) {
    DagParams p{};
    p.F = F; p.X = X; p.flags = flags; p.status = status_dev;
    p.d = d; p.wsf = wsf; p.T = (int)nblk; p.batch = (int)batch;
    p.hinv = hinv_dev; p.shinv = shinv;
    p.ntasks = (int)(batch * (nblk * nblk + 2 * nblk - 2));
    int dev = 0, ncu = 0, khz = 0;
    MQ_CHECK_HIP(hipGetDevice(&dev));
    MQ_CHECK_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    MQ_CHECK_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    // 2 s per wait; MI355Q_HINV_DAG_TIMEOUT_US overrides it (the tests force
    // the time-out path with a tiny value)
    uint64_t us = 2000000;
    if (const char* e = getenv("MI355Q_HINV_DAG_TIMEOUT_US")) us = strtoull(e, nullptr, 10);
    p.timeout = (uint64_t)(khz > 0 ? khz : 100000) * us / 1000ull;
    const int grid = p.ntasks < ncu ? p.ntasks : ncu;
    MQ_CHECK_ARG(grid > batch, "gptq_hinv: %d compute units leave no helper for %d chains", ncu, (int)batch);
    hipLaunchKernelGGL(chol_dag_kernel, dim3((unsigned)grid), dim3(PNT), 0, st, p);
    MQ_LAUNCH_CHECK();
    return MI355Q_OK;
  }

  // blocked right-looking Cholesky on F (lower), two levels: inside an outer
  // panel of OUTB blocks each 128-column block updates only the panel's
  // remaining columns (K = 128); the trailing matrix past the panel takes
  // one rank-(OUTB * 128) lower-only update (K up to 512)
  constexpr int64_t OUTB = 4;
  for (int64_t ob = 0; ob < nblk; ob += OUTB) {
    const int64_t oe = ob + OUTB < nblk ? ob + OUTB : nblk;
    const int64_t c0 = ob * NB, c_end = oe * NB < d ? oe * NB : d;
    for (int64_t kb = ob; kb < oe; ++kb) {
      const int64_t k0 = kb * NB;
      const int nb = (int)((d - k0) < NB ? (d - k0) : NB);
      hipLaunchKernelGGL(potf2_inv_kernel, dim3(nb_), dim3(PNT), 0, st, F, d, k0, nb, linv + kb * NB * NB,
                         status_dev, wsf);
      MQ_LAUNCH_CHECK();
      const int64_t rest = d - k0 - nb;
      if (rest <= 0) break;
      // panel: F[k0+nb:, k0:k0+nb] = F[...] * linv^T (in place, one workgroup per row tile)
      GemmArgs p{};
      p.A = F + (k0 + nb) * d + k0; p.lda = d; p.strideA = wsf;
      p.B = linv + kb * NB * NB; p.ldb = NB; p.strideB = wsf;
      p.C = F + (k0 + nb) * d + k0; p.ldc = d; p.strideC = wsf;
      p.M = rest; p.N = nb; p.K = nb; p.alpha = 1.f; p.beta = 0.f; p.in_place = 1;
      int rc = gemm_f32(p, true, (int)batch, st);
      if (rc) return rc;
      // inside the outer panel: F[k0+nb:, k0+nb:c_end] -= P P[:c_end-k0-nb]^T (lower)
      const int64_t nin = c_end - (k0 + nb);
      if (nin > 0) {
        GemmArgs s{};
        s.A = F + (k0 + nb) * d + k0; s.lda = d; s.strideA = wsf;
        s.B = F + (k0 + nb) * d + k0; s.ldb = d; s.strideB = wsf;
        s.C = F + (k0 + nb) * d + (k0 + nb); s.ldc = d; s.strideC = wsf;
        s.M = rest; s.N = nin; s.K = nb; s.alpha = -1.f; s.beta = 1.f; s.lower_only = 1;
        s.x6 = 2;
        rc = gemm_f32(s, true, (int)batch, st);
        if (rc) return rc;
      }
    }
    // past the outer panel: F[c_end:, c_end:] -= P P^T (lower), P = F[c_end:, c0:c_end],
    // one lower-only product (K up to OUTB * 128).  P is first copied into a
    // compact buffer (the doubling scratch T, unused until the inverse): its
    // rows d floats apart read markedly slower than rows kk floats apart.
    const int64_t rest2 = d - c_end, kk = c_end - c0;
    if (rest2 > 0) {
      const float* P = F + c_end * d + c0;
      int64_t ldp = d;
      if (rest2 * kk <= tfloats && kk % 4 == 0 && d % 4 == 0) {
        const int64_t n4 = rest2 * kk / 4;
        hipLaunchKernelGGL(copy_panel_kernel, dim3((unsigned)((n4 + 255) / 256 < 4096 ? (n4 + 255) / 256 : 4096), nb_),
                           dim3(256), 0, st, P, d, T, kk, rest2, kk, wsf);
        MQ_LAUNCH_CHECK();
        P = T;
        ldp = kk;
      }
      GemmArgs s{};
      s.A = P; s.lda = ldp; s.strideA = wsf;
      s.B = P; s.ldb = ldp; s.strideB = wsf;
      s.C = F + c_end * d + c_end; s.ldc = d; s.strideC = wsf;
      s.M = rest2; s.N = rest2; s.K = kk; s.alpha = -1.f; s.beta = 1.f; s.lower_only = 1;
      s.x6 = 1;
      int rc = gemm_f32(s, true, (int)batch, st);
      if (rc) return rc;
    }
  }

  // triangular inverse X = L^-1 by recursive doubling over NB blocks.  X is
  // not cleared: each product's tiles read a triangular operand only over
  // the K range where it can be nonzero, i.e. besides its lower blocks only
  // the diagonal NB blocks (placed whole, zeros above their diagonal), never
  // the unwritten part above them, and flip_out_kernel reads only X's lower
  // triangle (clearing it took 0.34 ms per 128 batched d = 2048 chains)
  hipLaunchKernelGGL(place_diag_inv_kernel, dim3((unsigned)nblk, nb_), dim3(256), 0, st, linv, d, X, wsf);
  MQ_LAUNCH_CHECK();
  for (int64_t s = NB; s < d; s *= 2) {
    // pairs (a0 = p*2s, c0 = a0 + s); full pairs batched, ragged tail alone
    const int64_t full = d / (2 * s);
    const int64_t tail_c0 = full * 2 * s + s;
    for (int pass = 0; pass < 2; ++pass) {
      int64_t npairs, a0, s2;
      if (pass == 0) {
        npairs = full; a0 = 0; s2 = s;
      } else {
        if (tail_c0 >= d) break;
        npairs = 1; a0 = full * 2 * s; s2 = d - tail_c0;
      }
      if (npairs == 0) continue;
      const int64_t c0 = a0 + s;
      const int64_t stride_diag = 2 * s * (d + 1);
      // each tile of the two products runs only the K range where its
      // triangular operand can be nonzero.
      // T = L[c0:c0+s2, a0:a0+s] * X[a0:a0+s, a0:a0+s] (X11 lower triangular)
      GemmArgs t1{};
      t1.A = F + c0 * d + a0; t1.lda = d; t1.strideA = stride_diag; t1.strideA2 = wsf;
      t1.B = X + a0 * d + a0; t1.ldb = d; t1.strideB = stride_diag; t1.strideB2 = wsf;
      t1.C = T; t1.ldc = s; t1.strideC = s2 * s; t1.strideC2 = wsf;
      t1.inner = npairs; t1.b_lower = 1;
      t1.M = s2; t1.N = s; t1.K = s; t1.alpha = 1.f; t1.beta = 0.f;
      t1.x6 = 1;
      int rc = gemm_f32(t1, false, (int)(npairs * batch), st);
      if (rc) return rc;
      // X[c0:c0+s2, a0:a0+s] = -X[c0:c0+s2, c0:c0+s2] * T (X22 lower triangular)
      GemmArgs t2{};
      t2.A = X + c0 * d + c0; t2.lda = d; t2.strideA = stride_diag; t2.strideA2 = wsf;
      t2.B = T; t2.ldb = s; t2.strideB = s2 * s; t2.strideB2 = wsf;
      t2.C = X + c0 * d + a0; t2.ldc = d; t2.strideC = stride_diag; t2.strideC2 = wsf;
      t2.inner = npairs; t2.a_lower = 1;
      t2.M = s2; t2.N = s; t2.K = s2; t2.alpha = -1.f; t2.beta = 0.f;
      t2.x6 = 1;
      rc = gemm_f32(t2, false, (int)(npairs * batch), st);
      if (rc) return rc;
    }
  }
  hipLaunchKernelGGL(flip_out_kernel, grid_for(vout), fb, 0, st, X, d, hinv_dev, wsf, shinv, vout ? 1 : 0);
  MQ_LAUNCH_CHECK();
  return MI355Q_OK;
}

}  // namespace
}  // namespace mi355q

extern "C" int mi355q_gptq_hinv(const float* h_dev, int64_t ldh, int64_t d, const int32_t* perm_dev,
                                float num_samples, float percdamp, float* hinv_dev, int32_t* dead_dev,
                                int32_t* status_dev, void* workspace_dev, size_t workspace_bytes,
                                void* stream) {
  MQ_CHECK_ARG(h_dev && hinv_dev && status_dev, "gptq_hinv: null pointer");
  MQ_CHECK_ARG(d > 0 && ldh >= d, "gptq_hinv: bad shape");
  MQ_CHECK_ARG(num_samples > 0.f, "gptq_hinv: num_samples must be positive");
  const HinvLayout L = hinv_layout(d);
  MQ_CHECK_ARG(workspace_dev && workspace_bytes >= L.total, "gptq_hinv: workspace too small (%zu < %zu)",
               workspace_bytes, L.total);
  return hinv_impl(h_dev, ldh, 0, d, 1, perm_dev, 0, nullptr, num_samples, percdamp, hinv_dev, 0, dead_dev,
                   status_dev, static_cast<char*>(workspace_dev), reinterpret_cast<hipStream_t>(stream));
}

extern "C" int mi355q_gptq_hinv_batched(const float* h_dev, int64_t ldh, int64_t stride_h, int64_t d,
                                        int64_t batch, const int32_t* perm_dev, int64_t stride_perm,
                                        const float* num_samples_dev, float percdamp, float* hinv_dev,
                                        int64_t stride_hinv, int32_t* dead_dev, int32_t* status_dev,
                                        void* workspace_dev, size_t workspace_bytes, void* stream) {
  MQ_CHECK_ARG(h_dev && hinv_dev && status_dev && num_samples_dev, "gptq_hinv_batched: null pointer");
  MQ_CHECK_ARG(d > 0 && ldh >= d && batch > 0 && batch <= 65535, "gptq_hinv_batched: bad shape");
  MQ_CHECK_ARG(stride_h >= ldh * d && stride_hinv >= d * d, "gptq_hinv_batched: matrices overlap");
  MQ_CHECK_ARG(!perm_dev || stride_perm >= 0, "gptq_hinv_batched: bad perm stride");
  const HinvLayout L = hinv_layout(d);
  MQ_CHECK_ARG(workspace_dev && workspace_bytes >= L.total * (size_t)batch,
               "gptq_hinv_batched: workspace too small (%zu < %zu)", workspace_bytes, L.total * (size_t)batch);
  return hinv_impl(h_dev, ldh, stride_h, d, batch, perm_dev, stride_perm, num_samples_dev, 0.f, percdamp,
                   hinv_dev, stride_hinv, dead_dev, status_dev, static_cast<char*>(workspace_dev),
                   reinterpret_cast<hipStream_t>(stream));
}

extern "C" int mi355q_gptq_hinv_fallback(float* hinv_dev, int64_t d, int64_t stride_hinv, int64_t batch,
                                         const int32_t* status_dev, void* stream) {
  MQ_CHECK_ARG(d > 0 && batch > 0 && batch <= 65535, "hinv fallback: bad d or batch");
  MQ_CHECK_ARG(stride_hinv >= d * d || batch == 1, "hinv fallback: stride_hinv below d * d");
  MQ_CHECK_ARG(hinv_dev != nullptr && status_dev != nullptr, "hinv fallback: null pointer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int64_t blocks = (d * d + 255) / 256;
  hipLaunchKernelGGL(identity_on_failure_kernel, dim3((unsigned)(blocks < 1024 ? blocks : 1024), (unsigned)batch),
                     dim3(256), 0, st, hinv_dev, d, stride_hinv, status_dev);
  MQ_LAUNCH_CHECK();
  return MI355Q_OK;
}
