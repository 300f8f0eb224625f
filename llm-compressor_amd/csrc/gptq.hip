// GPTQ blocked column sweep on gfx950.
//
// Replaces modifiers/gptq/gptq_quantize.py:199-277.  Rows of W are
// independent given Hinv and the (static) scales, so the serial column loop
// runs for all rows at once: a workgroup holds 16 rows, each row is shared by
// 16 lanes, and lane g owns the block columns j = 16 t + g (t = 0..7) in
// registers.  For column i the owner's value is broadcast to its 16 lanes,
// every lane quantises it (CT quantize/dequantize arithmetic), and each lane
// applies err * Hinv[i][j] to its own later columns as a rounded multiply
// followed by a rounded subtract (the reference's outer-product matmul and
// in-place subtract).  Hinv's diagonal block sits in LDS.  After each block
// the lazy update W[:, i2:] -= Err @ Hinv[i1:i2, i2:] runs as an fp32 MFMA
// GEMM whose output is rounded once and then subtracted, as in the reference.
#include "gptq_sweep.h"

#include <algorithm>
#include <mutex>

#pragma clang fp contract(off)

namespace mi355q {
int64_t gemm_cus();  // compute units (the GEMM dispatch's count)
namespace {

// One row per blockIdx.y, four consecutive output columns per thread.
// (matrix blockIdx.z of a batch: w + z sw elements, perm + z sp, dead + z cols,
// out + z rows cols)
__global__ void load_weight_kernel(const void* w, mi355q_dtype dt, int64_t rows, int64_t cols, int64_t ldw,
                                   const int32_t* perm, const int32_t* dead, float* out, int64_t sw, int64_t sp) {
  const int64_t z = blockIdx.z;
  w = dt == MI355Q_BF16 ? (const void*)(static_cast<const uint16_t*>(w) + z * sw)
                        : (const void*)(static_cast<const float*>(w) + z * sw);
  if (perm) perm += z * sp;
  if (dead) dead += z * cols;
  out += z * rows * cols;
  const int64_t r = blockIdx.y;
  // whole rows of bf16 without a permutation: 8-byte loads of four values
  const bool vec = !perm && dt == MI355Q_BF16 && (cols & 3) == 0 && (ldw & 3) == 0 &&
                   (reinterpret_cast<uintptr_t>(w) & 7) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(dead) & 15) == 0;
  for (int64_t j4 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4; j4 < cols;
       j4 += (int64_t)gridDim.x * blockDim.x * 4) {
    f32x4_t v;
    if (vec) {
      const uint2 u = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(w) + r * ldw + j4);
      v[0] = __uint_as_float(u.x << 16);
      v[1] = __uint_as_float(u.x & 0xffff0000u);
      v[2] = __uint_as_float(u.y << 16);
      v[3] = __uint_as_float(u.y & 0xffff0000u);
      if (dead) {
        const int4 dd = *reinterpret_cast<const int4*>(dead + j4);
        if (dd.x) v[0] = 0.f;
        if (dd.y) v[1] = 0.f;
        if (dd.z) v[2] = 0.f;
        if (dd.w) v[3] = 0.f;
      }
      *reinterpret_cast<f32x4_t*>(out + r * cols + j4) = v;
      continue;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t j = j4 + e < cols ? j4 + e : cols - 1;
      const int64_t src = perm ? perm[j] : j;
      float x = dt == MI355Q_BF16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(w)[r * ldw + src])
                                  : static_cast<const float*>(w)[r * ldw + src];
      v[e] = (dead && dead[j]) ? 0.f : x;
    }
    float* o = out + r * cols + j4;
    if ((cols & 3) == 0) {
      *reinterpret_cast<f32x4_t*>(o) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (j4 + e < cols) o[e] = v[e];
    }
  }
}

// (matrix blockIdx.z: w, cin, cout + z rows cols; invperm + z sp; out + z so)
__global__ void store_weight_kernel(const float* w, int64_t rows, int64_t cols, const int32_t* invperm,
                                    void* out, mi355q_dtype dt, int64_t ld_out, const int8_t* cin,
                                    int8_t* cout, int64_t sp, int64_t so) {
  const int64_t z = blockIdx.z;
  w += z * rows * cols;
  if (invperm) invperm += z * sp;
  out = dt == MI355Q_BF16 ? (void*)(static_cast<uint16_t*>(out) + z * so) : (void*)(static_cast<float*>(out) + z * so);
  if (cin) cin += z * rows * cols;
  if (cout) cout += z * rows * cols;
  const int64_t r = blockIdx.y;
  // whole rows to bf16 without a permutation: 16-byte loads, 8-byte stores
  const bool vec = !invperm && dt == MI355Q_BF16 && (cols & 3) == 0 && (ld_out & 3) == 0 &&
                   (reinterpret_cast<uintptr_t>(out) & 7) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(cin) & 3) == 0 && (reinterpret_cast<uintptr_t>(cout) & 3) == 0;
  for (int64_t j4 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4; j4 < cols;
       j4 += (int64_t)gridDim.x * blockDim.x * 4) {
    if (vec) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(w + r * cols + j4);
      uint2 u;
      u.x = f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16);
      u.y = f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16);
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + r * ld_out + j4) = u;
      if (cin && cout)
        *reinterpret_cast<uint32_t*>(cout + r * cols + j4) = *reinterpret_cast<const uint32_t*>(cin + r * cols + j4);
      continue;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t j = j4 + e;
      if (j >= cols) break;
      const int64_t src = r * cols + (invperm ? invperm[j] : j);
      const float v = w[src];
      if (dt == MI355Q_BF16)
        static_cast<uint16_t*>(out)[r * ld_out + j] = f32_to_bf16_bits(v);
      else
        static_cast<float*>(out)[r * ld_out + j] = v;
      if (cin && cout) cout[r * cols + j] = cin[src];
    }
  }
}

// Permuted rows: the row is read in order into LDS and gathered from there.
// A gather straight from global memory touches a 64-byte line per element and
// lane; from LDS the memory traffic is the rows themselves.  A workgroup
// takes `nr` rows so that the permutation is read once for all of them (nr
// rows of LDS words, at most PERM_LDS bytes, two workgroups per CU).
// Bound by HBM; measured, 14336 x 4096 with codes: load 191 -> 74 us (4.8
// TB/s), store 457 -> 95 us (5.0 TB/s).
constexpr int PERM_NT = 512;
constexpr int64_t PERM_LDS = 64 << 10;  // LDS bytes of the staged rows

constexpr int64_t PERM_MIN = 3 << 18;  // elements from which staging is the faster way

// Rows per workgroup for rows of `bytes` LDS bytes, few enough to leave no CU
// without one (256 x 4096 bf16 loaded on 32 workgroups of eight rows took 8.1
// us, on 256 of one 4.7); 0: gathered straight from memory, either because a
// row is too wide to stage or because the call is small: few workgroups then
// read, wait and gather in turn, where the direct gather is spread over the chip
// and takes hardly more than a launch (us, direct / staged, load bf16 | store
// bf16 with codes: 16 x 14336 4.3 / 6.7 | 4.9 / 7.7, 64 x 8192 4.3 / 5.0 | 5.3 /
// 5.9; from there on 64 x 14336 5.5 / 6.9 | 11.0 / 7.8, 128 x 8192 5.3 / 5.4 | 15.2
// / 5.9, 512 x 4096 6.2 / 5.2 | 20.5 / 5.7).
inline int perm_rows(int64_t bytes, int64_t rows, int64_t cols, int64_t batch) {
  if (rows * batch * cols < PERM_MIN) return 0;
  const int64_t n = PERM_LDS / bytes, most = std::max<int64_t>(rows * batch / gemm_cus(), 1);
  return (int)std::min<int64_t>(std::min<int64_t>(n, most), 8);
}

// out[r][j] = dead[j] ? 0 : w[r][perm[j]], rows nr blockIdx.x .. (matrix
// blockIdx.z as load_weight_kernel)
template <typename T>
__global__ __launch_bounds__(PERM_NT) void load_weight_perm_kernel(const T* w, int64_t rows, int64_t cols, int64_t ldw,
                                                                   const int32_t* perm, const int32_t* dead,
                                                                   float* out, int64_t sw, int64_t sp, int nr) {
  extern __shared__ __attribute__((aligned(16))) char perm_smem[];
  T* lw = reinterpret_cast<T*>(perm_smem);
  const int64_t z = blockIdx.z;
  w += z * sw;
  perm += z * sp;
  if (dead) dead += z * cols;
  out += z * rows * cols;
  const int64_t r0 = (int64_t)blockIdx.x * nr;
  const int n = (int)(rows - r0 < nr ? rows - r0 : nr);
  constexpr int V = 16 / sizeof(T);
  if (cols % V == 0 && ldw % V == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0) {
    for (int r = 0; r < n; ++r)
      for (int64_t j = (int64_t)threadIdx.x * V; j < cols; j += PERM_NT * V)
        *reinterpret_cast<u32x4_t*>(lw + r * cols + j) = *reinterpret_cast<const u32x4_t*>(w + (r0 + r) * ldw + j);
  } else {
    for (int r = 0; r < n; ++r)
      for (int64_t j = threadIdx.x; j < cols; j += PERM_NT) lw[r * cols + j] = w[(r0 + r) * ldw + j];
  }
  __syncthreads();
  const bool vec = (cols & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  for (int64_t j4 = (int64_t)threadIdx.x * 4; j4 < cols; j4 += PERM_NT * 4) {
    int src[4];
    bool off[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t j = j4 + e < cols ? j4 + e : cols - 1;
      src[e] = perm[j];
      off[e] = dead && dead[j];
    }
    for (int r = 0; r < n; ++r) {
      f32x4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const T x = lw[r * cols + src[e]];
        v[e] = off[e] ? 0.f : sizeof(T) == 2 ? bf16_bits_to_f32((uint16_t)x) : __uint_as_float((uint32_t)x);
      }
      float* o = out + (r0 + r) * cols + j4;
      if (vec) {
        *reinterpret_cast<f32x4_t*>(o) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (j4 + e < cols) o[e] = v[e];
      }
    }
  }
}

// out[r][j] = w[r][invperm[j]] (and the codes likewise) for rows nr
// blockIdx.x ..; a staged word holds the bf16 bits and the code above them,
// or, for fp32 (BF16 false), the value with the codes' bytes behind the rows.
template <bool BF16>
__global__ __launch_bounds__(PERM_NT) void store_weight_perm_kernel(const float* w, int64_t rows, int64_t cols,
                                                                    const int32_t* invperm, void* out,
                                                                    int64_t ld_out, const int8_t* cin, int8_t* cout,
                                                                    int64_t sp, int64_t so, int nr) {
  extern __shared__ __attribute__((aligned(16))) char perm_smem[];
  uint32_t* lw = reinterpret_cast<uint32_t*>(perm_smem);
  int8_t* lc = reinterpret_cast<int8_t*>(lw + (int64_t)nr * cols);
  const int64_t z = blockIdx.z;
  w += z * rows * cols;
  invperm += z * sp;
  uint16_t* ob = static_cast<uint16_t*>(out) + z * so;
  float* of = static_cast<float*>(out) + z * so;
  const bool codes = cin && cout;
  if (codes) {
    cin += z * rows * cols;
    cout += z * rows * cols;
  }
  const int64_t r0 = (int64_t)blockIdx.x * nr;
  const int n = (int)(rows - r0 < nr ? rows - r0 : nr);
  // the rows are consecutive: one run of n cols elements
  const float* wr = w + r0 * cols;
  const int8_t* cr = cin + r0 * cols;
  const int64_t total = (int64_t)n * cols;
  const bool vin = (cols & 3) == 0 && (reinterpret_cast<uintptr_t>(wr) & 15) == 0 &&
                   (!codes || (reinterpret_cast<uintptr_t>(cr) & 3) == 0);
  auto stage = [&](int64_t i, float x, uint32_t c) __attribute__((always_inline)) {
    if (BF16) {
      lw[i] = f32_to_bf16_bits(x) | (c << 16);
    } else {
      lw[i] = __float_as_uint(x);
      if (codes) lc[i] = (int8_t)c;
    }
  };
  if (vin) {
    for (int64_t i = (int64_t)threadIdx.x * 4; i < total; i += PERM_NT * 4) {
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(wr + i);
      const uint32_t c = codes ? *reinterpret_cast<const uint32_t*>(cr + i) : 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) stage(i + e, x[e], (c >> (8 * e)) & 0xffu);
    }
  } else {
    for (int64_t i = threadIdx.x; i < total; i += PERM_NT) stage(i, wr[i], codes ? (uint8_t)cr[i] : 0u);
  }
  __syncthreads();
  const bool vout = (cols & 3) == 0 && (ld_out & 3) == 0 && (reinterpret_cast<uintptr_t>(ob) & 7) == 0 &&
                    (BF16 || (reinterpret_cast<uintptr_t>(of) & 15) == 0) &&
                    (!codes || (reinterpret_cast<uintptr_t>(cout) & 3) == 0);
  for (int64_t j4 = (int64_t)threadIdx.x * 4; j4 < cols; j4 += PERM_NT * 4) {
    int src[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) src[e] = invperm[j4 + e < cols ? j4 + e : cols - 1];
    for (int r = 0; r < n; ++r) {
      uint32_t v[4], c[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t i = (int64_t)r * cols + src[e];
        v[e] = lw[i];
        c[e] = BF16 ? v[e] >> 16 : codes ? (uint8_t)lc[i] : 0u;
      }
      const int64_t ro = (r0 + r) * ld_out + j4, rc = (r0 + r) * cols + j4;
      if (vout) {
        if (BF16) {
          uint2 u;
          u.x = (v[0] & 0xffffu) | (v[1] << 16);
          u.y = (v[2] & 0xffffu) | (v[3] << 16);
          *reinterpret_cast<uint2*>(ob + ro) = u;
        } else {
          const u32x4_t u = {v[0], v[1], v[2], v[3]};
          *reinterpret_cast<u32x4_t*>(of + ro) = u;
        }
        if (codes)
          *reinterpret_cast<uint32_t*>(cout + rc) =
              (c[0] & 0xffu) | (c[1] & 0xffu) << 8 | (c[2] & 0xffu) << 16 | c[3] << 24;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (j4 + e < cols) {
            if (BF16)
              ob[ro + e] = (uint16_t)v[e];
            else
              of[ro + e] = __uint_as_float(v[e]);
            if (codes) cout[rc + e] = (int8_t)c[e];
          }
      }
    }
  }
}

inline dim3 grid_rows(int64_t rows, int64_t cols, int64_t batch = 1) {
  int64_t gx = (cols / 4 + 255) / 256;
  if (gx < 1) gx = 1;
  if (gx > 64) gx = 64;
  return dim3((unsigned)gx, (unsigned)rows, (unsigned)batch);
}

}  // namespace
}  // namespace mi355q

using namespace mi355q;
using namespace mi355q::sweep;
using mi355q::gsw::QK_INT;
using mi355q::gsw::QK_FP8;
using mi355q::gsw::QK_FP4;
using mi355q::gsw::SweepBatch;

extern "C" int mi355q_gptq_load_weight_batched(const void* w_dev, mi355q_dtype w_dtype, int64_t rows,
                                               int64_t cols, int64_t ldw, int64_t stride_w, int64_t batch,
                                               const int32_t* perm_dev, int64_t stride_perm,
                                               const int32_t* dead_dev, float* w_work_dev, void* stream) {
  MQ_CHECK_ARG(w_dev && w_work_dev, "gptq_load_weight: null pointer");
  MQ_CHECK_ARG(rows > 0 && cols > 0 && ldw >= cols && batch > 0, "gptq_load_weight: bad shape");
  MQ_CHECK_ARG(w_dtype == MI355Q_BF16 || w_dtype == MI355Q_F32, "gptq_load_weight: dtype must be bf16 or fp32");
  MQ_CHECK_ARG(rows <= 65535 && batch <= 65535, "gptq_load_weight: at most 65535 rows and matrices");
  MQ_CHECK_ARG(batch == 1 || stride_w >= rows * ldw, "gptq_load_weight: matrices overlap");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // a permutation gathers from rows staged in LDS, unless a row is too wide for
  // that (then straight from memory: 2.6 and 4.8 times the time) or the call small
  const int64_t row_bytes = cols * (w_dtype == MI355Q_BF16 ? 2 : 4);
  const int nr = perm_dev ? perm_rows(row_bytes, rows, cols, batch) : 0;
  const dim3 pgrid((unsigned)(nr ? (rows + nr - 1) / nr : 1), 1, (unsigned)batch);
  if (nr && w_dtype == MI355Q_BF16)
    hipLaunchKernelGGL(load_weight_perm_kernel<uint16_t>, pgrid, dim3(PERM_NT), (size_t)(nr * row_bytes), st,
                       static_cast<const uint16_t*>(w_dev), rows, cols, ldw, perm_dev, dead_dev, w_work_dev, stride_w,
                       stride_perm, nr);
  else if (nr)
    hipLaunchKernelGGL(load_weight_perm_kernel<uint32_t>, pgrid, dim3(PERM_NT), (size_t)(nr * row_bytes), st,
                       static_cast<const uint32_t*>(w_dev), rows, cols, ldw, perm_dev, dead_dev, w_work_dev, stride_w,
                       stride_perm, nr);
  else
    hipLaunchKernelGGL(load_weight_kernel, grid_rows(rows, cols, batch), dim3(256), 0, st, w_dev, w_dtype, rows, cols,
                       ldw, perm_dev, dead_dev, w_work_dev, stride_w, stride_perm);
  MQ_LAUNCH_CHECK();
  return MI355Q_OK;
}

extern "C" int mi355q_gptq_load_weight(const void* w_dev, mi355q_dtype w_dtype, int64_t rows, int64_t cols,
                                       int64_t ldw, const int32_t* perm_dev, const int32_t* dead_dev,
                                       float* w_work_dev, void* stream) {
  return mi355q_gptq_load_weight_batched(w_dev, w_dtype, rows, cols, ldw, 0, 1, perm_dev, 0, dead_dev,
                                         w_work_dev, stream);
}

extern "C" size_t mi355q_gptq_sweep_workspace_size(int64_t rows, int64_t cols, int64_t blocksize) {
  if (rows <= 0 || cols <= 0 || blocksize <= 0) return 0;
  return (size_t)rows * err_cols(cols, blocksize) * sizeof(float);
}

extern "C" int mi355q_gptq_sweep_typed_batched(float* w_work_dev, int64_t rows, int64_t cols, int64_t batch,
                                               const float* hinv_dev, int64_t stride_hinv, const float* scale_dev,
                                               const float* zp_dev, int64_t ld_scale, int64_t stride_scale,
                                               const int32_t* g_idx_dev, int64_t stride_gidx, int strategy,
                                               int block_h, int qtype, float qmin, float qmax,
                                               const float* global_scale_dev, int dequant_bf16, int64_t blocksize,
                                               int8_t* codes_dev, float* losses_dev, void* workspace_dev,
                                               size_t workspace_bytes, void* stream) {
  MQ_CHECK_ARG(w_work_dev && hinv_dev && scale_dev && codes_dev && losses_dev, "gptq_sweep: null pointer");
  MQ_CHECK_ARG(rows > 0 && cols > 0 && batch > 0 && batch <= 65535, "gptq_sweep: bad shape");
  MQ_CHECK_ARG(blocksize > 0, "gptq_sweep: blocksize must be positive");
  MQ_CHECK_ARG(strategy == MI355Q_TENSOR || strategy == MI355Q_CHANNEL || strategy == MI355Q_GROUP ||
                   strategy == MI355Q_BLOCK,
               "Quantization strategy is not supported for GPTQ: %d", strategy);
  MQ_CHECK_ARG((strategy != MI355Q_GROUP && strategy != MI355Q_BLOCK) || g_idx_dev,
               "gptq_sweep: group/block strategies need g_idx");
  MQ_CHECK_ARG(strategy != MI355Q_BLOCK || block_h > 0, "gptq_sweep: block_h must be positive");
  MQ_CHECK_ARG(qtype == MI355Q_QTYPE_INT || qtype == MI355Q_QTYPE_FP8_E4M3 || qtype == MI355Q_QTYPE_FP4_E2M1,
               "gptq_sweep: unknown value type %d", qtype);
  if (qtype == MI355Q_QTYPE_INT)
    MQ_CHECK_ARG(qmin < qmax && qmin >= -128.f && qmax <= 127.f, "gptq_sweep: integer range must fit int8");
  else
    MQ_CHECK_ARG(!zp_dev && qmin == -qmax && qmax <= (qtype == MI355Q_QTYPE_FP8_E4M3 ? 448.f : 6.f) && qmax > 0.f,
                 "gptq_sweep: float types are symmetric within the type's range");
  MQ_CHECK_ARG(batch == 1 || stride_hinv >= cols * cols, "gptq_sweep: Hinv matrices overlap");
  const size_t need = mi355q_gptq_sweep_workspace_size(rows, cols, blocksize) * (size_t)batch;
  MQ_CHECK_ARG(workspace_dev && workspace_bytes >= need, "gptq_sweep: workspace too small");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  float* err = static_cast<float*>(workspace_dev);
  const int64_t lde = err_cols(cols, blocksize);
  SweepBatch sb{rows * cols, stride_hinv, stride_scale, stride_gidx, rows * cols, rows, rows * lde};
  const int qk = qtype == MI355Q_QTYPE_FP8_E4M3 ? QK_FP8 : qtype == MI355Q_QTYPE_FP4_E2M1 ? QK_FP4 : QK_INT;
  // the sweep kernel holds at most MAXB columns; larger reference block
  // sizes give the same result up to fp32 rounding of the lazy update, so
  // they are processed in MAXB-wide sub-blocks
  const int64_t B = blocksize < MAXB ? blocksize : MAXB;
  const unsigned nwg = (unsigned)((rows + SW_ROWS - 1) / SW_ROWS);
  int dev = 0, ncu = 0;
  MQ_CHECK_HIP(hipGetDevice(&dev));
  MQ_CHECK_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  // Whole integer blocks with symmetric scales of grids with at least eight
  // 16-lane workgroups per CU take the 4-lane sweep (instruction issue, not
  // latency, bounds the 16-lane sweep there).
  const bool wide = (int64_t)nwg * batch >= 8 * (int64_t)ncu;
  // (npre > 0 only for whole blocks: the schedule pulls only in mid-blocks of whole blocks)
  auto block = [&](int64_t i1, int64_t i2, int64_t s0, int npre, int64_t m0) {
    const int count = (int)(i2 - i1);
    MQ_CHECK_ARG(npre == 0 || (count == MAXB && qk == QK_INT), "gptq_sweep: pulled updates need whole integer blocks");
    const gsw::SweepLaunch a{w_work_dev, rows, cols, hinv_dev, i1, count, scale_dev, zp_dev, ld_scale, g_idx_dev,
                             strategy, block_h, qmin, qmax, global_scale_dev, codes_dev, losses_dev, err, lde,
                             (int)(i1 - s0), npre, m0, (int)(m0 - s0), sb};
    const bool bf16 = dequant_bf16 != 0;
    const dim3 grid(nwg, (unsigned)batch);
    if (qk != QK_INT)
      gsw::launch_sweep_float(qk, count == MAXB, bf16, grid, st, a);
    else if (npre > 0)
      gsw::launch_sweep_pull(bf16, zp_dev != nullptr, grid, st, a);
    else if (wide && count == MAXB && !zp_dev)
      gsw::launch_sweep4(bf16, dim3((unsigned)((rows + gsw::W4_ROWS - 1) / gsw::W4_ROWS), (unsigned)batch), st, a);
    else
      gsw::launch_sweep_int(count == MAXB, bf16, zp_dev != nullptr, grid, st, a);
    MQ_LAUNCH_CHECK();
    return MI355Q_OK;
  };
  auto lazy = [&](int64_t k0, int64_t k1, int64_t s0, int64_t c0, int64_t c1) {
    return lazy_update(w_work_dev, rows, cols, batch, hinv_dev, stride_hinv, err, lde, k0, k1, s0, c0, c1, st);
  };
  // The sweep workgroups apply a mid-block's K = 128 updates themselves for
  // integer values when the sweep leaves the CUs room for it (at most two of
  // its workgroups per CU; with more, the separate products use the CUs
  // better) and the error tile can be read in 16-byte pieces.
  const bool can_pull = qk == QK_INT && (int64_t)nwg * batch <= 2 * (int64_t)ncu && lde % 4 == 0 &&
                        (reinterpret_cast<uintptr_t>(err) & 15) == 0;
  return blocked_schedule_pull(cols, B, can_pull, block, lazy);
}

extern "C" int mi355q_gptq_sweep_batched(float* w_work_dev, int64_t rows, int64_t cols, int64_t batch,
                                         const float* hinv_dev, int64_t stride_hinv, const float* scale_dev,
                                         const float* zp_dev, int64_t ld_scale, int64_t stride_scale,
                                         const int32_t* g_idx_dev, int64_t stride_gidx, int strategy, int block_h,
                                         float qmin, float qmax, int dequant_bf16, int64_t blocksize,
                                         int8_t* codes_dev, float* losses_dev, void* workspace_dev,
                                         size_t workspace_bytes, void* stream) {
  return mi355q_gptq_sweep_typed_batched(w_work_dev, rows, cols, batch, hinv_dev, stride_hinv, scale_dev, zp_dev,
                                         ld_scale, stride_scale, g_idx_dev, stride_gidx, strategy, block_h,
                                         MI355Q_QTYPE_INT, qmin, qmax, nullptr, dequant_bf16, blocksize, codes_dev,
                                         losses_dev, workspace_dev, workspace_bytes, stream);
}

extern "C" int mi355q_gptq_sweep(float* w_work_dev, int64_t rows, int64_t cols, const float* hinv_dev,
                                 const float* scale_dev, const float* zp_dev, int64_t ld_scale,
                                 const int32_t* g_idx_dev, int strategy, int block_h, float qmin, float qmax,
                                 int dequant_bf16, int64_t blocksize, int8_t* codes_dev, float* losses_dev,
                                 void* workspace_dev, size_t workspace_bytes, void* stream) {
  return mi355q_gptq_sweep_batched(w_work_dev, rows, cols, 1, hinv_dev, 0, scale_dev, zp_dev, ld_scale, 0,
                                   g_idx_dev, 0, strategy, block_h, qmin, qmax, dequant_bf16, blocksize,
                                   codes_dev, losses_dev, workspace_dev, workspace_bytes, stream);
}

extern "C" int mi355q_gptq_store_weight_batched(const float* w_work_dev, int64_t rows, int64_t cols,
                                                int64_t batch, const int32_t* invperm_dev, int64_t stride_perm,
                                                void* w_out_dev, mi355q_dtype out_dtype, int64_t ld_out,
                                                int64_t stride_out, const int8_t* codes_in_dev,
                                                int8_t* codes_out_dev, void* stream) {
  MQ_CHECK_ARG(w_work_dev && w_out_dev, "gptq_store_weight: null pointer");
  MQ_CHECK_ARG(rows > 0 && cols > 0 && ld_out >= cols && batch > 0, "gptq_store_weight: bad shape");
  MQ_CHECK_ARG(out_dtype == MI355Q_BF16 || out_dtype == MI355Q_F32, "gptq_store_weight: dtype must be bf16 or fp32");
  MQ_CHECK_ARG(codes_out_dev != codes_in_dev || !codes_in_dev, "gptq_store_weight: codes must not alias");
  MQ_CHECK_ARG(rows <= 65535 && batch <= 65535, "gptq_store_weight: at most 65535 rows and matrices");
  MQ_CHECK_ARG(batch == 1 || stride_out >= rows * ld_out, "gptq_store_weight: matrices overlap");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool bf16 = out_dtype == MI355Q_BF16;
  const int64_t row_bytes = cols * (bf16 ? 4 : 5);
  const int nr = invperm_dev ? perm_rows(row_bytes, rows, cols, batch) : 0;
  const dim3 pgrid((unsigned)(nr ? (rows + nr - 1) / nr : 1), 1, (unsigned)batch);
  if (nr && bf16)
    hipLaunchKernelGGL(store_weight_perm_kernel<true>, pgrid, dim3(PERM_NT), (size_t)(nr * row_bytes), st, w_work_dev,
                       rows, cols, invperm_dev, w_out_dev, ld_out, codes_in_dev, codes_out_dev, stride_perm,
                       stride_out, nr);
  else if (nr)
    hipLaunchKernelGGL(store_weight_perm_kernel<false>, pgrid, dim3(PERM_NT), (size_t)(nr * row_bytes), st, w_work_dev,
                       rows, cols, invperm_dev, w_out_dev, ld_out, codes_in_dev, codes_out_dev, stride_perm,
                       stride_out, nr);
  else
    hipLaunchKernelGGL(store_weight_kernel, grid_rows(rows, cols, batch), dim3(256), 0, st, w_work_dev, rows, cols,
                       invperm_dev, w_out_dev, out_dtype, ld_out, codes_in_dev, codes_out_dev, stride_perm,
                       stride_out);
  MQ_LAUNCH_CHECK();
  return MI355Q_OK;
}

extern "C" int mi355q_gptq_store_weight(const float* w_work_dev, int64_t rows, int64_t cols,
                                        const int32_t* invperm_dev, void* w_out_dev, mi355q_dtype out_dtype,
                                        int64_t ld_out, const int8_t* codes_in_dev, int8_t* codes_out_dev,
                                        void* stream) {
  return mi355q_gptq_store_weight_batched(w_work_dev, rows, cols, 1, invperm_dev, 0, w_out_dev, out_dtype,
                                          ld_out, 0, codes_in_dev, codes_out_dev, stream);
}

// ---------------------------------------------------------------- sweep without allocation
// The sweep's error workspace in a device array the library holds: one copy
// per GPU (each device's own address, from hipGetSymbolAddress with that
// device current, looked up once per device), alive until the process ends.
// Every call on a GPU shares that GPU's array, so calls that overlap on one
// GPU (different streams or threads) race; the sweep writes each error
// column before any product reads it, so nothing needs clearing between calls.
static constexpr size_t kSweepScratchBytes = size_t(64) << 20;
static __device__ __align__(256) float scratch[kSweepScratchBytes / sizeof(float)];

namespace {
struct ScratchSlot {
  std::once_flag once;
  void* ptr = nullptr;
  hipError_t err = hipSuccess;
};
constexpr int kMaxDevices = 64;
ScratchSlot g_scratch_slot[kMaxDevices];

int sweep_scratch(void** out) {
  int dev = 0;
  MQ_CHECK_HIP(hipGetDevice(&dev));
  MQ_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "gptq_sweep_noalloc: device index %d out of range", dev);
  ScratchSlot& s = g_scratch_slot[dev];
  std::call_once(s.once, [&s] { s.err = hipGetSymbolAddress(&s.ptr, HIP_SYMBOL(scratch)); });
  if (s.err != hipSuccess || s.ptr == nullptr) {
    set_error("gptq_sweep_noalloc: hipGetSymbolAddress of the scratch array failed on device %d: %s", dev,
              hipGetErrorString(s.err));
    return MI355Q_HIP_ERROR;
  }
  *out = s.ptr;
  return MI355Q_OK;
}
}  // namespace

extern "C" size_t mi355q_gptq_sweep_noalloc_max_bytes(void) { return kSweepScratchBytes; }

extern "C" int mi355q_gptq_sweep_noalloc(float* w_work_dev, int64_t rows, int64_t cols, const float* hinv_dev,
                                         const float* scale_dev, const float* zp_dev, int64_t ld_scale,
                                         const int32_t* g_idx_dev, int strategy, int block_h, float qmin, float qmax,
                                         int dequant_bf16, int64_t blocksize, int8_t* codes_dev, float* losses_dev,
                                         void* stream) {
  MQ_CHECK_ARG(rows > 0 && cols > 0 && blocksize > 0, "gptq_sweep_noalloc: bad shape");
  const size_t need = mi355q_gptq_sweep_workspace_size(rows, cols, blocksize);
  MQ_CHECK_ARG(need <= kSweepScratchBytes,
               "gptq_sweep_noalloc: the error workspace of %lld x %lld needs %zu bytes, above the %zu-byte scratch "
               "array (rows * min(1024, cols) fp32); use mi355q_gptq_sweep with a caller workspace",
               (long long)rows, (long long)cols, need, kSweepScratchBytes);
  void* ws = nullptr;
  const int rc = sweep_scratch(&ws);
  if (rc) return rc;
  return mi355q_gptq_sweep(w_work_dev, rows, cols, hinv_dev, scale_dev, zp_dev, ld_scale, g_idx_dev, strategy, block_h,
                           qmin, qmax, dequant_bf16, blocksize, codes_dev, losses_dev, ws, kSweepScratchBytes, stream);
}
