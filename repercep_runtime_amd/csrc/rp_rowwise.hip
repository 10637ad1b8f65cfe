// Row-wise FP8 quantization for gfx950, and the row kernels of the unfused
// FP8 attention built on it.
//
// Semantics follow _rowwise_quantize of the reference's unfused FP8
// attention (src/repercep/attention/fp8_scaled_mm.py:107-133) with the OCP
// e4m3fn constants (FP8_MAX 448, target 0.95 * 448 -> 425.6f as torch applies
// the Python scalar), the same adaptation the OCP siblings of the per-(b,h)
// quantizer make (kernels/triton_kernels/fp8_flash_attn_hopper.py:374-398).
// For each row of `cols` elements, in the input dtype (bf16 or fp16):
//   amax    = max |x| over the row, clamped below at dtype(1e-6)
//   qmul    = dtype(dtype(1 / amax) * 425.6f)  -- torch's `target / amax` is
//             amax.reciprocal() * target: two roundings to the dtype
//   dequant = dtype(amax / 425.6)                -- as the per-(b,h) scale
//   codes   = e4m3fn(clamp(fp32(x) * qmul, -448, 448)), round to nearest even
// so a row's largest element maps to ~425.6, like the per-(b,h) path, but
// through a 16-bit multiplier instead of the fp32 reciprocal of the scale.
//
// Kernels:
// * rowwise_quant_kernel<DT, TPR>: rows of at most 2048 elements; TPR
//   consecutive lanes hold one row (<= 4 16-byte vectors each), reduce its
//   maximum with a butterfly and write its codes: one read, one write.
// * rowwise_quant_long_kernel<DT>: longer rows, one workgroup per row, the
//   row read twice (the second read mostly from L2).
// * transpose16_kernel: a 16-bit (R, C) -> (C, R) transpose through LDS, for
//   V^T, whose rows (one per head-dim index) the P.V product quantizes.
// * softmax_rowquant_vec_kernel: rows of raw scores held in registers:
//   s = bf16(raw * scale), the causal mask, P = softmax(s) rounded to bf16
//   as torch's bf16 softmax returns it, and P's row-wise codes and scale.
//   The row maximum of P is bf16(1 / sum) -- exp(0) = 1 at the row's largest
//   score, and rounding is monotone -- so P's scale is known before its
//   codes are written, and the row is read once.
// * softmax_rowquant_kernel: the same for rows the register kernel does not
//   take (too long, or not whole 16-byte vectors), in three passes over the
//   row (max, sum, output).

#include <type_traits>

#include "rp_common.h"

namespace rp {
namespace {

constexpr int kRThreads = 256;
typedef unsigned int u32x4r __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2r __attribute__((ext_vector_type(2)));

// qmul and dequant of a row from the bit pattern of its |x| maximum.
template <int DT>
__device__ __forceinline__ void rowwise_scales(uint32_t amax_bits, float* qmul, float* dequant) {
  if constexpr (DT == kInF16) {
    const float lo = 17.0f * 0x1p-24f;  // fp16(1e-6)
    float a = f16_to_f32(amax_bits);
    if (!(a != a) && a < lo) a = lo;
    const float r = f16_round(1.0f / a);
    *qmul = f16_round(r * kScaleDivisor);
    *dequant = f16_round(a * (1.0f / kScaleDivisor));
  } else {
    const float lo = __uint_as_float(0x3586u << 16);  // bf16(1e-6)
    float a = bf16_to_f32(amax_bits);
    if (!(a != a) && a < lo) a = lo;
    const float r = bf16_round(1.0f / a);
    *qmul = bf16_round(r * kScaleDivisor);
    *dequant = bf16_round(a / kScaleDivisor);
  }
}

__device__ __forceinline__ uint32_t pk_umax16r(uint32_t a, uint32_t b) {
  const uint32_t lo = umax32(a & 0xffffu, b & 0xffffu);
  const uint32_t hi = umax32(a >> 16, b >> 16);
  return lo | (hi << 16);
}

// Eight inputs (one 16-byte vector) -> eight codes.
template <int DT>
__device__ __forceinline__ uint2 quant8(const u32x4r& v, float qm) {
  uint2 o;
  const float a0 = clamp_e4m3(in_to_f32<DT>(v[0] & 0xffffu) * qm);
  const float a1 = clamp_e4m3(in_to_f32<DT>(v[0] >> 16) * qm);
  const float a2 = clamp_e4m3(in_to_f32<DT>(v[1] & 0xffffu) * qm);
  const float a3 = clamp_e4m3(in_to_f32<DT>(v[1] >> 16) * qm);
  const float a4 = clamp_e4m3(in_to_f32<DT>(v[2] & 0xffffu) * qm);
  const float a5 = clamp_e4m3(in_to_f32<DT>(v[2] >> 16) * qm);
  const float a6 = clamp_e4m3(in_to_f32<DT>(v[3] & 0xffffu) * qm);
  const float a7 = clamp_e4m3(in_to_f32<DT>(v[3] >> 16) * qm);
  o.x = pack4_e4m3(a0, a1, a2, a3);
  o.y = pack4_e4m3(a4, a5, a6, a7);
  return o;
}

__device__ __forceinline__ uint32_t absmax8(const u32x4r& v) {
  uint32_t m = pk_umax16r(v[0] & 0x7fff7fffu, v[1] & 0x7fff7fffu);
  m = pk_umax16r(m, pk_umax16r(v[2] & 0x7fff7fffu, v[3] & 0x7fff7fffu));
  return umax32(m & 0xffffu, m >> 16);
}

// Rows of at most 4 * 8 * TPR elements: TPR lanes per row (TPR divides 64).
template <int DT, int TPR>
__global__ __launch_bounds__(kRThreads) void rowwise_quant_kernel(const uint16_t* x, int64_t rows,
                                                                  int64_t cols, int64_t ldx,
                                                                  float* dequant, uint8_t* codes,
                                                                  int64_t ldq) {
  constexpr int RPB = kRThreads / TPR;
  const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / TPR;
  const int t = threadIdx.x % TPR;
  const int nv = (int)(cols >> 3);
  const bool live = row < rows;
  const u32x4r* src = reinterpret_cast<const u32x4r*>(x + (live ? row : 0) * ldx);
  u32x4r v[4];
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int vi = t + i * TPR;
    v[i] = (live && vi < nv) ? src[vi] : u32x4r{0u, 0u, 0u, 0u};
    m = umax32(m, absmax8(v[i]));
  }
#pragma unroll
  for (int o = TPR / 2; o >= 1; o >>= 1) m = umax32(m, (uint32_t)__shfl_xor((int)m, o, kWave));
  if (!live) return;
  float qm, dq;
  rowwise_scales<DT>(m, &qm, &dq);
  uint8_t* dst = codes + row * ldq;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int vi = t + i * TPR;
    if (vi < nv) *reinterpret_cast<uint2*>(dst + 8 * vi) = quant8<DT>(v[i], qm);
  }
  if (t == 0) dequant[row] = dq;
}

// Rows longer than 2048 elements: one workgroup per row.
template <int DT>
__global__ __launch_bounds__(kRThreads) void rowwise_quant_long_kernel(const uint16_t* x,
                                                                       int64_t cols, int64_t ldx,
                                                                       float* dequant,
                                                                       uint8_t* codes,
                                                                       int64_t ldq) {
  const int64_t row = blockIdx.x;
  const int64_t nv = cols >> 3;
  const u32x4r* src = reinterpret_cast<const u32x4r*>(x + row * ldx);
  uint32_t m = 0;
  for (int64_t vi = threadIdx.x; vi < nv; vi += kRThreads) m = umax32(m, absmax8(src[vi]));
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = umax32(m, (uint32_t)__shfl_xor((int)m, o, kWave));
  __shared__ uint32_t wmax[kRThreads / kWave];
  if ((threadIdx.x & (kWave - 1)) == 0) wmax[threadIdx.x / kWave] = m;
  __syncthreads();
  m = umax32(umax32(wmax[0], wmax[1]), umax32(wmax[2], wmax[3]));
  float qm, dq;
  rowwise_scales<DT>(m, &qm, &dq);
  uint8_t* dst = codes + row * ldq;
  for (int64_t vi = threadIdx.x; vi < nv; vi += kRThreads)
    *reinterpret_cast<uint2*>(dst + 8 * vi) = quant8<DT>(src[vi], qm);
  if (threadIdx.x == 0) dequant[row] = dq;
}

// 16-bit transpose of each of `batch` (R, C) matrices: dst (C, R), row
// strides lds / ldd elements, batch strides bs / bd.  64 x 64 tiles.
__global__ __launch_bounds__(kRThreads) void transpose16_kernel(const uint16_t* src, uint16_t* dst,
                                                                int64_t R, int64_t C, int64_t lds,
                                                                int64_t ldd, int64_t bs,
                                                                int64_t bd) {
  __shared__ uint16_t tile[64][65];
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
  src += (int64_t)blockIdx.z * bs;
  dst += (int64_t)blockIdx.z * bd;
  for (int i = threadIdx.x; i < 64 * 64; i += kRThreads) {
    const int r = i >> 6, c = i & 63;
    if (r0 + r < R && c0 + c < C) tile[r][c] = src[(r0 + r) * lds + c0 + c];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * 64; i += kRThreads) {
    const int c = i >> 6, r = i & 63;
    if (r0 + r < R && c0 + c < C) dst[(c0 + c) * ldd + r0 + r] = tile[r][c];
  }
}

// The same for R, C and every stride a multiple of 8 elements and 16-byte
// aligned matrices: 16-byte loads of rows and stores of columns, each thread
// gathering the eight rows of a column from LDS.  A pitch of 66 elements
// (33 words) spreads the eight row octets over the banks.  V of 40 heads x
// 3600 x 128: 34 us element by element, 18 us here (74 MB; 15 us at the rate
// of a large copy).
__global__ __launch_bounds__(kRThreads) void transpose16_vec_kernel(
    const uint16_t* src, uint16_t* dst, int64_t R, int64_t C, int64_t lds, int64_t ldd, int64_t bs,
    int64_t bd) {
  __shared__ uint32_t tile[64][33];
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
  src += (int64_t)blockIdx.z * bs;
  dst += (int64_t)blockIdx.z * bd;
  const int k = threadIdx.x & 7;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int r = (threadIdx.x >> 3) + 32 * it;
    if (r0 + r < R && c0 + 8 * k < C) {
      const u32x4r v = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4r*>(src + (r0 + r) * lds + c0 + 8 * k));
#pragma unroll
      for (int i = 0; i < 4; ++i) tile[r][4 * k + i] = v[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int c = (threadIdx.x >> 3) + 32 * it;
    if (c0 + c < C && r0 + 8 * k < R) {
      u32x4r v;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t a = tile[8 * k + 2 * i][c >> 1], b = tile[8 * k + 2 * i + 1][c >> 1];
        v[i] = c & 1 ? (a >> 16) | (b & 0xffff0000u) : (a & 0xffffu) | (b << 16);
      }
      *reinterpret_cast<u32x4r*>(dst + (c0 + c) * ldd + r0 + 8 * k) = v;
    }
  }
}

// max that propagates NaN, as torch's softmax does
__device__ __forceinline__ float nmax(float a, float b) {
  return (a != a) ? a : ((b != b) ? b : fmaxf(a, b));
}

// Block-wide reductions of one value per thread (256 threads).
__device__ __forceinline__ float block_max(float v, float* red) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = nmax(v, __shfl_xor(v, o, kWave));
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = v;
  __syncthreads();
  return nmax(nmax(red[0], red[1]), nmax(red[2], red[3]));
}
__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, kWave);
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// s = bf16(raw * scale), -inf past the row's causal limit
__device__ __forceinline__ float score(uint32_t raw_bits, float scale, int64_t j, int64_t lim) {
  const float s = bf16_round(bf16_to_f32(raw_bits) * scale);
  return j <= lim ? s : -__builtin_inff();
}

// One workgroup per row r of `rows` raw score rows (bf16, `cols` each, row
// stride lds); query index q = r % sq gives the causal limit (keys j <= q).
__global__ __launch_bounds__(kRThreads) void softmax_rowquant_kernel(const uint16_t* scores,
                                                                     int64_t cols, int64_t lds,
                                                                     int64_t sq, int causal,
                                                                     float scale, float* dequant,
                                                                     uint8_t* codes, int64_t ldq) {
  __shared__ float red[kRThreads / kWave];
  const int64_t row = blockIdx.x;
  const int64_t lim = causal ? row % sq : cols;
  const uint16_t* src = scores + row * lds;
  const int64_t npair = cols >> 1;
  const uint32_t* s2 = reinterpret_cast<const uint32_t*>(src);
  float m = -__builtin_inff();
  for (int64_t i = threadIdx.x; i < npair; i += kRThreads) {
    const uint32_t w = s2[i];
    m = nmax(m, nmax(score(w & 0xffffu, scale, 2 * i, lim), score(w >> 16, scale, 2 * i + 1, lim)));
  }
  m = block_max(m, red);
  float sum = 0.0f;
  for (int64_t i = threadIdx.x; i < npair; i += kRThreads) {
    const uint32_t w = s2[i];
    sum += expf(score(w & 0xffffu, scale, 2 * i, lim) - m);
    sum += expf(score(w >> 16, scale, 2 * i + 1, lim) - m);
  }
  sum = block_sum(sum, red);
  // P's row maximum is bf16(1 / sum): its scales, then its codes
  float qm, dq;
  rowwise_scales<kInBf16>(f32_to_bf16_bits(1.0f / sum), &qm, &dq);
  uint8_t* dst = codes + row * ldq;
  for (int64_t i = threadIdx.x; i < npair; i += kRThreads) {
    const uint32_t w = s2[i];
    const float p0 = bf16_round(expf(score(w & 0xffffu, scale, 2 * i, lim) - m) / sum);
    const float p1 = bf16_round(expf(score(w >> 16, scale, 2 * i + 1, lim) - m) / sum);
    int pk;
    asm("v_cvt_pk_fp8_f32 %0, %1, %2" : "=v"(pk) : "v"(clamp_e4m3(p0 * qm)), "v"(clamp_e4m3(p1 * qm)));
    *reinterpret_cast<uint16_t*>(dst + 2 * i) = (uint16_t)pk;
  }
  if (threadIdx.x == 0) dequant[row] = dq;
}

// exp(x) for x <= 0 (or NaN) to about one fp32 ulp: x * log2(e) as a rounded
// product and its remainder, exp2 of the product by v_exp_f32, the remainder
// applied to first order.  Arguments below -200 give 0 (so does -inf, whose
// remainder would be NaN); NaN stays NaN.  expf's range reduction and
// overflow branches, which such arguments never need, are left out.
__device__ __forceinline__ float exp_nonpos(float x) {
  constexpr float kL = 1.4426950408889634f;              // fp32 log2(e)
  constexpr float kLlo = 1.925963033500011079e-08f;      // log2(e) - kL
  constexpr float kLn2 = 0.693147180559945309f;
  x = __builtin_elementwise_maximum(x, -200.0f);
  const float t = x * kL;
  const float lo = __builtin_fmaf(x, kLlo, __builtin_fmaf(x, kL, -t));
  const float e = __builtin_amdgcn_exp2f(t);
  return __builtin_fmaf(e, lo * kLn2, e);
}

// fp32 pair -> bf16 pair (one v_cvt_pk_bf16_f32, round to nearest even)
__device__ __forceinline__ uint32_t pack_bf16r(float lo, float hi) {
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
}

// The softmax rows that fit registers: WPR waves (1 or 4) hold one row, NV
// 16-byte vectors of eight scores per lane, so a row of up to 512 * NV * WPR
// scores is read once and every score is exponentiated once (the general
// kernel reads it three times and exponentiates twice).  Vector i of lane l
// of the row is vector l + 64 * WPR * i: whole lines per instruction, the
// codes stored eight bytes per lane.  One wave per row needs no LDS and no
// barrier; four waves combine their maxima and sums through LDS.
//
// Bound by the VALU about as much as by memory: ~25 instructions per score
// (two bf16 roundings, exp, the division, the conversion).  The quotient
// e / sum is e * r corrected by its remainder (r = 1 / sum once per row),
// three instructions against about ten of the IEEE sequence, which it equals
// but for the last bit of rare quotients, far below the bf16 rounding that
// follows.  P's code needs no clamp: p <= bf16(1 / sum), whose product with
// the row's multiplier is at most 425.6 (1 + 2^-9)^2 < 448.
// Measured at 40 heads x 3600 x 3600 scores (1.56 GB read and written):
// 0.39-0.42 ms (3.7-4.0 TB/s) against 1.41-1.49 ms of the general kernel.
template <int NV, int WPR, bool CAUSAL>
__global__ __launch_bounds__(kRThreads) void softmax_rowquant_vec_kernel(
    const uint16_t* scores, int64_t rows, int cols, int64_t lds, int64_t sq, float scale,
    float* dequant, uint8_t* codes, int64_t ldq) {
  constexpr int RPB = kRThreads / kWave / WPR;       // rows per workgroup
  constexpr int TPR = kWave * WPR;
  static_assert(WPR == 1 || WPR == kRThreads / kWave, "waves per row");
  __shared__ float red[2][kRThreads / kWave];
  const int64_t row = (int64_t)blockIdx.x * RPB + (WPR == 1 ? threadIdx.x / kWave : 0);
  // a whole wave leaves; with four waves per row the grid is exact
  if (WPR == 1 && row >= rows) return;
  const int t = WPR == 1 ? threadIdx.x % kWave : threadIdx.x;
  const int nv = cols >> 3;
  const int lim = CAUSAL ? (int)min(row % sq, (int64_t)cols) : cols;   // last visible key
  const u32x4r* src = reinterpret_cast<const u32x4r*>(scores + row * lds);
  u32x4r raw[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = t + i * TPR;
    raw[i] = vi < nv ? __builtin_nontemporal_load(src + vi) : u32x4r{0u, 0u, 0u, 0u};
  }
  const float ninf = -__builtin_inff();
  float s[NV][8];
  float m = ninf;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = t + i * TPR;
    const bool in = vi < nv;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = raw[i][j];
      const uint32_t r = pack_bf16r(bf16_to_f32(w & 0xffffu) * scale, bf16_to_f32(w >> 16) * scale);
      float a = bf16_to_f32(r & 0xffffu), b = bf16_to_f32(r >> 16);
      bool ina = in, inb = in;
      if constexpr (CAUSAL) {
        ina = ina && 8 * vi + 2 * j <= lim;
        inb = inb && 8 * vi + 2 * j + 1 <= lim;
      }
      a = ina ? a : ninf;
      b = inb ? b : ninf;
      s[i][2 * j] = a;
      s[i][2 * j + 1] = b;
      // a NaN score is caught by the sum: its exponential is NaN
      m = fmaxf(m, fmaxf(a, b));
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, kWave));
  if constexpr (WPR > 1) {
    if ((threadIdx.x & (kWave - 1)) == 0) red[0][threadIdx.x / kWave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
  }
  float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s[i][j] = exp_nonpos(s[i][j] - m);
      part[j & 3] += s[i][j];
    }
  float sum = (part[0] + part[1]) + (part[2] + part[3]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, kWave);
  if constexpr (WPR > 1) {
    if ((threadIdx.x & (kWave - 1)) == 0) red[1][threadIdx.x / kWave] = sum;
    __syncthreads();
    sum = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
  }
  const float r = 1.0f / sum;
  float qm, dq;
  rowwise_scales<kInBf16>(f32_to_bf16_bits(r), &qm, &dq);
  uint8_t* dst = codes + row * ldq;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = t + i * TPR;
    float p[8];
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      float q0 = s[i][j] * r, q1 = s[i][j + 1] * r;
      q0 = __builtin_fmaf(__builtin_fmaf(-q0, sum, s[i][j]), r, q0);
      q1 = __builtin_fmaf(__builtin_fmaf(-q1, sum, s[i][j + 1]), r, q1);
      const uint32_t b = pack_bf16r(q0, q1);
      p[j] = bf16_to_f32(b & 0xffffu) * qm;
      p[j + 1] = bf16_to_f32(b >> 16) * qm;
    }
    const u32x2r o = {pack4_e4m3(p[0], p[1], p[2], p[3]), pack4_e4m3(p[4], p[5], p[6], p[7])};
    if (vi < nv) __builtin_nontemporal_store(o, reinterpret_cast<u32x2r*>(dst + 8 * vi));
  }
  if (t == 0) dequant[row] = dq;
}

template <int NV, int WPR>
void launch_softmax_vec(const uint16_t* s, int64_t rows, int cols, int64_t lds, int64_t sq,
                        int causal, float scale, float* dq, uint8_t* codes, int64_t ldq,
                        hipStream_t st) {
  const int64_t rpb = kRThreads / kWave / WPR;
  const dim3 g((unsigned)((rows + rpb - 1) / rpb)), b(kRThreads);
  if (causal)
    hipLaunchKernelGGL((softmax_rowquant_vec_kernel<NV, WPR, true>), g, b, 0, st, s, rows, cols,
                       lds, sq, scale, dq, codes, ldq);
  else
    hipLaunchKernelGGL((softmax_rowquant_vec_kernel<NV, WPR, false>), g, b, 0, st, s, rows, cols,
                       lds, sq, scale, dq, codes, ldq);
}

int rw_check(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    rp_set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return RP_ERR_LAUNCH;
  }
  return RP_OK;
}

template <int DT>
int launch_rowwise(const uint16_t* x, int64_t rows, int64_t cols, int64_t ldx, float* dq,
                   uint8_t* codes, int64_t ldq, hipStream_t st) {
  const int64_t nv = cols / 8;
  if (nv > 256) {
    if (rows > 0x7fffffff) {
      rp_set_error("rowwise_quantize: too many rows");
      return RP_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(rowwise_quant_long_kernel<DT>, dim3((unsigned)rows), dim3(kRThreads), 0,
                       st, x, cols, ldx, dq, codes, ldq);
    return rw_check("rowwise_quant_long");
  }
  // lanes per row: the smallest power of two with at most 4 vectors each
  int tpr = 8;
  while (tpr < 64 && (nv + tpr - 1) / tpr > 4) tpr *= 2;
  const int64_t rpb = kRThreads / tpr;
  const int64_t blocks = (rows + rpb - 1) / rpb;
  if (blocks > 0x7fffffff) {
    rp_set_error("rowwise_quantize: too many rows");
    return RP_ERR_UNSUPPORTED;
  }
  const dim3 g((unsigned)blocks), b(kRThreads);
  switch (tpr) {
    case 8: hipLaunchKernelGGL((rowwise_quant_kernel<DT, 8>), g, b, 0, st, x, rows, cols, ldx, dq, codes, ldq); break;
    case 16: hipLaunchKernelGGL((rowwise_quant_kernel<DT, 16>), g, b, 0, st, x, rows, cols, ldx, dq, codes, ldq); break;
    case 32: hipLaunchKernelGGL((rowwise_quant_kernel<DT, 32>), g, b, 0, st, x, rows, cols, ldx, dq, codes, ldq); break;
    default: hipLaunchKernelGGL((rowwise_quant_kernel<DT, 64>), g, b, 0, st, x, rows, cols, ldx, dq, codes, ldq); break;
  }
  return rw_check("rowwise_quant");
}

}  // namespace
}  // namespace rp

using namespace rp;

extern "C" int rp_fp8_rowwise_quantize(const void* x, int x_dtype, int64_t rows, int64_t cols,
                                       int64_t ldx, float* dequant_out, uint8_t* codes,
                                       int64_t ldq, void* stream) {
  if (!x || !dequant_out || !codes) {
    rp_set_error("rowwise_quantize: null pointer");
    return RP_ERR_INVALID_ARGUMENT;
  }
  if (x_dtype != RP_DTYPE_BF16 && x_dtype != RP_DTYPE_F16) {
    rp_set_error("rowwise_quantize: unknown input dtype %d", x_dtype);
    return RP_ERR_INVALID_ARGUMENT;
  }
  if (rows <= 0 || cols <= 0 || ldx < cols || ldq < cols) {
    rp_set_error("rowwise_quantize: bad sizes rows=%lld cols=%lld ldx=%lld ldq=%lld",
                 (long long)rows, (long long)cols, (long long)ldx, (long long)ldq);
    return RP_ERR_INVALID_ARGUMENT;
  }
  if (cols % 8 != 0 || ldx % 8 != 0 || ldq % 8 != 0 ||
      reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(codes) % 8 != 0) {
    rp_set_error("rowwise_quantize: needs cols, ldx, ldq multiples of 8, x 16-byte and codes "
                 "8-byte aligned");
    return RP_ERR_UNSUPPORTED;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t* xp = static_cast<const uint16_t*>(x);
  if (x_dtype == RP_DTYPE_F16)
    return launch_rowwise<kInF16>(xp, rows, cols, ldx, dequant_out, codes, ldq, st);
  return launch_rowwise<kInBf16>(xp, rows, cols, ldx, dequant_out, codes, ldq, st);
}

extern "C" int rp_transpose16(const void* src, void* dst, int64_t batch, int64_t R, int64_t C,
                              int64_t lds, int64_t ldd, int64_t bs, int64_t bd, void* stream) {
  if (!src || !dst || batch <= 0 || R <= 0 || C <= 0 || lds < C || ldd < R) {
    rp_set_error("transpose16: bad arguments");
    return RP_ERR_INVALID_ARGUMENT;
  }
  const dim3 grid((unsigned)((C + 63) / 64), (unsigned)((R + 63) / 64), (unsigned)batch);
  if ((R + 63) / 64 > 65535 || batch > 65535 || (C + 63) / 64 > 0x7fffffff) {
    rp_set_error("transpose16: matrix or batch too large");
    return RP_ERR_UNSUPPORTED;
  }
  if (((R | C | lds | ldd | bs | bd) & 7) == 0 &&
      ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) == 0) {
    hipLaunchKernelGGL(transpose16_vec_kernel, grid, dim3(kRThreads), 0,
                       static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(src),
                       static_cast<uint16_t*>(dst), R, C, lds, ldd, bs, bd);
    return rw_check("transpose16");
  }
  hipLaunchKernelGGL(transpose16_kernel, grid, dim3(kRThreads), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint16_t*>(src), static_cast<uint16_t*>(dst), R, C, lds, ldd,
                     bs, bd);
  return rw_check("transpose16");
}

extern "C" int rp_fp8_softmax_rowwise_quantize(const void* scores, int64_t rows, int64_t cols,
                                               int64_t lds, int64_t sq, int causal, float scale,
                                               float* dequant_out, uint8_t* codes, int64_t ldq,
                                               void* stream) {
  if (!scores || !dequant_out || !codes) {
    rp_set_error("softmax_rowwise_quantize: null pointer");
    return RP_ERR_INVALID_ARGUMENT;
  }
  if (rows <= 0 || cols <= 0 || lds < cols || ldq < cols || sq <= 0 || !(scale == scale)) {
    rp_set_error("softmax_rowwise_quantize: bad arguments");
    return RP_ERR_INVALID_ARGUMENT;
  }
  if (cols % 2 != 0 || lds % 2 != 0 || ldq % 2 != 0 ||
      reinterpret_cast<uintptr_t>(scores) % 4 != 0 || reinterpret_cast<uintptr_t>(codes) % 2 != 0) {
    rp_set_error("softmax_rowwise_quantize: needs even cols, lds, ldq and aligned rows");
    return RP_ERR_UNSUPPORTED;
  }
  if (rows > 0x7fffffff) {
    rp_set_error("softmax_rowwise_quantize: too many rows");
    return RP_ERR_UNSUPPORTED;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t* sp = static_cast<const uint16_t*>(scores);
  // whole 16-byte vectors of scores and 8-byte vectors of codes, a row in
  // the registers of one wave (up to 4096 scores) or of four (up to 16384)
  const bool vec = cols % 8 == 0 && lds % 8 == 0 && ldq % 8 == 0 && cols <= 16384 &&
                   reinterpret_cast<uintptr_t>(scores) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(codes) % 8 == 0;
  if (vec) {
    auto go = [&](auto nv, auto wpr) {
      launch_softmax_vec<decltype(nv)::value, decltype(wpr)::value>(
          sp, rows, (int)cols, lds, sq, causal, scale, dequant_out, codes, ldq, st);
    };
    using std::integral_constant;
    if (cols <= 512) go(integral_constant<int, 1>{}, integral_constant<int, 1>{});
    else if (cols <= 1024) go(integral_constant<int, 2>{}, integral_constant<int, 1>{});
    else if (cols <= 2048) go(integral_constant<int, 4>{}, integral_constant<int, 1>{});
    else if (cols <= 3072) go(integral_constant<int, 6>{}, integral_constant<int, 1>{});
    else if (cols <= 4096) go(integral_constant<int, 8>{}, integral_constant<int, 1>{});
    else if (cols <= 8192) go(integral_constant<int, 4>{}, integral_constant<int, 4>{});
    else go(integral_constant<int, 8>{}, integral_constant<int, 4>{});
    return rw_check("softmax_rowquant");
  }
  hipLaunchKernelGGL(softmax_rowquant_kernel, dim3((unsigned)rows), dim3(kRThreads), 0, st, sp,
                     cols, lds, sq, causal ? 1 : 0, scale, dequant_out, codes, ldq);
  return rw_check("softmax_rowquant");
}
