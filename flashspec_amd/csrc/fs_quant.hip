// Affine per-block INT8 quantization kernels for gfx950, bit-exact with the float32 op
// sequence of reference src/flashspec/quant.py:141-158:
//     scale = max((mx - mn) / 255, 1e-8)        (IEEE float32 division)
//     zero  = clamp(rint(-mn / scale), 0, 255)
//     q     = clamp(rint(x / scale + zero), 0, 255),  stored as q - 128
// Contraction is disabled so `x / scale + zero` keeps its two roundings; division is the
// correctly rounded HIP default.  One wavefront quantizes one [rows, head_dim] group.

#include <type_traits>

#include "fs_common.h"

#pragma clang fp contract(off)

namespace fs {

template <typename Get>
__device__ __forceinline__ void quantize_group(const Get& get, int rows, int D, int8_t* dst, float* scale_out,
                                               int16_t* zero_out, int lane) {
  const int n = rows * D;
  float mn = __builtin_huge_valf(), mx = -__builtin_huge_valf();
  for (int r = 0; r < rows; ++r) {
    for (int d = lane; d < D; d += kWave) {
      const float x = get(r, d);
      mn = fminf(mn, x);
      mx = fmaxf(mx, x);
    }
  }
  mn = wave_min(mn);
  mx = wave_max(mx);
  const float scale = fmaxf((mx - mn) / 255.0f, 1.0e-8f);
  const float zero = fminf(fmaxf(__builtin_rintf(-mn / scale), 0.0f), 255.0f);
  for (int r = 0; r < rows; ++r) {
    for (int d = lane; d < D; d += kWave) {
      const float x = get(r, d);
      const float qv = fminf(fmaxf(__builtin_rintf(x / scale + zero), 0.0f), 255.0f);
      dst[(size_t)r * D + d] = (int8_t)((int)qv - 128);
    }
  }
  (void)n;
  if (lane == 0) {
    *scale_out = scale;
    *zero_out = (int16_t)zero;
  }
}

// FP8 E4M3 (OCP) per group, symmetric, no zero point:
//     scale = max(absmax / 448, 1e-8)        (IEEE float32 division)
//     code  = E4M3_RNE(clamp(x / scale, -448, 448))
// v_cvt_pk_fp8_f32 rounds to nearest even like torch's float8_e4m3fn conversion (checked over
// every code and every rounding tie on gfx950); the clamp keeps values in the finite range,
// where the instruction would otherwise give NaN past 464.  The zero point is written as 0.
template <typename Get>
__device__ __forceinline__ void quantize_group_fp8(const Get& get, int rows, int D, int8_t* dst, float* scale_out,
                                                   int16_t* zero_out, int lane) {
  float am = 0.0f;
  for (int r = 0; r < rows; ++r) {
    for (int d = lane; d < D; d += kWave) am = fmaxf(am, fabsf(get(r, d)));
  }
  am = wave_max(am);
  const float scale = fmaxf(am / 448.0f, 1.0e-8f);
  for (int r = 0; r < rows; ++r) {
    for (int d = lane; d < D; d += kWave) {
      const float y = fminf(fmaxf(get(r, d) / scale, -448.0f), 448.0f);
      dst[(size_t)r * D + d] = (int8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(y, y, 0, false) & 0xff);
    }
  }
  if (lane == 0) {
    *scale_out = scale;
    if (zero_out) *zero_out = 0;
  }
}

// Affine INT8 per channel over a group of `rows` tokens: quantize_group's float32 op sequence
// applied to each channel column (one scale / zero point per channel, D of each per group).
template <typename Get>
__device__ __forceinline__ void quantize_channel_group(const Get& get, int rows, int D, int8_t* dst,
                                                       float* scale_out, int16_t* zero_out, int lane) {
  for (int d = lane; d < D; d += kWave) {
    float mn = __builtin_huge_valf(), mx = -__builtin_huge_valf();
    for (int r = 0; r < rows; ++r) {
      const float x = get(r, d);
      mn = fminf(mn, x);
      mx = fmaxf(mx, x);
    }
    const float scale = fmaxf((mx - mn) / 255.0f, 1.0e-8f);
    const float zero = fminf(fmaxf(__builtin_rintf(-mn / scale), 0.0f), 255.0f);
    for (int r = 0; r < rows; ++r) {
      const float qv = fminf(fmaxf(__builtin_rintf(get(r, d) / scale + zero), 0.0f), 255.0f);
      dst[(size_t)r * D + d] = (int8_t)((int)qv - 128);
    }
    scale_out[d] = scale;
    zero_out[d] = (int16_t)zero;
  }
}

// Symmetric absmax INT8 over a group of `rows` tokens, one scale per token row:
// scale = max(absmax / 127, 1e-8), q = clamp(rint(x / scale), -127, 127), zero point 128.
template <typename Get>
__device__ __forceinline__ void quantize_token_group(const Get& get, int rows, int D, int8_t* dst, float* scale_out,
                                                     int16_t* zero_out, int lane) {
  for (int r = 0; r < rows; ++r) {
    float am = 0.0f;
    for (int d = lane; d < D; d += kWave) am = fmaxf(am, fabsf(get(r, d)));
    am = wave_max(am);
    const float s = fmaxf(am / 127.0f, 1.0e-8f);
    for (int d = lane; d < D; d += kWave)
      dst[(size_t)r * D + d] = (int8_t)(int)fminf(fmaxf(__builtin_rintf(get(r, d) / s), -127.0f), 127.0f);
    if (lane == 0) {
      scale_out[r] = s;
      zero_out[r] = 128;
    }
  }
}

// A launch's waves take the groups [first, groups) in order, one each (launch_ranges).
__device__ __forceinline__ int64_t wave_in_grid() { return ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave; }

// Group formats of the block / page quantizers.
enum GroupFormat : int {
  kGfAffine = 0,   // affine INT8, one scale / zero per group
  kGfFp8 = 1,      // FP8 E4M3, one scale per group, zero 0
  kGfChannel = 2,  // affine INT8, one scale / zero per channel of the group
  kGfToken = 3,    // symmetric INT8, one scale per row of the group, zero 128
};

// scale / zero entries of one group
template <int GF>
__host__ __device__ constexpr int group_params(int rows, int D) {
  return GF == kGfChannel ? D : (GF == kGfToken ? rows : 1);
}

template <int GF, typename Get>
__device__ __forceinline__ void quantize_any_group(const Get& get, int rows, int D, int8_t* dst, float* scale,
                                                   int16_t* zero, int64_t grp, int lane) {
  scale += (size_t)grp * group_params<GF>(rows, D);
  if (zero) zero += (size_t)grp * group_params<GF>(rows, D);
  if constexpr (GF == kGfFp8)
    quantize_group_fp8(get, rows, D, dst, scale, zero, lane);
  else if constexpr (GF == kGfChannel)
    quantize_channel_group(get, rows, D, dst, scale, zero, lane);
  else if constexpr (GF == kGfToken)
    quantize_token_group(get, rows, D, dst, scale, zero, lane);
  else
    quantize_group(get, rows, D, dst, scale, zero, lane);
}

// ---- vectorized group quantizer --------------------------------------------------------------
// Same arithmetic as the element-wise groups above, for a group of `rows` contiguous source rows of
// D values with D % 8 == 0, held in registers: read once from HBM with 16-byte loads (non-temporal:
// the source is read exactly once) and written back as 8-byte packed stores.  Lane l holds, of every
// chunk c < CH, the 8 values at c * step + 8 l (LaneMap).  With one parameter per group a chunk is
// 512 values in a row.  With one per channel or row a chunk is as many whole rows as 64 lanes hold,
// so that a lane keeps its 8 channels in every chunk and a row stays in neighbouring lanes.  Lanes
// and chunks past the group's n values hold values of the group again (of the same channels), which
// leaves every extreme as it is, and store nothing.
//
// Bound by HBM: 2 bytes read and 1 written per 16-bit value.  The element-wise kernels read every
// value twice (once for the range) and divided it with the 10-instruction IEEE sequence.  Measured on
// MI355X, from_dense of bf16 [4, 32, 2039, 128] to shuffled FP8 pages, the whole call: 174 us (2 x 78 us
// of element-wise kernels) -> 76.8 us with a launch per tensor (54 us with both in one, PagesSource).

typedef uint32_t q_u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ q_u32x4_t nt_load16(const void* p) {
  return __builtin_nontemporal_load((const q_u32x4_t*)p);
}

__device__ __forceinline__ void nt_store8(int8_t* p, uint32_t a, uint32_t b) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  __builtin_nontemporal_store(u32x2{a, b}, (u32x2*)p);
}

__device__ __forceinline__ void load8(const float* p, float* f) {
  const q_u32x4_t a = nt_load16(p), b = nt_load16(p + 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[i] = __uint_as_float(a[i]);
    f[4 + i] = __uint_as_float(b[i]);
  }
}

__device__ __forceinline__ void load8(const __half* p, float* f) {
  const q_u32x4_t a = nt_load16(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __half2float(__ushort_as_half((unsigned short)(a[i] & 0xffffu)));
    f[2 * i + 1] = __half2float(__ushort_as_half((unsigned short)(a[i] >> 16)));
  }
}

__device__ __forceinline__ void load8(const __hip_bfloat16* p, float* f) {
  const q_u32x4_t a = nt_load16(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(a[i] << 16);
    f[2 * i + 1] = __uint_as_float(a[i] & 0xffff0000u);
  }
}


// Chunks that a group running as CH chunks surely fills (group_chunks rounds 5, 7 and 9 to 15 up).
constexpr int sure_chunks(int CH) { return CH <= 4 ? CH - 1 : (CH == 6 ? 4 : (CH == 8 ? 6 : 8)); }

// Whether the lane has values of its own in chunk c, at e.
template <int GF, int CH>
__device__ __forceinline__ bool has_values(int c, int e, int n) {
  return (GF != kGfChannel && GF != kGfToken && c < sure_chunks(CH)) || e < n;
}

// Quantize CH chunks of 8 values held by this lane and store them as packed bytes.
template <int CH, bool RCP>
__device__ __forceinline__ void store_chunks(const float (&x)[CH][8], float scale, float rcp, float zero,
                                             int8_t* dst, int n, int lane) {
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    uint32_t w[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float qd = RCP ? div_by_scale(x[c][i], scale, rcp) : x[c][i] / scale;
      const float qv = fminf(fmaxf(__builtin_rintf(qd + zero), 0.0f), 255.0f);
      // qv is an integer in [0, 255]: the byte conversion is exact
      w[i / 4] = __builtin_amdgcn_cvt_pk_u8_f32(qv, i % 4, w[i / 4]);
    }
    // stored as q - 128: flip the top bit of every byte
    const int e = c * 512 + lane * 8;
    if (has_values<kGfAffine, CH>(c, e, n)) nt_store8(dst + e, w[0] ^ 0x80808080u, w[1] ^ 0x80808080u);
  }
}

// One lane's share of a vectorized group as loaded: CH chunks of 8 source values (16 bytes each
// for 16-bit types, 32 for fp32); values past the group's valid ones are zero.
template <int CH, typename XT>
struct RawGroup {
  static constexpr int kWords = sizeof(XT) == 4 ? 2 * CH : CH;
  q_u32x4_t w[kWords];
};

struct LaneMap {
  int step;   // values per chunk
  int first;  // the lane's first value in a chunk (n or more: the lane holds none of its own)
  int alt;    // what it holds where it has none
  int lpr, rpw;  // row formats: lanes per row, rows per chunk
  int row, col;  // the lane's row within a chunk and lane within the row
};

template <int GF>
__device__ __forceinline__ LaneMap lane_map(int n, int D, int lane) {
  LaneMap m{512, lane * 8, 0, 0, 0, 0, 0};
  if constexpr (GF == kGfChannel || GF == kGfToken) {
    m.lpr = D / 8;
    m.rpw = kWave / m.lpr;
    m.row = lane / m.lpr;
    m.col = lane - m.row * m.lpr;
    m.step = m.rpw * D;
    m.first = m.row < m.rpw ? lane * 8 : n;
    m.alt = m.col * 8;
  }
  return m;
}

// `valid`: the group's values that exist in the source, `n` its values with the zero rows.
template <int GF, int CH, typename XT>
__device__ __forceinline__ void load_raw(RawGroup<CH, XT>& r, const XT* src, int valid, int n, const LaneMap& m) {
  constexpr int per = RawGroup<CH, XT>::kWords / CH;  // 16-byte words per chunk
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int at = c * m.step + m.first;
    const int e = has_values<GF, CH>(c, at, n) ? at : m.alt;
    const bool ok = e < valid;
#pragma unroll
    for (int i = 0; i < per; ++i)
      r.w[c * per + i] = ok ? nt_load16((const char*)(src + e) + 16 * i) : q_u32x4_t{0u, 0u, 0u, 0u};
  }
}

__device__ __forceinline__ void unpack8(const q_u32x4_t* w, const float*, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[i] = __uint_as_float(w[0][i]);
    f[4 + i] = __uint_as_float(w[1][i]);
  }
}

__device__ __forceinline__ void unpack8(const q_u32x4_t* w, const __half*, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __half2float(__ushort_as_half((unsigned short)(w[0][i] & 0xffffu)));
    f[2 * i + 1] = __half2float(__ushort_as_half((unsigned short)(w[0][i] >> 16)));
  }
}

__device__ __forceinline__ void unpack8(const q_u32x4_t* w, const __hip_bfloat16*, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(w[0][i] << 16);
    f[2 * i + 1] = __uint_as_float(w[0][i] & 0xffff0000u);
  }
}

// Quantizes a group held in registers (quantize_group's float32 op sequence).
template <int CH>
__device__ __forceinline__ void quantize_regs(const float (&x)[CH][8], int8_t* dst, float* scale_out,
                                              int16_t* zero_out, int n, int lane) {
  float mn = __builtin_huge_valf(), mx = -__builtin_huge_valf();
#pragma unroll
  for (int c = 0; c < CH; ++c) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      mn = fminf(mn, x[c][i]);
      mx = fmaxf(mx, x[c][i]);
    }
  }
  // min / max are exact whatever the order; lane swaps and DPP keep them off the LDS
  mn = wave_min_valu(mn);
  mx = wave_max_valu(mx);
  const float scale = fmaxf((mx - mn) / 255.0f, 1.0e-8f);
  const float zero = fminf(fmaxf(__builtin_rintf(-mn / scale), 0.0f), 255.0f);
  const float rcp = 1.0f / scale;  // correctly rounded
  // |x| <= max(|mn|, |mx|) for every value of the group, and rounding is monotonic: if the
  // largest product is finite, all are (wave-uniform test)
  if (__builtin_isfinite(fmaxf(fabsf(mn), fabsf(mx)) * rcp))
    store_chunks<CH, true>(x, scale, rcp, zero, dst, n, lane);
  else
    store_chunks<CH, false>(x, scale, rcp, zero, dst, n, lane);
  if (lane == 0) {
    *scale_out = scale;
    *zero_out = (int16_t)zero;
  }
}

// FP8 E4M3 (quantize_group_fp8's op sequence).  The quotient takes its value's sign back: the
// correction step loses the sign of a zero quotient, and FP8 codes keep it.
template <int CH, bool RCP>
__device__ __forceinline__ void store_chunks_fp8(const float (&x)[CH][8], float scale, float rcp, int8_t* dst, int n,
                                                 int lane) {
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float qd = RCP ? __builtin_copysignf(div_by_scale(x[c][i], scale, rcp), x[c][i]) : x[c][i] / scale;
      y[i] = fminf(fmaxf(qd, -448.0f), 448.0f);
    }
    int w[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      w[j] = __builtin_amdgcn_cvt_pk_fp8_f32(y[4 * j], y[4 * j + 1], 0, false);
      w[j] = __builtin_amdgcn_cvt_pk_fp8_f32(y[4 * j + 2], y[4 * j + 3], w[j], true);
    }
    const int e = c * 512 + lane * 8;
    if (has_values<kGfFp8, CH>(c, e, n)) *(uint2*)(dst + e) = make_uint2((uint32_t)w[0], (uint32_t)w[1]);
  }
}

template <int CH>
__device__ __forceinline__ void quantize_regs_fp8(const float (&x)[CH][8], int8_t* dst, float* scale_out,
                                                  int16_t* zero_out, int n, int lane) {
  float am = 0.0f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
#pragma unroll
    for (int i = 0; i < 8; ++i) am = fmaxf(am, fabsf(x[c][i]));
  }
  am = wave_max_valu(am);
  const float scale = fmaxf(am / 448.0f, 1.0e-8f);
  const float rcp = 1.0f / scale;
  if (__builtin_isfinite(am * rcp))  // wave-uniform, as in quantize_regs
    store_chunks_fp8<CH, true>(x, scale, rcp, dst, n, lane);
  else
    store_chunks_fp8<CH, false>(x, scale, rcp, dst, n, lane);
  if (lane == 0) {
    *scale_out = scale;
    if (zero_out) *zero_out = 0;
  }
}

// Per channel (quantize_channel_group's op sequence): each lane reduces its 8 channels over its own
// rows, then over the lanes that hold the same channels.
template <int CH, bool RCP>
__device__ __forceinline__ void store_chunks_channel(const float (&x)[CH][8], const float (&scale)[8],
                                                     const float (&rcp)[8], const float (&zero)[8], int8_t* dst, int n,
                                                     const LaneMap& m) {
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    uint32_t w[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float qd = RCP ? div_by_scale(x[c][i], scale[i], rcp[i]) : x[c][i] / scale[i];
      const float qv = fminf(fmaxf(__builtin_rintf(qd + zero[i]), 0.0f), 255.0f);
      w[i / 4] = __builtin_amdgcn_cvt_pk_u8_f32(qv, i % 4, w[i / 4]);
    }
    const int e = c * m.step + m.first;
    if (e < n) nt_store8(dst + e, w[0] ^ 0x80808080u, w[1] ^ 0x80808080u);
  }
}

template <int CH>
__device__ __forceinline__ void quantize_regs_channel(const float (&x)[CH][8], int8_t* dst, float* scale_out,
                                                      int16_t* zero_out, int n, const LaneMap& m) {
  float mn[8], mx[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    mn[i] = __builtin_huge_valf();
    mx[i] = -__builtin_huge_valf();
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      mn[i] = fminf(mn[i], x[c][i]);
      mx[i] = fmaxf(mx[i], x[c][i]);
    }
  }
  if ((m.lpr & (m.lpr - 1)) == 0) {
    for (int off = m.lpr; off < kWave; off <<= 1) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        mn[i] = fminf(mn[i], __shfl_xor(mn[i], off, kWave));
        mx[i] = fmaxf(mx[i], __shfl_xor(mx[i], off, kWave));
      }
    }
  } else {
    float own_mn[8], own_mx[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      own_mn[i] = mn[i];
      own_mx[i] = mx[i];
    }
    for (int r = 0; r < m.rpw; ++r) {  // the lanes of every row in turn
      const int from = r * m.lpr + m.col;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        mn[i] = fminf(mn[i], __shfl(own_mn[i], from, kWave));
        mx[i] = fmaxf(mx[i], __shfl(own_mx[i], from, kWave));
      }
    }
  }
  float scale[8], zero[8], rcp[8];
  bool finite = true;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    scale[i] = fmaxf((mx[i] - mn[i]) / 255.0f, 1.0e-8f);
    zero[i] = fminf(fmaxf(__builtin_rintf(-mn[i] / scale[i]), 0.0f), 255.0f);
    rcp[i] = 1.0f / scale[i];
    finite = finite && __builtin_isfinite(fmaxf(fabsf(mn[i]), fabsf(mx[i])) * rcp[i]);
  }
  if (__all(finite))
    store_chunks_channel<CH, true>(x, scale, rcp, zero, dst, n, m);
  else
    store_chunks_channel<CH, false>(x, scale, rcp, zero, dst, n, m);
  if (m.row == 0) {
    float4* so = (float4*)(scale_out + 8 * m.col);
    so[0] = make_float4(scale[0], scale[1], scale[2], scale[3]);
    so[1] = make_float4(scale[4], scale[5], scale[6], scale[7]);
    uint32_t z[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) z[i] = (uint32_t)(int)zero[2 * i] | ((uint32_t)(int)zero[2 * i + 1] << 16);
    *(uint4*)(zero_out + 8 * m.col) = make_uint4(z[0], z[1], z[2], z[3]);
  }
}

// Symmetric per row (quantize_token_group's op sequence): a row's lanes are neighbours.
template <int CH, bool RCP>
__device__ __forceinline__ void store_chunks_token(const float (&x)[CH][8], const float (&scale)[CH],
                                                   const float (&rcp)[CH], int8_t* dst, int n, const LaneMap& m) {
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    uint32_t w[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float qd = RCP ? div_by_scale(x[c][i], scale[c], rcp[c]) : x[c][i] / scale[c];
      const float qv = fminf(fmaxf(__builtin_rintf(qd), -127.0f), 127.0f);
      w[i / 4] = __builtin_amdgcn_cvt_pk_u8_f32(qv + 128.0f, i % 4, w[i / 4]);  // 1 .. 255: exact
    }
    const int e = c * m.step + m.first;
    if (e < n) nt_store8(dst + e, w[0] ^ 0x80808080u, w[1] ^ 0x80808080u);
  }
}

template <int CH>
__device__ __forceinline__ void quantize_regs_token(const float (&x)[CH][8], int8_t* dst, float* scale_out,
                                                    int16_t* zero_out, int n, const LaneMap& m) {
  float scale[CH], rcp[CH];
  bool finite = true;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    float am = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) am = fmaxf(am, fabsf(x[c][i]));
    if ((m.lpr & (m.lpr - 1)) == 0) {
      for (int off = 1; off < m.lpr; off <<= 1) am = fmaxf(am, __shfl_xor(am, off, kWave));
    } else {
      const float own = am;
      for (int j = 0; j < m.lpr; ++j) am = fmaxf(am, __shfl(own, (m.row < m.rpw ? m.row : 0) * m.lpr + j, kWave));
    }
    scale[c] = fmaxf(am / 127.0f, 1.0e-8f);
    rcp[c] = 1.0f / scale[c];
    finite = finite && __builtin_isfinite(am * rcp[c]);
  }
  if (__all(finite))
    store_chunks_token<CH, true>(x, scale, rcp, dst, n, m);
  else
    store_chunks_token<CH, false>(x, scale, rcp, dst, n, m);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    if (m.col == 0 && c * m.step + m.first < n) {
      const int r = c * m.rpw + m.row;
      scale_out[r] = scale[c];
      zero_out[r] = 128;
    }
  }
}

template <int GF, int CH>
__device__ __forceinline__ void quantize_any_regs(const float (&x)[CH][8], int8_t* dst, float* scale, int16_t* zero,
                                                  int n, const LaneMap& m, int lane) {
  if constexpr (GF == kGfFp8)
    quantize_regs_fp8<CH>(x, dst, scale, zero, n, lane);
  else if constexpr (GF == kGfChannel)
    quantize_regs_channel<CH>(x, dst, scale, zero, n, m);
  else if constexpr (GF == kGfToken)
    quantize_regs_token<CH>(x, dst, scale, zero, n, m);
  else
    quantize_regs<CH>(x, dst, scale, zero, n, lane);
}

template <int CH, typename XT>
__device__ __forceinline__ void unpack_group(const RawGroup<CH, XT>& r, float (&x)[CH][8]) {
  constexpr int per = RawGroup<CH, XT>::kWords / CH;
#pragma unroll
  for (int c = 0; c < CH; ++c) unpack8(&r.w[c * per], (const XT*)nullptr, x[c]);
}

// Where group `grp` of a vectorized quantize pass reads and writes.
template <typename XT>
struct GroupRef {
  const XT* src;
  int valid_rows;
  int8_t* dst;
  float* scale;
  int16_t* zero;
};

// One group per wave, the grid as large as that takes: the dispatcher's waves then cover each other's
// loads, and workgroups that end early are replaced at once.  Looping over groups in 4096 workgroups
// with the next group's loads in flight held 92 registers a lane and kept the waves in step: measured
// on MI355X, from_dense's launch of fp16 [8, 32, 4096, 128] K and V (6 rotated tensors), with cached
// stores 163 us, with non-temporal ones 150.5; 32768 workgroups without a loop
// (44 registers) 129.6, 6.2 TB/s.
template <int GF, int CH, typename XT, typename Map>
__device__ __forceinline__ void quantize_group_vec(const Map& map, int64_t first, int64_t groups, int rows, int D) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t grp = first + wave_in_grid();
  if (grp >= groups) return;
  const int n = rows * D;
  const LaneMap m = lane_map<GF>(n, D, lane);
  const GroupRef<XT> ref = map(grp);
  RawGroup<CH, XT> raw;
  load_raw<GF>(raw, ref.src, ref.valid_rows * D, n, m);
  float x[CH][8];
  unpack_group(raw, x);
  quantize_any_regs<GF, CH>(x, ref.dst, ref.scale, ref.zero, n, m, lane);
}

// Chunks of a group of `rows` rows when the vectorized quantizers apply (rounded up to an instantiated
// count), else 0.  `by_row`: the formats whose chunks are whole rows (kGfChannel, kGfToken).
static int group_chunks(int64_t rows, int D, bool by_row) {
  if (D % 8 != 0 || rows * D > 16 * 512 || (by_row && D > 512)) return 0;
  const int64_t per = by_row ? kWave / (D / 8) : 512;
  const int64_t ch = ((by_row ? rows : rows * D) + per - 1) / per;
  return ch <= 4 ? (int)ch : (ch <= 6 ? 6 : (ch <= 8 ? 8 : (ch <= 16 ? 16 : 0)));
}

// Whether scale / zero can be stored 16 bytes at a time (kGfChannel stores them so).
static bool wide_params(const void* scale, const void* zero) {
  return ((uintptr_t)scale % 16) == 0 && ((uintptr_t)zero % 16) == 0;
}

// Chunks of 512 values per group when the vectorized append applies, else 0.
__host__ __device__ constexpr int vec_chunks(int rows, int D) {
  return (D % 8 == 0 && (rows * D) % 512 == 0 && rows * D / 512 <= 8) ? rows * D / 512 : 0;
}

// x [outer, S, D] -> values [outer, nb, bs, D]; groups (o, block), vectorized.
template <int GF, int CH, typename XT>
__global__ void __launch_bounds__(256)
quantize_blocks_vec_kernel(const XT* x, int64_t first, int64_t groups, int S, int D, int bs, int nb, int8_t* values,
                           float* scale, int16_t* zero) {
  const int per = group_params<GF>(bs, D);
  auto map = [=](int64_t grp) {
    const int64_t o = grp / nb;
    const int blk = (int)(grp - o * nb);
    return GroupRef<XT>{x + ((size_t)o * S + (size_t)blk * bs) * D, min(S - blk * bs, bs), values + (size_t)grp * bs * D,
                        scale + (size_t)grp * per, zero ? zero + (size_t)grp * per : nullptr};
  };
  quantize_group_vec<GF, CH, XT>(map, first, groups, bs, D);
}

struct PageStore {
  int8_t* values;
  float* scale;
  int16_t* zero;
};

// Dense K and V [B, H, S, D] -> page stores [P, H, page, D] (v null: K alone): physical page j holds
// batch-major logical page page_src[j]; without a list it holds page j, or with `interleaved` page
// (j % B) * nbps + j / B.  The launch also writes what the cache needs beside the pages, where asked
// for: table[o] = the physical page of logical page o, and every request's length S.  One launch for
// both tensors and both lists saves the gaps and the tails of five: measured on MI355X, from_dense
// of fp16 [8, 32, 4096, 128] 160.7 -> 129.4 us (with one group per wave), of bf16 [4, 32, 2039, 128] to shuffled FP8 pages
// 76.8 -> 55 us (torch.randperm's own launches remain).
template <typename XT>
struct PagesSource {
  const XT* k;
  const XT* v;
  PageStore ks, vs;
  const int64_t* page_src;
  int64_t* table;
  int64_t* lengths;
  int64_t P;
  int B, H, S, D, page, nbps, interleaved;
};

// Where group grp (K groups first, then V's; heads innermost) reads and writes.  I: index type; the
// vectorized kernel takes 32 bits (the host keeps P * H < 2^31), a 64-bit division per group having
// sat on the critical path to the next group's loads.
template <int GF, typename I, typename XT>
__device__ __forceinline__ GroupRef<XT> page_group(const PagesSource<XT>& s, int64_t group, int lane) {
  const I per = (I)s.P * (I)s.H;
  I g = sizeof(I) == 4 ? (I)__builtin_amdgcn_readfirstlane((int)group) : (I)group;  // one group per wave
  const bool second = g >= per;
  if (second) g -= per;
  const I j = g / (I)s.H;
  const int h = (int)(g - j * (I)s.H);
  const I o = s.page_src ? (I)s.page_src[j] : (s.interleaved ? (j % (I)s.B) * (I)s.nbps + j / (I)s.B : j);
  const I b = o / (I)s.nbps;
  const int lb = (int)(o - b * (I)s.nbps);
  if (h == 0 && !second && lane == 0) {
    if (s.table) s.table[o] = (int64_t)j;
    if (s.lengths && lb == 0) s.lengths[b] = s.S;
  }
  const PageStore st = second ? s.vs : s.ks;
  const int params = group_params<GF>(s.page, s.D);
  return GroupRef<XT>{(second ? s.v : s.k) + ((size_t)(b * (I)s.H + (I)h) * s.S + (size_t)lb * s.page) * s.D,
                      min(s.S - lb * s.page, s.page), st.values + (size_t)g * s.page * s.D,
                      st.scale + (size_t)g * params, st.zero ? st.zero + (size_t)g * params : nullptr};
}

template <int GF, int CH, typename XT>
__global__ void __launch_bounds__(256)
quantize_pages_vec_kernel(const PagesSource<XT> s, int64_t first, int64_t groups) {
  const int lane = threadIdx.x & (kWave - 1);
  auto map = [&](int64_t grp) { return page_group<GF, unsigned>(s, grp, lane); };
  quantize_group_vec<GF, CH, XT>(map, first, groups, s.page, s.D);
}

// x [outer, S, D] -> values [outer, nb, bs, D]; group = (o, block); rows past S read as 0.
// GF: group format (GroupFormat); with kGfFp8 zero may be null, with kGfChannel scale and zero
// hold D entries per group.
template <typename XT, int GF = kGfAffine>
__global__ void __launch_bounds__(256)
quantize_blocks_kernel(const XT* x, int64_t first, int64_t groups, int S, int D, int bs, int nb, int8_t* values,
                       float* scale, int16_t* zero) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t grp = first + wave_in_grid();
  if (grp >= groups) return;
  const int64_t o = grp / nb;
  const int blk = (int)(grp - o * nb);
  const XT* src = x + ((size_t)o * S) * D;
  auto get = [&](int r, int d) -> float {
    const int s = blk * bs + r;
    return s < S ? to_f32(src[(size_t)s * D + d]) : 0.0f;
  };
  quantize_any_group<GF>(get, bs, D, values + (size_t)grp * bs * D, scale, zero, grp, lane);
}

// quantize_pages_vec_kernel for any sizes and addresses; rows past S read as 0.
template <typename XT, int GF>
__global__ void __launch_bounds__(256)
quantize_pages_kernel(const PagesSource<XT> s, int64_t first, int64_t groups) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t grp = first + wave_in_grid();
  if (grp >= groups) return;
  const GroupRef<XT> ref = page_group<GF, int64_t>(s, grp, lane);
  auto get = [&](int r, int d) -> float { return r < ref.valid_rows ? to_f32(ref.src[(size_t)r * s.D + d]) : 0.0f; };
  quantize_any_group<GF>(get, s.page, s.D, ref.dst, ref.scale, ref.zero, 0, lane);
}

// Rewrite listed pages (see fs_update_pages_i8).
template <typename XT>
__global__ void __launch_bounds__(256)
update_pages_kernel(const int8_t* in_values, const float* in_scale, const int16_t* in_zero, int64_t in_pages,
                    int in_qb, int8_t* out_values, float* out_scale, int16_t* out_zero, const int64_t* pages,
                    const uint8_t* fresh, int64_t first, int64_t groups, const int32_t* row_src, const XT* src,
                    int src_tokens, int H, int page, int D) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t grp = first + wave_in_grid();
  if (grp >= groups) return;
  const int64_t i = grp / H;
  const int h = (int)(grp - i * H);
  const int64_t pg = pages ? pages[i] : i;
  const bool from_zero = pg >= in_pages || (fresh != nullptr && fresh[i] != 0);
  const int nqb_in = page / in_qb;
  const int32_t* rs = row_src + (size_t)i * page;
  auto get = [&](int r, int d) -> float {
    const int32_t si = rs[r];
    if (si >= 0) {
      const int n = si / src_tokens;
      const int t = si - n * src_tokens;
      return to_f32(src[(((size_t)n * H + h) * src_tokens + t) * D + d]);
    }
    if (from_zero) return 0.0f;
    const int qb = r / in_qb;
    const int qo = r - qb * in_qb;
    const int64_t sidx = (pg * H + h) * nqb_in + qb;
    const int u = (int)in_values[((size_t)sidx * in_qb + qo) * D + d] + 128;
    return ((float)u - (float)in_zero[sidx]) * in_scale[sidx];
  };
  const int64_t og = pg * H + h;
  quantize_group(get, page, D, out_values + (size_t)og * page * D, out_scale + og, out_zero + og, lane);
}

// Prompt admission (see fs_write_prompt_i8): one request's K and V rows [H, src_tokens, D] into the
// pages of a store, group = (K or V, logical page, head).  The page ids travel in the launch's
// arguments, so admitting a prompt needs no device copy of its page list: the reference-shaped path
// (fs_update_pages_i8, one launch per tensor) uploaded a page list, a row map and a flag per page
// for each tensor, six blocking copies of ~3.6 us, and read every source value twice.  Bound by HBM
// (read 2 B, write 1 B per value).  Measured on MI355X, 3001 tokens, H32 D128 fp16, 49 MB read and
// 25 MB written: the whole add_request 298 us -> 17.1 us (two element-wise kernels of 56 us before).
constexpr int kPromptPages = 896;  // page ids per launch: 3.5 KiB of the 4 KiB argument limit
struct PromptPages {
  int32_t id[kPromptPages];
};

template <typename XT>
struct PromptSource {
  const XT* k;
  const XT* v;
  PageStore ks, vs;
  int H, src_tokens, length, D, page;
  int first, n;  // logical pages [first, first + n)
};

// Group grp of a prompt's pages: K groups first, then V groups, heads innermost (a page's heads are
// consecutive in the store).
template <typename XT>
__device__ __forceinline__ GroupRef<XT> prompt_group(const PromptSource<XT>& s, const PromptPages& pages,
                                                     int64_t grp) {
  const unsigned per = (unsigned)s.n * (unsigned)s.H;
  unsigned g = __builtin_amdgcn_readfirstlane((unsigned)grp);  // one group per wave
  const bool second = g >= per;
  if (second) g -= per;
  const unsigned i = g / (unsigned)s.H;
  const unsigned h = g - i * (unsigned)s.H;
  const int row0 = (s.first + (int)i) * s.page;
  const PageStore st = second ? s.vs : s.ks;
  const size_t og = (size_t)pages.id[i] * s.H + h;
  return GroupRef<XT>{(second ? s.v : s.k) + ((size_t)h * s.src_tokens + row0) * s.D,
                      min(s.length - row0, s.page), st.values + og * s.page * s.D, st.scale + og, st.zero + og};
}

template <int CH, typename XT>
__global__ void __launch_bounds__(256)
prompt_pages_vec_kernel(const PromptSource<XT> s, int64_t first, int64_t groups, const PromptPages pages) {
  auto map = [&](int64_t grp) { return prompt_group(s, pages, grp); };
  quantize_group_vec<kGfAffine, CH, XT>(map, first, groups, s.page, s.D);
}

template <typename XT>
__global__ void __launch_bounds__(256)
prompt_pages_kernel(const PromptSource<XT> s, int64_t first, int64_t groups, const PromptPages pages) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t grp = first + wave_in_grid();
  if (grp >= groups) return;
  const GroupRef<XT> ref = prompt_group(s, pages, grp);
  auto get = [&](int r, int d) -> float { return r < ref.valid_rows ? to_f32(ref.src[(size_t)r * s.D + d]) : 0.0f; };
  quantize_group(get, s.page, s.D, ref.dst, ref.scale, ref.zero, lane);
}

// The advanced length of request b after its token at `pos` was stored (ok) or dropped; a dropped
// token also counts into *dropped when the caller gave a counter.
__device__ __forceinline__ void count_append(int64_t* lengths_out, unsigned* dropped, int b, int64_t pos, bool ok) {
  lengths_out[b] = ok ? pos + 1 : pos;
  if (!ok && dropped != nullptr) __hip_atomic_fetch_add(dropped, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One decode token per request (see fs_append_tokens_i8).  Group (kv, b, h): position
// pos = lengths_in[b] lands in row pos % page of page table[b, pos / page]; the page is
// dequantized (stale rows included), that row replaced, and the page requantized in place.
template <typename XT, typename IT>
__global__ void __launch_bounds__(256)
append_tokens_kernel(const XT* k_new, const XT* v_new, PageStore ks, PageStore vs, int64_t num_pages,
                     const IT* table, int table_cols, const int64_t* lengths_in, int64_t* lengths_out,
                     unsigned* dropped, int B, int H, int page, int D) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t grp = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t rows = (int64_t)B * H;
  if (grp >= 2 * rows) return;
  const int kv = grp >= rows ? 1 : 0;
  const int64_t bh = grp - kv * rows;
  const int b = (int)(bh / H);
  const int h = (int)(bh - (int64_t)b * H);
  const int64_t pos = lengths_in[b];
  const int64_t lp = pos >= 0 ? pos / page : -1;
  const int64_t pg = (lp >= 0 && lp < table_cols) ? (int64_t)table[(size_t)b * table_cols + lp] : -1;
  const bool ok = pg >= 0 && pg < num_pages;
  if (kv == 0 && h == 0 && lane == 0) count_append(lengths_out, dropped, b, pos, ok);
  if (!ok) return;
  const int off = (int)(pos - lp * page);
  const PageStore st = kv ? vs : ks;
  const XT* src = (kv ? v_new : k_new) + (size_t)bh * D;
  const int64_t sidx = pg * H + h;
  const int8_t* vals = st.values + (size_t)sidx * page * D;
  auto get = [&](int r, int d) -> float {
    if (r == off) return to_f32(src[d]);
    const int u = (int)vals[(size_t)r * D + d] + 128;
    return ((float)u - (float)st.zero[sidx]) * st.scale[sidx];
  };
  quantize_group(get, page, D, st.values + (size_t)sidx * page * D, st.scale + sidx, st.zero + sidx, lane);
}

// Vectorized append_tokens_kernel for page * D = CH * 512, D % 8 == 0: the page is read once
// into registers (8 bytes per lane and chunk), the new row comes straight from the token, and
// the requantized page is written back with the register-resident quantizer.  block_table
// entries are int32 (table_bytes 4) or int64.
template <int CH, typename XT>
__global__ void __launch_bounds__(256)
append_tokens_vec_kernel(const XT* k_new, const XT* v_new, PageStore ks, PageStore vs, int64_t num_pages,
                         const void* table, int table_bytes, int table_cols, const int64_t* lengths_in,
                         int64_t* lengths_out, unsigned* dropped, int B, int H, int page, int D) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t grp = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t rows = (int64_t)B * H;
  if (grp >= 2 * rows) return;
  const int kv = grp >= rows ? 1 : 0;
  const int64_t bh = grp - kv * rows;
  const int b = (int)(bh / H);
  const int h = (int)(bh - (int64_t)b * H);
  const int64_t pos = lengths_in[b];
  const int64_t lp = pos >= 0 ? pos / page : -1;
  int64_t pg = -1;
  if (lp >= 0 && lp < table_cols) {
    const size_t ti = (size_t)b * table_cols + lp;
    pg = table_bytes == 4 ? (int64_t)((const int32_t*)table)[ti] : ((const int64_t*)table)[ti];
  }
  const bool ok = pg >= 0 && pg < num_pages;
  if (kv == 0 && h == 0 && lane == 0) count_append(lengths_out, dropped, b, pos, ok);
  if (!ok) return;
  const int off = (int)(pos - lp * page);
  const PageStore st = kv ? vs : ks;
  const XT* src = (kv ? v_new : k_new) + (size_t)bh * D;
  const int64_t sidx = pg * H + h;
  int8_t* vals = st.values + (size_t)sidx * page * D;
  const float s_old = st.scale[sidx], z_old = (float)st.zero[sidx];
  float x[CH][8];
  float mn = __builtin_huge_valf(), mx = -__builtin_huge_valf();
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int e = c * 512 + lane * 8;
    const int r = e / D;
    if (r == off) {
      load8(src + (e - r * D), x[c]);
    } else {
      const uint2 raw = *(const uint2*)(vals + e);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t wv = i < 4 ? raw.x : raw.y;
        const int u = (int)((wv >> (8 * (i % 4))) & 0xffu) ^ 0x80;  // stored int8 + 128
        x[c][i] = ((float)u - z_old) * s_old;
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      mn = fminf(mn, x[c][i]);
      mx = fmaxf(mx, x[c][i]);
    }
  }
  mn = wave_min_valu(mn);  // DPP and lane swaps: no LDS round trips on the append's latency chain
  mx = wave_max_valu(mx);
  const float scale = fmaxf((mx - mn) / 255.0f, 1.0e-8f);
  const float zero = fminf(fmaxf(__builtin_rintf(-mn / scale), 0.0f), 255.0f);
  const float rcp = 1.0f / scale;
  if (__builtin_isfinite(fmaxf(fabsf(mn), fabsf(mx)) * rcp))
    store_chunks<CH, true>(x, scale, rcp, zero, vals, CH * 512, lane);
  else
    store_chunks<CH, false>(x, scale, rcp, zero, vals, CH * 512, lane);
  if (lane == 0) {
    st.scale[sidx] = scale;
    st.zero[sidx] = (int16_t)zero;
  }
}

// Symmetric absmax INT8, one scale per token row: scale = max(absmax / 127, 1e-8),
// q = clamp(rint(x / scale), -127, 127), stored in the affine layout with block 1 and zero
// point 128 (dequantized value (q + 128 - 128) * scale).  LPR = head_dim / 8 lanes per row,
// each holding 8 contiguous values; 64 / LPR rows per wave.
template <int LPR, typename XT>
__global__ void __launch_bounds__(256)
quantize_sym_rows_kernel(const XT* x, int64_t rows, int D, int8_t* values, float* scale, int16_t* zero) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t r = wave * (kWave / LPR) + lane / LPR;
  const int c = lane % LPR;
  const bool live = r < rows;
  float v[8];
  if (live) {
    load8(x + (size_t)r * D + 8 * c, v);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = 0.0f;
  }
  float am = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) am = fmaxf(am, fabsf(v[i]));
#pragma unroll
  for (int off = 1; off < LPR; off <<= 1) am = fmaxf(am, __shfl_xor(am, off, kWave));
  const float s = fmaxf(am / 127.0f, 1.0e-8f);
  if (!live) return;
  uint32_t w[2] = {0u, 0u};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float qv = fminf(fmaxf(__builtin_rintf(v[i] / s), -127.0f), 127.0f);
    w[i / 4] |= ((uint32_t)(int)qv & 0xffu) << (8 * (i % 4));
  }
  *(uint2*)(values + (size_t)r * D + 8 * c) = make_uint2(w[0], w[1]);
  if (c == 0) {
    scale[r] = s;
    zero[r] = 128;
  }
}

// Same quantizer, one wave per row, for head dims that are not a power-of-two multiple of 8.
template <typename XT>
__global__ void __launch_bounds__(256)
quantize_sym_rows_generic_kernel(const XT* x, int64_t rows, int D, int8_t* values, float* scale, int16_t* zero) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t r = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  if (r >= rows) return;
  const XT* src = x + (size_t)r * D;
  float am = 0.0f;
  for (int d = lane; d < D; d += kWave) am = fmaxf(am, fabsf(to_f32(src[d])));
  am = wave_max(am);
  const float s = fmaxf(am / 127.0f, 1.0e-8f);
  for (int d = lane; d < D; d += kWave)
    values[(size_t)r * D + d] = (int8_t)(int)fminf(fmaxf(__builtin_rintf(to_f32(src[d]) / s), -127.0f), 127.0f);
  if (lane == 0) {
    scale[r] = s;
    zero[r] = 128;
  }
}

// ---- reading quantized rows back ---------------------------------------------------------------
// Rows of one or two stores (K, and V unless null) as dense [B, H, S, D]: out[b, h, s] is row s % page
// of page table[b, s / page] of head h (table null: page b), ((float)u - zero) * scale or
// float(code) * scale.  A page's rows hold nb quant blocks of qb rows each.  A -1 entry reads page 0,
// as the reference's clamp does; an entry past the store reads as NaN.
//
// One wave per `unit` rows (about 2048 values), W values per lane and step, all loads of the wave
// issued before its stores.  Bound by the fp32 stores (4 of 5 bytes).  The cache read back through
// dequantize, gather and permute moved every fp32 value three times: measured on MI355X, to_dense of
// [4, 32, 2039, 128] 396 -> 62 us (5.4 TB/s).
struct ReadParams {
  const int8_t* values[2];
  const float* scale[2];
  const int16_t* zero[2];
  void* out[2];
  const void* table;
  int table_bytes, cols;
  int64_t P;
  int B, H, S, D, page, nb, qb;
  int unit, per_page;  // rows per wave, waves per page
};

enum ReadFormat : int { kRfInt8 = 0, kRfFp8 = 1, kRfChannel = 2 };
constexpr int kReadSteps = 8;
typedef float f32x4_q __attribute__((ext_vector_type(4)));

template <int RF, typename OT>
__device__ __forceinline__ OT read_value(uint32_t byte, float scale, float zero) {
  if constexpr (RF == kRfFp8) return from_f32<OT>(__builtin_amdgcn_cvt_pk_f32_fp8(byte, false)[0] * scale);
  return from_f32<OT>(((float)(int)(byte ^ 0x80u) - zero) * scale);
}

template <int RF, int W, typename OT, typename I>
__global__ void __launch_bounds__(256)
read_rows_kernel(const ReadParams p, int64_t first, int64_t units) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t wave = first + wave_in_grid();
  if (wave >= units) return;
  I t = sizeof(I) == 4 ? (I)__builtin_amdgcn_readfirstlane((int)wave) : (I)wave;
  // unit -> (tensor, b, h, page of the row, part of the page); neighbouring waves write neighbouring rows
  const I per_row = (I)p.cols * (I)p.per_page;
  I bh = t / per_row;
  const I rest = t - bh * per_row;
  const int lp = (int)(rest / (I)p.per_page);
  const int r0 = (int)(rest - (I)lp * (I)p.per_page) * p.unit;
  const int side = bh >= (I)p.B * (I)p.H ? 1 : 0;
  if (side) bh -= (I)p.B * (I)p.H;
  const int64_t b = (int64_t)(bh / (I)p.H);
  const int h = (int)(bh - (I)b * (I)p.H);
  const int64_t s0 = (int64_t)lp * p.page + r0;
  if (s0 >= p.S) return;
  const int rows = (int)min((int64_t)min(p.unit, p.page - r0), p.S - s0);
  int64_t pg = b;
  if (p.table) {
    const size_t ti = (size_t)b * p.cols + lp;
    pg = p.table_bytes == 4 ? (int64_t)((const int32_t*)p.table)[ti] : ((const int64_t*)p.table)[ti];
    if (pg < 0) pg = 0;
  }
  OT* out = (OT*)p.out[side] + (((size_t)b * p.H + h) * p.S + s0) * p.D;
  const int n = rows * p.D;
  if (pg >= p.P) {
    for (int e = lane; e < n; e += kWave) out[e] = from_f32<OT>(__builtin_nanf(""));
    return;
  }
  const size_t head = (size_t)pg * p.H + h;
  const int8_t* src = p.values[side] + (head * p.nb * p.qb + r0) * p.D;
  const float* scale = p.scale[side] + head * p.nb * (RF == kRfChannel ? p.D : 1);
  const int16_t* zero = RF == kRfFp8 ? nullptr : p.zero[side] + head * p.nb * (RF == kRfChannel ? p.D : 1);
  // the lane's values at lane * W + i * 64 W, as (row, dim) kept by increments
  int r = lane * W / p.D, d = lane * W - r * p.D;
  const int dr = kWave * W / p.D, dd = kWave * W - dr * p.D;
  for (int e0 = lane * W; e0 < n; e0 += kReadSteps * kWave * W) {
    uint32_t w[kReadSteps];
    float sc[kReadSteps][RF == kRfChannel ? W : 1], zp[kReadSteps][RF == kRfChannel ? W : 1];
#pragma unroll
    for (int i = 0; i < kReadSteps; ++i) {
      const int e = e0 + i * kWave * W;
      const bool ok = e < n;
      if constexpr (W == 4)
        w[i] = ok ? __builtin_nontemporal_load((const uint32_t*)(src + e)) : 0u;
      else
        w[i] = ok ? (uint32_t)(uint8_t)src[e] : 0u;
      const int blk = ok ? (r0 + r) / p.qb : 0;
      if constexpr (RF == kRfChannel) {
#pragma unroll
        for (int j = 0; j < W; ++j) {
          sc[i][j] = scale[(size_t)blk * p.D + d + j];
          zp[i][j] = (float)zero[(size_t)blk * p.D + d + j];
        }
      } else {
        sc[i][0] = scale[blk];
        zp[i][0] = RF == kRfFp8 ? 0.f : (float)zero[blk];
      }
      r += dr;
      d += dd;
      if (d >= p.D) {
        d -= p.D;
        ++r;
      }
    }
#pragma unroll
    for (int i = 0; i < kReadSteps; ++i) {
      const int e = e0 + i * kWave * W;
      if (e >= n) break;
      if constexpr (W == 4 && std::is_same<OT, float>::value) {
        f32x4_q v;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v[j] = read_value<RF, float>((w[i] >> (8 * j)) & 0xffu, sc[i][RF == kRfChannel ? j : 0], zp[i][RF == kRfChannel ? j : 0]);
        __builtin_nontemporal_store(v, (f32x4_q*)(out + e));
      } else {
        OT v[W];
#pragma unroll
        for (int j = 0; j < W; ++j)
          v[j] = read_value<RF, OT>((w[i] >> (8 * j)) & 0xffu, sc[i][RF == kRfChannel ? j : 0], zp[i][RF == kRfChannel ? j : 0]);
        __builtin_memcpy(out + e, v, sizeof(v));
      }
    }
  }
}

static dim3 wave_grid(int64_t groups) { return dim3((unsigned)((groups + 3) / 4)); }

// HIP launches fewer than 2^32 threads at a time: 2^24 - 1 workgroups of 4 waves.  go(first, grid) launches
// one range of the groups (one wave each); all but enormous calls are a single range.
constexpr int64_t kRangeGroups = 4 * ((1LL << 24) - 1);
template <typename F>
static void launch_ranges(int64_t groups, F&& go) {
  for (int64_t first = 0; first < groups; first += kRangeGroups)
    go(first, wave_grid(groups - first < kRangeGroups ? groups - first : kRangeGroups));
}

static bool is_pow2_chunks(int ch) { return ch == 1 || ch == 2 || ch == 4 || ch == 8; }

// f(integral_constant<CH>) for the instantiated chunk counts of group_chunks.
template <typename F>
static void by_chunks(int ch, F&& f) {
  switch (ch) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    default: f(std::integral_constant<int, 16>{}); break;
  }
}

// f(typed null pointer) for a source dtype code; false for an unknown code.
template <typename F>
static bool by_dtype(int dtype, F&& f) {
  switch (dtype) {
    case FS_F32: f((const float*)nullptr); return true;
    case FS_F16: f((const __half*)nullptr); return true;
    case FS_BF16: f((const __hip_bfloat16*)nullptr); return true;
    default: return false;
  }
}
template <typename T>
using value_of = std::remove_cv_t<std::remove_pointer_t<T>>;

template <typename XT>
static int launch_vec_append(int ch, dim3 grid, hipStream_t st, const XT* k_new, const XT* v_new, PageStore ks,
                             PageStore vs, int64_t num_pages, const void* table, int table_bytes, int table_cols,
                             const int64_t* lengths_in, int64_t* lengths_out, unsigned* dropped, int B, int H,
                             int page, int D) {
  const dim3 block(256);
  switch (ch) {
    case 1: hipLaunchKernelGGL((append_tokens_vec_kernel<1, XT>), grid, block, 0, st, k_new, v_new, ks, vs, num_pages, table, table_bytes, table_cols, lengths_in, lengths_out, dropped, B, H, page, D); break;
    case 2: hipLaunchKernelGGL((append_tokens_vec_kernel<2, XT>), grid, block, 0, st, k_new, v_new, ks, vs, num_pages, table, table_bytes, table_cols, lengths_in, lengths_out, dropped, B, H, page, D); break;
    case 4: hipLaunchKernelGGL((append_tokens_vec_kernel<4, XT>), grid, block, 0, st, k_new, v_new, ks, vs, num_pages, table, table_bytes, table_cols, lengths_in, lengths_out, dropped, B, H, page, D); break;
    default: hipLaunchKernelGGL((append_tokens_vec_kernel<8, XT>), grid, block, 0, st, k_new, v_new, ks, vs, num_pages, table, table_bytes, table_cols, lengths_in, lengths_out, dropped, B, H, page, D); break;
  }
  return check_launch("append_tokens");
}

// One launch of read_rows_kernel; B, H, S, D > 0.
static int launch_read(const char* what, ReadParams p, int sides, int rf, int out_dtype, hipStream_t st) {
  p.unit = p.D >= 2048 ? 1 : 2048 / p.D;
  if (p.unit > p.page) p.unit = p.page;
  p.per_page = (p.page + p.unit - 1) / p.unit;
  const int64_t units = (int64_t)sides * p.B * p.H * p.cols * p.per_page;
  const size_t esize = out_dtype == FS_F32 ? 4 : 2;
  bool four = p.D % 4 == 0;
  for (int i = 0; i < sides; ++i)
    four = four && (uintptr_t)p.values[i] % 4 == 0 && (uintptr_t)p.out[i] % (4 * esize) == 0;
  const bool known = by_dtype(out_dtype, [&](auto tag) {
    using OT = value_of<decltype(tag)>;
    auto go = [&](auto rf_c, auto w_c) {
      constexpr int RF = decltype(rf_c)::value, W = decltype(w_c)::value;
      launch_ranges(units, [&](int64_t first, dim3 grid) {
        if (units <= 0x7fffffffLL)
          hipLaunchKernelGGL((read_rows_kernel<RF, W, OT, unsigned>), grid, dim3(256), 0, st, p, first, units);
        else
          hipLaunchKernelGGL((read_rows_kernel<RF, W, OT, int64_t>), grid, dim3(256), 0, st, p, first, units);
      });
    };
    auto by_width = [&](auto rf_c) {
      if (four)
        go(rf_c, std::integral_constant<int, 4>{});
      else
        go(rf_c, std::integral_constant<int, 1>{});
    };
    if (rf == kRfFp8)
      by_width(std::integral_constant<int, kRfFp8>{});
    else if (rf == kRfChannel)
      by_width(std::integral_constant<int, kRfChannel>{});
    else
      by_width(std::integral_constant<int, kRfInt8>{});
  });
  return known ? check_launch(what) : set_error(FS_ERR_INVALID, std::string(what) + ": dtype code must be 0, 1 or 2");
}

// Blocks [outer, n_blocks, block_size, head_dim] -> [outer, seq_len, head_dim]: each outer entry is a
// page of seq_len rows.
static int launch_dequantize(const char* what, const int8_t* values, const float* scale, const int16_t* zero,
                             int64_t outer, int n_blocks, int block_size, int head_dim, int seq_len, void* out,
                             int out_dtype, int rf, hipStream_t st) {
  if (outer <= 0 || n_blocks <= 0 || block_size <= 0 || head_dim <= 0 || seq_len < 0 ||
      (int64_t)n_blocks * block_size < seq_len)
    return set_error(FS_ERR_INVALID, std::string(what) + ": invalid sizes");
  if (!values || !scale || (!zero && rf != kRfFp8) || !out)
    return set_error(FS_ERR_INVALID, std::string(what) + ": null pointer");
  if (out_dtype != FS_F32 && out_dtype != FS_F16 && out_dtype != FS_BF16)
    return set_error(FS_ERR_INVALID, std::string(what) + ": dtype code must be 0, 1 or 2");
  if (seq_len == 0) return FS_OK;
  const size_t esize = out_dtype == FS_F32 ? 4 : 2;
  constexpr int64_t kOuter = 1 << 20;  // entries per launch (B is an int)
  for (int64_t o = 0; o < outer; o += kOuter) {
    ReadParams p{};
    p.values[0] = values + (size_t)o * n_blocks * block_size * head_dim;
    p.scale[0] = scale + (size_t)o * n_blocks;
    p.zero[0] = zero ? zero + (size_t)o * n_blocks : nullptr;
    p.out[0] = (char*)out + (size_t)o * seq_len * head_dim * esize;
    p.B = (int)(outer - o < kOuter ? outer - o : kOuter);
    p.P = p.B;
    p.H = p.cols = 1;
    p.S = p.page = seq_len;
    p.D = head_dim;
    p.nb = n_blocks;
    p.qb = block_size;
    if (const int rc = launch_read(what, p, 1, rf, out_dtype, st)) return rc;
  }
  return FS_OK;
}

// One launch of the block quantizer of format GF.
template <int GF>
static int launch_blocks(const char* what, const void* x, int x_dtype, int64_t outer, int S, int D, int bs,
                         int8_t* values, float* scale, int16_t* zero, hipStream_t st) {
  if (outer <= 0 || S <= 0 || D <= 0 || bs <= 0)
    return set_error(FS_ERR_INVALID, std::string(what) + ": sizes must be positive");
  if (!x || !values || !scale || (!zero && GF != kGfFp8))
    return set_error(FS_ERR_INVALID, std::string(what) + ": null pointer");
  const int nb = (S + bs - 1) / bs;
  const int64_t groups = outer * nb;
  if ((groups + 3) / 4 > 0x7fffffffLL) return set_error(FS_ERR_INVALID, std::string(what) + ": too many groups");
  const bool aligned = ((uintptr_t)x % 16) == 0 && ((uintptr_t)values % 8) == 0 &&
                       (GF != kGfChannel || wide_params(scale, zero));
  const int ch = aligned ? group_chunks(bs, D, GF == kGfChannel || GF == kGfToken) : 0;
  const bool known = by_dtype(x_dtype, [&](auto tag) {
    using XT = value_of<decltype(tag)>;
    const XT* src = (const XT*)x;
    launch_ranges(groups, [&](int64_t first, dim3 grid) {
      if (ch == 0)
        hipLaunchKernelGGL((quantize_blocks_kernel<XT, GF>), grid, dim3(256), 0, st, src, first, groups, S, D, bs, nb, values, scale, zero);
      else
        by_chunks(ch, [&](auto c) {
          hipLaunchKernelGGL((quantize_blocks_vec_kernel<GF, decltype(c)::value, XT>), grid, dim3(256), 0, st, src, first, groups, S, D, bs, nb, values, scale, zero);
        });
    });
  });
  return known ? check_launch(what) : set_error(FS_ERR_INVALID, std::string(what) + ": dtype code must be 0, 1 or 2");
}

// Where a page quantize launch places its pages, and the lists it writes beside them.
struct PagePlan {
  const int64_t* page_src;
  int interleaved;
  int64_t P;
  int64_t* table;
  int64_t* lengths;
};

// One launch of the page quantizer of format GF, for K and V (v null: K alone).
template <int GF>
static int launch_pages(const char* what, const void* k, const void* v, int x_dtype, int batch, int H, int S, int D,
                        int page, const PagePlan& plan, PageStore ks, PageStore vs, hipStream_t st) {
  if (batch <= 0 || H <= 0 || S <= 0 || D <= 0 || page <= 0)
    return set_error(FS_ERR_INVALID, std::string(what) + ": sizes must be positive");
  auto whole = [](const PageStore& p) { return p.values && p.scale && (p.zero || GF == kGfFp8); };
  if (!k || !whole(ks) || (v && !whole(vs))) return set_error(FS_ERR_INVALID, std::string(what) + ": null pointer");
  const int nbps = (S + page - 1) / page;
  if (plan.P != (int64_t)batch * nbps)
    return set_error(FS_ERR_INVALID, std::string(what) + ": num_pages must equal batch * ceil(seq_len / page)");
  const bool counted = plan.P * H <= 0x7fffffffLL;  // the vectorized kernel's index arithmetic is 32-bit
  if (!counted && GF == kGfAffine)
    return set_error(FS_ERR_INVALID, std::string(what) + ": more than 2^31 (page, head) groups");
  const int64_t groups = plan.P * H * (v ? 2 : 1);
  auto aligned = [](const void* x, const PageStore& p) {
    return ((uintptr_t)x % 16) == 0 && ((uintptr_t)p.values % 8) == 0 &&
           (GF != kGfChannel || wide_params(p.scale, p.zero));
  };
  const int ch = counted && aligned(k, ks) && (!v || aligned(v, vs))
                     ? group_chunks(page, D, GF == kGfChannel || GF == kGfToken) : 0;
  const bool known = by_dtype(x_dtype, [&](auto tag) {
    using XT = value_of<decltype(tag)>;
    const PagesSource<XT> s{(const XT*)k, (const XT*)v, ks, vs, plan.page_src, plan.table, plan.lengths, plan.P,
                            batch, H, S, D, page, nbps, plan.interleaved};
    launch_ranges(groups, [&](int64_t first, dim3 grid) {
      if (ch == 0)
        hipLaunchKernelGGL((quantize_pages_kernel<XT, GF>), grid, dim3(256), 0, st, s, first, groups);
      else
        by_chunks(ch, [&](auto c) {
          hipLaunchKernelGGL((quantize_pages_vec_kernel<GF, decltype(c)::value, XT>), grid, dim3(256), 0, st, s, first, groups);
        });
    });
  });
  return known ? check_launch(what) : set_error(FS_ERR_INVALID, std::string(what) + ": dtype code must be 0, 1 or 2");
}

}  // namespace fs

using namespace fs;

extern "C" int fs_quantize_i8(const void* x, int x_dtype, int64_t outer, int seq_len, int head_dim, int block_size,
                              int8_t* values, float* scale, int16_t* zero, void* stream) {
  return launch_blocks<kGfAffine>("quantize", x, x_dtype, outer, seq_len, head_dim, block_size, values, scale, zero,
                                  (hipStream_t)stream);
}

extern "C" int fs_dequantize_i8(const int8_t* values, const float* scale, const int16_t* zero, int64_t outer,
                                int n_blocks, int block_size, int head_dim, int seq_len, void* out, int out_dtype,
                                void* stream) {
  return launch_dequantize("dequantize", values, scale, zero, outer, n_blocks, block_size, head_dim, seq_len, out,
                           out_dtype, kRfInt8, (hipStream_t)stream);
}

extern "C" int fs_quantize_pages_i8(const void* x, int x_dtype, int batch, int heads, int seq_len, int head_dim,
                                    int page_size, const int64_t* page_src, int64_t num_pages, int8_t* values,
                                    float* scale, int16_t* zero, void* stream) {
  return launch_pages<kGfAffine>("quantize_pages", x, nullptr, x_dtype, batch, heads, seq_len, head_dim, page_size,
                      PagePlan{page_src, 0, num_pages, nullptr, nullptr}, PageStore{values, scale, zero},
                      PageStore{}, (hipStream_t)stream);
}

extern "C" int fs_write_prompt_i8(const void* k, const void* v, int src_dtype, int src_tokens, int length, int heads,
                                  int head_dim, int page_size, int8_t* k_values, float* k_scale, int16_t* k_zero,
                                  int8_t* v_values, float* v_scale, int16_t* v_zero, int64_t num_pages,
                                  const int32_t* pages, int n_pages, void* stream) {
  if (heads <= 0 || head_dim <= 0 || page_size <= 0 || length <= 0 || src_tokens < length || num_pages <= 0)
    return set_error(FS_ERR_INVALID, "write_prompt: sizes must be positive and length at most src_tokens");
  if (n_pages != (int)(((int64_t)length + page_size - 1) / page_size))
    return set_error(FS_ERR_INVALID, "write_prompt: n_pages must equal ceil(length / page_size)");
  if (!k || !pages || !k_values || !k_scale || !k_zero || (v && (!v_values || !v_scale || !v_zero)))
    return set_error(FS_ERR_INVALID, "write_prompt: null pointer");
  if ((int64_t)n_pages * page_size > 0x7fffffffLL || (int64_t)page_size * head_dim > 0x7fffffffLL)
    return set_error(FS_ERR_INVALID, "write_prompt: sizes past 2^31");
  for (int i = 0; i < n_pages; ++i)
    if (pages[i] < 0 || pages[i] >= num_pages) return set_error(FS_ERR_INVALID, "write_prompt: page id out of range");
  hipStream_t st = (hipStream_t)stream;
  const uintptr_t src_bits = (uintptr_t)k | (uintptr_t)v, dst_bits = (uintptr_t)k_values | (v ? (uintptr_t)v_values : 0);
  const int ch = src_bits % 16 == 0 && dst_bits % 8 == 0 ? group_chunks(page_size, head_dim, false) : 0;
  const int sides = v ? 2 : 1;
  // pages per launch: what the arguments hold, of a group count within the kernel's 32-bit index
  const int64_t most = 0x7fffffffLL / ((int64_t)sides * heads);
  if (most < 1) return set_error(FS_ERR_INVALID, "write_prompt: more than 2^31 heads of K and V");
  const int step = most < kPromptPages ? (int)most : kPromptPages;
  PromptPages ids;
  for (int first = 0; first < n_pages; first += step) {
    const int n = n_pages - first < step ? n_pages - first : step;
    for (int i = 0; i < n; ++i) ids.id[i] = pages[first + i];
    for (int i = n; i < kPromptPages; ++i) ids.id[i] = 0;
    const int64_t groups = (int64_t)sides * n * heads;
    const bool known = by_dtype(src_dtype, [&](auto tag) {
      using XT = value_of<decltype(tag)>;
      const PromptSource<XT> s{(const XT*)k, (const XT*)v, {k_values, k_scale, k_zero}, {v_values, v_scale, v_zero},
                               heads, src_tokens, length, head_dim, page_size, first, n};
      launch_ranges(groups, [&](int64_t at, dim3 grid) {
        if (ch == 0)
          hipLaunchKernelGGL(prompt_pages_kernel<XT>, grid, dim3(256), 0, st, s, at, groups, ids);
        else
          by_chunks(ch, [&](auto c) {
            hipLaunchKernelGGL((prompt_pages_vec_kernel<decltype(c)::value, XT>), grid, dim3(256), 0, st, s, at, groups, ids);
          });
      });
    });
    if (!known) return set_error(FS_ERR_INVALID, "write_prompt: dtype code must be 0, 1 or 2");
    if (const int rc = check_launch("write_prompt")) return rc;
  }
  return FS_OK;
}

extern "C" int fs_update_pages_i8(const int8_t* in_values, const float* in_scale, const int16_t* in_zero,
                                  int64_t in_pages, int in_quant_block, int8_t* out_values, float* out_scale,
                                  int16_t* out_zero, const int64_t* pages, const uint8_t* fresh, int64_t n_pages,
                                  const int32_t* row_src, const void* src, int src_dtype, int src_tokens, int heads,
                                  int page_size, int head_dim, void* stream) {
  if (n_pages <= 0) return FS_OK;
  if (heads <= 0 || page_size <= 0 || head_dim <= 0 || src_tokens <= 0 || in_pages < 0)
    return set_error(FS_ERR_INVALID, "update_pages: sizes must be positive");
  if (in_quant_block <= 0 || page_size % in_quant_block != 0)
    return set_error(FS_ERR_INVALID, "update_pages: page_size must be a multiple of the input quant block");
  if (in_values == out_values && in_quant_block != page_size)
    return set_error(FS_ERR_INVALID, "update_pages: in-place update needs quant block == page_size");
  if (!out_values || !out_scale || !out_zero || !row_src || !src)
    return set_error(FS_ERR_INVALID, "update_pages: null pointer");
  if (in_pages > 0 && (!in_values || !in_scale || !in_zero)) return set_error(FS_ERR_INVALID, "update_pages: null input store");
  const int64_t groups = n_pages * heads;
  hipStream_t st = (hipStream_t)stream;
  const bool known = by_dtype(src_dtype, [&](auto tag) {
    using XT = value_of<decltype(tag)>;
    launch_ranges(groups, [&](int64_t first, dim3 grid) {
      hipLaunchKernelGGL(update_pages_kernel<XT>, grid, dim3(256), 0, st, in_values, in_scale, in_zero, in_pages, in_quant_block, out_values, out_scale, out_zero, pages, fresh, first, groups, row_src, (const XT*)src, src_tokens, heads, page_size, head_dim);
    });
  });
  if (!known) return set_error(FS_ERR_INVALID, "update_pages: dtype code must be 0, 1 or 2");
  return check_launch("update_pages");
}

extern "C" int fs_append_tokens_i8(const void* k_new, const void* v_new, int src_dtype, int8_t* k_values,
                                   float* k_scale, int16_t* k_zero, int8_t* v_values, float* v_scale,
                                   int16_t* v_zero, int64_t num_pages, const void* block_table,
                                   int table_index_bytes, int table_cols, const int64_t* lengths_in,
                                   int64_t* lengths_out, int batch, int heads, int head_dim, int page_size,
                                   unsigned* dropped, void* stream) {
  if (batch <= 0) return FS_OK;
  if (heads <= 0 || head_dim <= 0 || page_size <= 0 || num_pages <= 0 || table_cols <= 0)
    return set_error(FS_ERR_INVALID, "append_tokens: sizes must be positive");
  if (table_index_bytes != 4 && table_index_bytes != 8)
    return set_error(FS_ERR_INVALID, "append_tokens: block_table must be int32 or int64");
  if (!k_new || !v_new || !k_values || !k_scale || !k_zero || !v_values || !v_scale || !v_zero || !block_table ||
      !lengths_in || !lengths_out)
    return set_error(FS_ERR_INVALID, "append_tokens: null pointer");
  if (lengths_in == lengths_out)
    return set_error(FS_ERR_INVALID, "append_tokens: lengths_in and lengths_out must be different buffers");
  const PageStore ks{k_values, k_scale, k_zero}, vs{v_values, v_scale, v_zero};
  const int64_t groups = 2LL * batch * heads;
  if (groups > kRangeGroups) return set_error(FS_ERR_INVALID, "append_tokens: more than 2^25 - 2 (request, head) pairs");
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid = wave_grid(groups), block(256);
  const int ch = vec_chunks(page_size, head_dim);
  if (is_pow2_chunks(ch) && ((uintptr_t)k_new % 16) == 0 && ((uintptr_t)v_new % 16) == 0 &&
      ((uintptr_t)k_values % 8) == 0 && ((uintptr_t)v_values % 8) == 0) {
    switch (src_dtype) {
      case FS_F32: return launch_vec_append<float>(ch, grid, st, (const float*)k_new, (const float*)v_new, ks, vs, num_pages, block_table, table_index_bytes, table_cols, lengths_in, lengths_out, dropped, batch, heads, page_size, head_dim);
      case FS_F16: return launch_vec_append<__half>(ch, grid, st, (const __half*)k_new, (const __half*)v_new, ks, vs, num_pages, block_table, table_index_bytes, table_cols, lengths_in, lengths_out, dropped, batch, heads, page_size, head_dim);
      case FS_BF16: return launch_vec_append<__hip_bfloat16>(ch, grid, st, (const __hip_bfloat16*)k_new, (const __hip_bfloat16*)v_new, ks, vs, num_pages, block_table, table_index_bytes, table_cols, lengths_in, lengths_out, dropped, batch, heads, page_size, head_dim);
      default: return set_error(FS_ERR_INVALID, "append_tokens: dtype code must be 0, 1 or 2");
    }
  }
#define FS_APPEND(XT, IT)                                                                                       \
  hipLaunchKernelGGL((append_tokens_kernel<XT, IT>), grid, block, 0, st, (const XT*)k_new, (const XT*)v_new, ks, \
                     vs, num_pages, (const IT*)block_table, table_cols, lengths_in, lengths_out, dropped, batch, \
                     heads, page_size, head_dim)
#define FS_APPEND_IDX(XT) \
  if (table_index_bytes == 4) FS_APPEND(XT, int32_t); else FS_APPEND(XT, int64_t)
  switch (src_dtype) {
    case FS_F32: FS_APPEND_IDX(float); break;
    case FS_F16: FS_APPEND_IDX(__half); break;
    case FS_BF16: FS_APPEND_IDX(__hip_bfloat16); break;
    default: return set_error(FS_ERR_INVALID, "append_tokens: dtype code must be 0, 1 or 2");
  }
#undef FS_APPEND_IDX
#undef FS_APPEND
  return check_launch("append_tokens");
}

template <typename XT>
static int launch_quantize_sym(const XT* x, int64_t rows, int D, int8_t* values, float* scale, int16_t* zero,
                               hipStream_t st) {
  const int lpr = D / 8;
  const bool vec = D % 8 == 0 && lpr <= kWave && (lpr & (lpr - 1)) == 0 && ((uintptr_t)x % 16) == 0 &&
                   ((uintptr_t)values % 8) == 0;
  const int per_wave = vec ? kWave / lpr : 1;
  launch_ranges((rows + per_wave - 1) / per_wave, [&](int64_t first, dim3 grid) {
    const int64_t r0 = first * per_wave, n = rows - r0;
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, x + r0 * D, n, D, values + r0 * D, scale + r0, zero + r0);
    };
    switch (vec ? lpr : 0) {
      case 0: go(quantize_sym_rows_generic_kernel<XT>); break;
      case 1: go(quantize_sym_rows_kernel<1, XT>); break;
      case 2: go(quantize_sym_rows_kernel<2, XT>); break;
      case 4: go(quantize_sym_rows_kernel<4, XT>); break;
      case 8: go(quantize_sym_rows_kernel<8, XT>); break;
      case 16: go(quantize_sym_rows_kernel<16, XT>); break;
      case 32: go(quantize_sym_rows_kernel<32, XT>); break;
      default: go(quantize_sym_rows_kernel<64, XT>); break;
    }
  });
  return check_launch("quantize_symmetric_per_token");
}

extern "C" int fs_quantize_sym_i8(const void* x, int x_dtype, int64_t rows, int head_dim, int8_t* values,
                                  float* scale, int16_t* zero, void* stream) {
  if (rows <= 0 || head_dim <= 0) return set_error(FS_ERR_INVALID, "quantize_symmetric: sizes must be positive");
  if (!x || !values || !scale || !zero) return set_error(FS_ERR_INVALID, "quantize_symmetric: null pointer");
  hipStream_t st = (hipStream_t)stream;
  switch (x_dtype) {
    case FS_F32: return launch_quantize_sym((const float*)x, rows, head_dim, values, scale, zero, st);
    case FS_F16: return launch_quantize_sym((const __half*)x, rows, head_dim, values, scale, zero, st);
    case FS_BF16: return launch_quantize_sym((const __hip_bfloat16*)x, rows, head_dim, values, scale, zero, st);
    default: return set_error(FS_ERR_INVALID, "quantize_symmetric: dtype code must be 0, 1 or 2");
  }
}

extern "C" int fs_quantize_fp8(const void* x, int x_dtype, int64_t outer, int seq_len, int head_dim, int block_size,
                               uint8_t* values, float* scale, int16_t* zero, void* stream) {
  return launch_blocks<kGfFp8>("quantize_fp8", x, x_dtype, outer, seq_len, head_dim, block_size, (int8_t*)values, scale,
                               zero, (hipStream_t)stream);
}

extern "C" int fs_quantize_pages_fp8(const void* x, int x_dtype, int batch, int heads, int seq_len, int head_dim,
                                     int page_size, const int64_t* page_src, int64_t num_pages, uint8_t* values,
                                     float* scale, int16_t* zero, void* stream) {
  return launch_pages<kGfFp8>("quantize_pages_fp8", x, nullptr, x_dtype, batch, heads, seq_len, head_dim, page_size,
                      PagePlan{page_src, 0, num_pages, nullptr, nullptr}, PageStore{(int8_t*)values, scale, zero},
                      PageStore{}, (hipStream_t)stream);
}

extern "C" int fs_dequantize_fp8(const uint8_t* values, const float* scale, int64_t outer, int n_blocks,
                                 int block_size, int head_dim, int seq_len, void* out, int out_dtype, void* stream) {
  return launch_dequantize("dequantize_fp8", (const int8_t*)values, scale, nullptr, outer, n_blocks, block_size, head_dim,
                           seq_len, out, out_dtype, kRfFp8, (hipStream_t)stream);
}

extern "C" int fs_quantize_i8_channel(const void* x, int x_dtype, int64_t outer, int seq_len, int head_dim,
                                      int block_size, int8_t* values, float* scale, int16_t* zero, void* stream) {
  return launch_blocks<kGfChannel>("quantize_channel", x, x_dtype, outer, seq_len, head_dim, block_size, values, scale,
                                   zero, (hipStream_t)stream);
}

extern "C" int fs_quantize_pages_i8_channel(const void* x, int x_dtype, int batch, int heads, int seq_len,
                                            int head_dim, int page_size, const int64_t* page_src, int64_t num_pages,
                                            int8_t* values, float* scale, int16_t* zero, void* stream) {
  return launch_pages<kGfChannel>("quantize_pages_channel", x, nullptr, x_dtype, batch, heads, seq_len, head_dim, page_size,
                      PagePlan{page_src, 0, num_pages, nullptr, nullptr}, PageStore{values, scale, zero},
                      PageStore{}, (hipStream_t)stream);
}

extern "C" int fs_build_cache(const void* k, const void* v, int src_dtype, int kv_format, int batch, int heads,
                              int seq_len, int head_dim, int page_size, const int64_t* page_src, int interleaved,
                              int64_t num_pages, void* k_values, float* k_scale, int16_t* k_zero, void* v_values,
                              float* v_scale, int16_t* v_zero, int64_t* block_table, int64_t* lengths, void* stream) {
  if (!v) return set_error(FS_ERR_INVALID, "build_cache: null pointer");
  const PagePlan plan{page_src, interleaved, num_pages, block_table, lengths};
  const PageStore ks{(int8_t*)k_values, k_scale, k_zero}, vs{(int8_t*)v_values, v_scale, v_zero};
  const hipStream_t st = (hipStream_t)stream;
  switch (kv_format) {
    case 0: return launch_pages<kGfAffine>("build_cache", k, v, src_dtype, batch, heads, seq_len, head_dim, page_size, plan, ks, vs, st);
    case 1: return launch_pages<kGfFp8>("build_cache", k, v, src_dtype, batch, heads, seq_len, head_dim, page_size, plan, ks, vs, st);
    case 2: return launch_pages<kGfChannel>("build_cache", k, v, src_dtype, batch, heads, seq_len, head_dim, page_size, plan, ks, vs, st);
    case 3: return launch_pages<kGfToken>("build_cache", k, v, src_dtype, batch, heads, seq_len, head_dim, page_size, plan, ks, vs, st);
    default: return set_error(FS_ERR_INVALID, "build_cache: kv_format must be 0 to 3");
  }
}

extern "C" int fs_read_cache(const void* k_values, const float* k_scale, const int16_t* k_zero, const void* v_values,
                             const float* v_scale, const int16_t* v_zero, int kv_format, const void* block_table,
                             int table_index_bytes, int table_cols, int batch, int heads, int seq_len, int head_dim,
                             int64_t num_pages, int page_size, int n_blocks, int quant_block, void* k_out, void* v_out,
                             int out_dtype, void* stream) {
  if (batch <= 0 || heads <= 0 || seq_len <= 0 || head_dim <= 0 || num_pages <= 0 || page_size <= 0 || n_blocks <= 0 ||
      quant_block <= 0 || table_cols <= 0)
    return set_error(FS_ERR_INVALID, "read_cache: sizes must be positive");
  if ((int64_t)n_blocks * quant_block < page_size || (int64_t)table_cols * page_size < seq_len)
    return set_error(FS_ERR_INVALID, "read_cache: the table does not cover seq_len");
  if (table_index_bytes != 4 && table_index_bytes != 8)
    return set_error(FS_ERR_INVALID, "read_cache: block_table must be int32 or int64");
  if (kv_format < 0 || kv_format > 2) return set_error(FS_ERR_INVALID, "read_cache: kv_format must be 0, 1 or 2");
  const bool zp = kv_format != kRfFp8;
  if (!k_values || !k_scale || !k_out || !block_table || (zp && !k_zero) ||
      (v_values && (!v_scale || !v_out || (zp && !v_zero))))
    return set_error(FS_ERR_INVALID, "read_cache: null pointer");
  const ReadParams p{{(const int8_t*)k_values, (const int8_t*)v_values}, {k_scale, v_scale}, {k_zero, v_zero},
                     {k_out, v_out}, block_table, table_index_bytes, table_cols, num_pages, batch, heads, seq_len,
                     head_dim, page_size, n_blocks, quant_block, 0, 0};
  return launch_read("read_cache", p, v_values ? 2 : 1, kv_format, out_dtype, (hipStream_t)stream);
}
