// Layout and producer kernels around the INT4 matmul:
//   repack   storage layout -> kernel layout (+ optional act_order permutation)
//   zeros    fp32 zero points -> u8, counting values that are not integers in [0,15]
//   dequant  packed INT4 -> fp16 / bf16 / fp32 weights (bit-exact with the reference)
//   rtn      fp weights -> (packed, scale, zero) with per-group min/max RTN
//   awq      AWQ-GEMM int32 words <-> storage layout, fp16 [G,N] <-> fp32 [N,G]
// All are integer/byte or elementwise work bound by HBM bandwidth.
#include "../../include/pare_amd.h"
#include "pmi_common.h"
#include "pmi_launch.h"

namespace pmi {
namespace {

constexpr int kBlock = 256;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

PMI_DEV uint32_t nibble_at(const uint8_t* __restrict__ row, int64_t col) {
  return (row[col >> 1] >> ((col & 1) * 4)) & 0xFu;
}

PMI_DEV int64_t safe_col(const int32_t* __restrict__ perm, int64_t k, int64_t K) {
  if (!perm) return k;
  const int32_t p = perm[k];
  return (p >= 0 && p < K) ? (int64_t)p : k;
}

// Output byte j of a row holds, inside its group tile t (hgs = gs/2 bytes),
// column t*gs + (j - t*hgs) in bits 0-3 and that column + hgs in bits 4-7
// (pare/core/pack.py:123-130). One thread writes 4 consecutive output bytes.
__global__ void repack_kernel(const uint8_t* __restrict__ packed, uint8_t* __restrict__ out,
                              const int32_t* __restrict__ perm, int64_t N, int64_t K, int64_t gs) {
  const int64_t row_bytes = K >> 1;
  const int64_t words_per_row = row_bytes >> 2;
  const int64_t hgs = gs >> 1;
  const int64_t total = N * words_per_row;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t n = idx / words_per_row;
    const int64_t jw = (idx - n * words_per_row) << 2;
    const uint8_t* src = packed + n * row_bytes;
    uint32_t word = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int64_t j = jw + b;
      const int64_t t = j / hgs;
      const int64_t k_lo = t * gs + (j - t * hgs);
      const uint32_t lo = nibble_at(src, safe_col(perm, k_lo, K));
      const uint32_t hi = nibble_at(src, safe_col(perm, k_lo + hgs, K));
      word |= (lo | (hi << 4)) << (8 * b);
    }
    *reinterpret_cast<uint32_t*>(out + n * row_bytes + jw) = word;
  }
}

// The same without a permutation, for gs % 32 == 0: 16 output bytes per thread.
// Tiles and rows are contiguous, so output byte o of the whole weight lies in
// tile o / hgs and its nibbles come from two runs of eight source bytes, hgs / 2
// apart. 14336 x 4096 at gs 128: 48.2 us a nibble at a time with 64-bit
// divisions per byte, 11.2 (5.2 TB/s) this way.
__global__ __launch_bounds__(kBlock) void repack16_kernel(const uint8_t* __restrict__ packed,
                                                          uint8_t* __restrict__ out, uint32_t chunks,
                                                          uint32_t per_tile, uint32_t per_tile_m) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= chunks) return;
  const uint32_t t = udiv(i, per_tile, per_tile_m), r = i - t * per_tile;
  // hgs = 16 per_tile bytes per tile; source bytes 8 r of its two halves
  const uint8_t* src = packed + (size_t)t * per_tile * 16 + 8 * r;
  const u32x2 lo = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(src));
  const u32x2 hi = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(src + 8 * per_tile));
  u32x4 v;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t even = (lo[k] & 0x0F0F0F0Fu) | ((hi[k] & 0x0F0F0F0Fu) << 4);
    const uint32_t odd = ((lo[k] >> 4) & 0x0F0F0F0Fu) | (hi[k] & 0xF0F0F0F0u);
    v[2 * k] = __builtin_amdgcn_perm(odd, even, 0x05010400u);
    v[2 * k + 1] = __builtin_amdgcn_perm(odd, even, 0x07030602u);
  }
  reinterpret_cast<u32x4*>(out)[i] = v;
}

__global__ void zeros_to_u8_kernel(const float* __restrict__ zeros, uint8_t* __restrict__ out,
                                   int32_t* __restrict__ bad, int64_t count) {
  int local_bad = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float z = zeros[i];
    const bool ok = z >= 0.f && z <= 15.f && z == rintf(z);  // false for NaN
    local_bad += ok ? 0 : 1;
    out[i] = ok ? (uint8_t)(int)z : (uint8_t)0;
  }
  if (bad && local_bad) atomicAdd(bad, local_bad);
}

// int32 act_order permutation -> its 16-bit copy (K <= 65536) for the GEMV's
// LDS gather. Entries outside [0, K) become 0, as the kernels clamp them at
// use, and are counted into *bad (nullable).
__global__ void perm_u16_kernel(const int32_t* __restrict__ perm, uint16_t* __restrict__ out,
                                int32_t* __restrict__ bad, int64_t K) {
  int local_bad = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < K;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t p = perm[i];
    const bool ok = p >= 0 && (int64_t)p < K;
    local_bad += ok ? 0 : 1;
    out[i] = ok ? (uint16_t)p : (uint16_t)0;
  }
  if (bad && local_bad) atomicAdd(bad, local_bad);
}

// [N, G] -> [G, N] copies of the scales and zero points. strict: zeros that are
// not integers in [0, 15] become 0 and are counted like zeros_to_u8_kernel;
// otherwise they are converted as the matmul kernels convert them. A workgroup
// turns 32 rows x 32 groups in LDS, four elements per thread with their loads
// in flight together, so that reads run along G and writes along N (14336 x 32:
// 6.4 us with reads G apart, 4.0).
__global__ __launch_bounds__(kBlock) void sz_group_major_kernel(
    const float* __restrict__ scales, const void* __restrict__ zeros, int zero_u8, int strict,
    float* __restrict__ s_gm, uint8_t* __restrict__ z_gm, int32_t* __restrict__ bad, int64_t N,
    int64_t G) {
  __shared__ float st[32][33];
  __shared__ uint8_t zt[32][36];
  const int64_t n0 = (int64_t)blockIdx.x * 32;
  const int c = threadIdx.x & 31, r0 = threadIdx.x >> 5;  // 8 rows of 32
  int local_bad = 0;
  for (int64_t g0 = (int64_t)blockIdx.y * 32; g0 < G; g0 += (int64_t)gridDim.y * 32) {
    float sv[4], zf[4];
    uint32_t zb[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t n = n0 + r0 + 8 * k < N ? n0 + r0 + 8 * k : N - 1, g = g0 + c < G ? g0 + c : G - 1;
      const int64_t i = n * G + g;
      sv[k] = scales[i];
      if (zero_u8) zb[k] = ((const uint8_t*)zeros)[i];
      else zf[k] = ((const float*)zeros)[i];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      bool ok;
      if (zero_u8) {
        ok = zb[k] <= 15 || !strict;
      } else {
        ok = (zf[k] >= 0.f && zf[k] <= 15.f && zf[k] == rintf(zf[k])) || !strict;  // false for NaN
        zb[k] = (uint32_t)(int)zf[k];
      }
      local_bad += ok || n0 + r0 + 8 * k >= N || g0 + c >= G ? 0 : 1;
      st[c][r0 + 8 * k] = sv[k];
      zt[c][r0 + 8 * k] = ok ? (uint8_t)zb[k] : (uint8_t)0;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int q = r0 + 8 * k;
      if (n0 + c < N && g0 + q < G) {
        s_gm[(g0 + q) * N + n0 + c] = st[q][c];
        z_gm[(g0 + q) * N + n0 + c] = zt[q][c];
      }
    }
    __syncthreads();
  }
  if (bad && local_bad) atomicAdd(bad, local_bad);
}

// w_hat = (float(q) - zero) * scale in fp32, then one rounding to out dtype
// (pare/core/functional.py:90-91, pare/layers/linear.py:129).
template <int OUT>
__global__ void dequant_kernel(const uint8_t* __restrict__ w, int layout,
                               const float* __restrict__ scales, const void* __restrict__ zeros,
                               int zero_u8, const int32_t* __restrict__ idx,
                               void* __restrict__ out, int64_t N, int64_t K, int64_t gs) {
  const int64_t row_bytes = K >> 1;
  const int64_t hgs = gs >> 1;
  const int64_t G = K / gs;
  const int64_t total = N * K;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t n = e / K;
    const int64_t j = e - n * K;
    const uint8_t* row = w + n * row_bytes;
    uint32_t q;
    int64_t g, col;
    if (layout == PMI_LAYOUT_KERNEL) {
      const int64_t t = j / gs;
      const int64_t r = j - t * gs;
      const int64_t byte = t * hgs + (r < hgs ? r : r - hgs);
      q = (row[byte] >> (r < hgs ? 0 : 4)) & 0xFu;
      g = t;
      col = safe_col(idx, j, K);
    } else {
      q = nibble_at(row, j);
      g = idx ? (int64_t)idx[j] : j / gs;
      col = j;
    }
    float v;
    if (g < 0 || g >= G) {
      v = __builtin_nanf("");
    } else {
      const int64_t sz = n * G + g;
      const float z = zero_u8 ? (float)((const uint8_t*)zeros)[sz] : ((const float*)zeros)[sz];
      v = ((float)q - z) * scales[sz];
    }
    const int64_t o = n * K + col;
    if constexpr (OUT == PMI_F32) {
      ((float*)out)[o] = v;
    } else if constexpr (OUT == PMI_F16) {
      ((f16*)out)[o] = f32_to_f16_rne(v);
    } else {
      ((uint16_t*)out)[o] = f32_to_bf16_rne(v);
    }
  }
}

// The same for the storage layout without g_idx and gs % 8 == 0: eight columns
// (one word of codes, one scale and zero point, 16 or 32 output bytes) per
// thread and step, four steps in flight. Groups and rows are contiguous: the
// group of eight columns is their number over gs / 8, no row needed. 14336 x
// 4096 to bf16: 139.5 us a column at a time with two 64-bit divisions each, 27.2
// (5.4 TB/s) this way.
template <int OUT, bool ZU8>
__global__ __launch_bounds__(kBlock) void dequant8_kernel(const uint8_t* __restrict__ w,
                                                          const float* __restrict__ scales,
                                                          const void* __restrict__ zeros, void* __restrict__ out,
                                                          uint32_t chunks, uint32_t per_group,
                                                          uint32_t per_group_m) {
  constexpr int kSteps = 4;
  const uint32_t i0 = blockIdx.x * (kBlock * kSteps) + threadIdx.x;
  uint32_t q[kSteps];
  float sc[kSteps], z[kSteps];
#pragma unroll
  for (int k = 0; k < kSteps; ++k) {
    uint32_t i = i0 + k * kBlock;
    i = i < chunks ? i : chunks - 1;
    const uint32_t g = udiv(i, per_group, per_group_m);
    q[k] = reinterpret_cast<const uint32_t*>(w)[i];
    sc[k] = scales[g];
    if constexpr (ZU8) z[k] = (float)((const uint8_t*)zeros)[g];
    else z[k] = ((const float*)zeros)[g];
  }
#pragma unroll
  for (int k = 0; k < kSteps; ++k) {
    const uint32_t i = i0 + k * kBlock;
    if (i >= chunks) return;
    float v[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = ((float)((q[k] >> (4 * c)) & 0xFu) - z[k]) * sc[k];
    if constexpr (OUT == PMI_F32) {
      f32x4* o = reinterpret_cast<f32x4*>(out) + 2 * (size_t)i;
      o[0] = f32x4{v[0], v[1], v[2], v[3]};
      o[1] = f32x4{v[4], v[5], v[6], v[7]};
    } else {
      u32x4 o;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        uint32_t lo, hi;
        if constexpr (OUT == PMI_F16) {
          lo = __builtin_bit_cast(uint16_t, f32_to_f16_rne(v[2 * c]));
          hi = __builtin_bit_cast(uint16_t, f32_to_f16_rne(v[2 * c + 1]));
        } else {
          lo = f32_to_bf16_rne(v[2 * c]);
          hi = f32_to_bf16_rne(v[2 * c + 1]);
        }
        o[c] = lo | (hi << 16);
      }
      reinterpret_cast<u32x4*>(out)[i] = o;
    }
  }
}

// AWQ-GEMM int32 words (pare/model/export_awq.py:37-49): word c of a row packs
// output columns 8c..8c+7, column 8c + order[i] in bits 4i..4i+3 with
// order = [0,2,4,6,1,3,5,7]. awq_slot(o) is the inverse: the nibble index of
// column 8c + o.
PMI_DEV int awq_slot(int o) { return (o >> 1) | ((o & 1) << 2); }

// qweight int32 [K, N/8] -> storage layout u8 [N, K/2]. One thread per
// (32-column block kb of K, word column c): 32 coalesced word loads down K,
// then eight 16-byte row writes (rows 8c..8c+7, bytes 16kb..16kb+15).
__global__ void awq_to_storage_kernel(const int32_t* __restrict__ qweight,
                                      uint8_t* __restrict__ packed, int64_t N, int64_t K) {
  const int64_t NC = N >> 3;
  const int64_t total = (K >> 5) * NC;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t kb = idx / NC, c = idx - kb * NC;
    const int32_t* src = qweight + (kb << 5) * NC + c;
    uint32_t out[8][4];
#pragma unroll
    for (int o = 0; o < 8; ++o)
#pragma unroll
      for (int s = 0; s < 4; ++s) out[o][s] = 0;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const uint32_t w = (uint32_t)src[(int64_t)(8 * s + t) * NC];
#pragma unroll
        for (int o = 0; o < 8; ++o) out[o][s] |= ((w >> (4 * awq_slot(o))) & 0xFu) << (4 * t);
      }
    }
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      u32x4 v = {out[o][0], out[o][1], out[o][2], out[o][3]};
      *reinterpret_cast<u32x4*>(packed + (8 * c + o) * (K >> 1) + (kb << 4)) = v;
    }
  }
}

// qzeros int32 [G, N/8], scales fp16 [G, N] -> zero, scale fp32 [N, G].
__global__ void awq_sz_to_rows_kernel(const int32_t* __restrict__ qzeros,
                                      const f16* __restrict__ scales, float* __restrict__ scale,
                                      float* __restrict__ zero, int64_t N, int64_t G) {
  const int64_t NC = N >> 3;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < G * NC;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t g = idx / NC, c = idx - g * NC;
    const uint32_t z = (uint32_t)qzeros[idx];
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      const int64_t n = 8 * c + o;
      zero[n * G + g] = (float)((z >> (4 * awq_slot(o))) & 0xFu);
      scale[n * G + g] = (float)scales[g * N + n];
    }
  }
}

// Storage layout u8 [N, K/2] -> qweight int32 [K, N/8]; the inverse of
// awq_to_storage_kernel with the same thread mapping (coalesced word stores).
__global__ void storage_to_awq_kernel(const uint8_t* __restrict__ packed,
                                      int32_t* __restrict__ qweight, int64_t N, int64_t K) {
  const int64_t NC = N >> 3;
  const int64_t total = (K >> 5) * NC;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t kb = idx / NC, c = idx - kb * NC;
    u32x4 in[8];
#pragma unroll
    for (int o = 0; o < 8; ++o)
      in[o] = *reinterpret_cast<const u32x4*>(packed + (8 * c + o) * (K >> 1) + (kb << 4));
    int32_t* dst = qweight + (kb << 5) * NC + c;
#pragma unroll
    for (int t = 0; t < 32; ++t) {
      uint32_t w = 0;
#pragma unroll
      for (int o = 0; o < 8; ++o)
        w |= ((in[o][t >> 3] >> (4 * (t & 7))) & 0xFu) << (4 * awq_slot(o));
      dst[(int64_t)t * NC] = (int32_t)w;
    }
  }
}

// zero (PMI_F32 or PMI_U8) and scale fp32 [N, G] -> qzeros int32 [G, N/8] and
// scales fp16 [G, N]. fp32 zeros are rounded half-to-even first
// (pare/model/export_awq.py:85); a zero outside [0, 15] after rounding is
// counted in *bad and packed as 0.
__global__ void awq_sz_from_rows_kernel(const float* __restrict__ scale,
                                        const void* __restrict__ zero, int zero_u8,
                                        int32_t* __restrict__ qzeros, f16* __restrict__ scales,
                                        int32_t* __restrict__ bad, int64_t N, int64_t G) {
  const int64_t NC = N >> 3;
  int local_bad = 0;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < G * NC;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t g = idx / NC, c = idx - g * NC;
    uint32_t w = 0;
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      const int64_t n = 8 * c + o;
      uint32_t z;
      if (zero_u8) {
        z = ((const uint8_t*)zero)[n * G + g];
      } else {
        const float r = rintf(((const float*)zero)[n * G + g]);
        z = (r >= 0.f && r <= 15.f) ? (uint32_t)(int)r : 16u;  // NaN -> 16
      }
      local_bad += z <= 15u ? 0 : 1;
      w |= (z <= 15u ? z : 0u) << (4 * awq_slot(o));
      scales[g * N + n] = f32_to_f16_rne(scale[n * G + g]);
    }
    qzeros[idx] = (int32_t)w;
  }
  if (bad && local_bad) atomicAdd(bad, local_bad);
}

template <int IN>
PMI_DEV float load_as_f32(const void* p, int64_t i) {
  if constexpr (IN == PMI_F32) {
    return ((const float*)p)[i];
  } else if constexpr (IN == PMI_F16) {
    return (float)((const f16*)p)[i];
  } else {
    return __builtin_bit_cast(float, (uint32_t)((const uint16_t*)p)[i] << 16);
  }
}

PMI_DEV float wave_min(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}
PMI_DEV float wave_max(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// One wave per (row, group): min/max -> (scale, zero) -> q -> packed bytes.
// Formulas of pare/core/scale.py:73-91 and pare/core/functional.py:68-75 with
// qmin = 0, qmax = 15 (unsigned INT4); rintf is round-half-to-even like
// torch.round.
template <int IN>
__global__ void rtn_kernel(const void* __restrict__ w, uint8_t* __restrict__ packed,
                           float* __restrict__ scale_out, float* __restrict__ zero_out, int64_t N,
                           int64_t K, int64_t gs, int sym) {
  const int lane = threadIdx.x & 63;
  const int64_t G = K / gs;
  const int64_t unit = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (unit >= N * G) return;
  const int64_t n = unit / G;
  const int64_t g = unit - n * G;
  const int64_t base = n * K + g * gs;
  const int64_t pairs = gs >> 1;

  float mn = __builtin_inff(), mx = -__builtin_inff();
  for (int64_t p = lane; p < pairs; p += 64) {
    const float a = load_as_f32<IN>(w, base + 2 * p);
    const float b = load_as_f32<IN>(w, base + 2 * p + 1);
    mn = fminf(mn, fminf(a, b));
    mx = fmaxf(mx, fmaxf(a, b));
  }
  mn = wave_min(mn);
  mx = wave_max(mx);

  float scale, zero;
  scale_zero_from_minmax(mn, mx, sym, scale, zero);
  if (lane == 0) {
    scale_out[unit] = scale;
    zero_out[unit] = zero;
  }
  for (int64_t p = lane; p < pairs; p += 64) {
    const float a = load_as_f32<IN>(w, base + 2 * p);
    const float b = load_as_f32<IN>(w, base + 2 * p + 1);
    const float qa = fminf(fmaxf(rintf(a / scale + zero), 0.0f), 15.0f);
    const float qb = fminf(fmaxf(rintf(b / scale + zero), 0.0f), 15.0f);
    packed[(base >> 1) + p] = (uint8_t)((int)qa | ((int)qb << 4));
  }
}

// The same for groups of 16 to 1024 columns that are a power of two: 16 columns
// per lane, a group on LANES = gs / 16 neighbouring lanes, so the weight is read
// once, in 16-byte loads, and quantised from registers. 14336 x 4096 bf16 at gs
// 128: 157.4 us with a wave per group and two passes of 2-byte loads, 27 (5.4
// TB/s) this way.
// min (or max) of v over aligned runs of LANES lanes, in every lane; DPP inside
// rows of 16 (xor 1, xor 2, mirror of 8, mirror of 16).
template <int CTRL>
PMI_DEV float dpp(float v) {
  const int i = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, CTRL, 0xF, 0xF, false));
}
template <int LANES, bool MAX>
PMI_DEV float run_minmax(float v) {
  auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : fminf(a, b); };
  if constexpr (LANES >= 2) v = op(v, dpp<0xB1>(v));
  if constexpr (LANES >= 4) v = op(v, dpp<0x4E>(v));
  if constexpr (LANES >= 8) v = op(v, dpp<0x141>(v));
  if constexpr (LANES >= 16) v = op(v, dpp<0x140>(v));
  if constexpr (LANES >= 32) v = op(v, __shfl_xor(v, 16, 64));
  if constexpr (LANES >= 64) v = op(v, __shfl_xor(v, 32, 64));
  return v;
}

template <int IN, int LANES>
__global__ __launch_bounds__(kBlock) void rtn16_kernel(const void* __restrict__ w, uint8_t* __restrict__ packed,
                                                       float* __restrict__ scale_out,
                                                       float* __restrict__ zero_out, uint32_t chunks, int sym) {
  const uint32_t i0 = blockIdx.x * kBlock + threadIdx.x;
  // whole groups: past the end nothing is stored
  const uint32_t i = i0 < chunks ? i0 : chunks - 1;
  float v[16];
  if constexpr (IN == PMI_F32) {
    const f32x4* p = reinterpret_cast<const f32x4*>(w) + 4 * (size_t)i;
    f32x4 d[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) d[k] = p[k];
#pragma unroll
    for (int c = 0; c < 16; ++c) v[c] = d[c >> 2][c & 3];
  } else {
    const u32x4* p = reinterpret_cast<const u32x4*>(w) + 2 * (size_t)i;
    const u32x4 d[2] = {p[0], p[1]};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const uint32_t x = d[c >> 2][c & 3];
      if constexpr (IN == PMI_F16) {
        const f16x2 h = as_f16x2(x);
        v[2 * c] = (float)h[0], v[2 * c + 1] = (float)h[1];
      } else {
        v[2 * c] = __builtin_bit_cast(float, x << 16);
        v[2 * c + 1] = __builtin_bit_cast(float, x & 0xFFFF0000u);
      }
    }
  }
  float mn = __builtin_inff(), mx = -__builtin_inff();
#pragma unroll
  for (int c = 0; c < 16; ++c) mn = fminf(mn, v[c]), mx = fmaxf(mx, v[c]);
  mn = run_minmax<LANES, false>(mn);
  mx = run_minmax<LANES, true>(mx);
  float scale, zero;
  scale_zero_from_minmax(mn, mx, sym, scale, zero);
  // t = v / scale + zero with both roundings. 16-bit weights land on rounding
  // boundaries often (a fifth of bf16 groups hold an exact tie), so their
  // quotients are the correctly rounded ones, from a refined reciprocal and one
  // remainder step (Markstein). fp32 weights hardly ever do: t = v * (1 / scale) +
  // zero is within 1e-5 there, and lanes nearer than that to a boundary divide, as
  // do those whose scale the steps do not cover. Dividing everywhere: 44 us.
  // Adding 1.5 * 2^23 rounds to an integer in the low bits; a NaN clamps to 0
  // here as it does below.
  const float magic = 12582912.0f;
  float inv = __builtin_amdgcn_rcpf(scale);
  inv = fmaf(fmaf(-scale, inv, 1.0f), inv, inv);
  inv = fmaf(fmaf(-scale, inv, 1.0f), inv, inv);
  u32x2 q = {0u, 0u};
  float off = 0.f;
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    float t;
    if constexpr (IN == PMI_F32) {
      t = fmaf(v[c], inv, zero);
    } else {
      const float q0 = v[c] * inv;
      t = fmaf(fmaf(-scale, q0, v[c]), inv, q0) + zero;
    }
    t = __builtin_amdgcn_fmed3f(t, 0.0f, 15.0f);
    const float m = t + magic;
    if constexpr (IN == PMI_F32) off = fmaxf(off, fabsf(t - (m - magic)));
    q[c >> 3] += (__builtin_bit_cast(uint32_t, m) - 0x4B400000u) << (4 * (c & 7));
  }
  if (off > 0.49999f || !(scale < 1e30f)) {
    q = u32x2{0u, 0u};
#pragma unroll
    for (int c = 0; c < 16; ++c)
      q[c >> 3] |= (uint32_t)(int)fminf(fmaxf(rintf(v[c] / scale + zero), 0.0f), 15.0f) << (4 * (c & 7));
  }
  if (i0 < chunks) {
    reinterpret_cast<u32x2*>(packed)[i] = q;
    if (threadIdx.x % LANES == 0) {
      scale_out[i / LANES] = scale;
      zero_out[i / LANES] = zero;
    }
  }
}

template <int IN>
bool launch_rtn16(const void* w, uint8_t* packed, float* scale, float* zero, uint32_t chunks, int64_t gs, int sym,
                  hipStream_t stream) {
  const dim3 grid((chunks + kBlock - 1) / kBlock), block(kBlock);
#define PMI_RTN16(GS)                                                                                              \
  case GS:                                                                                                         \
    hipLaunchKernelGGL((rtn16_kernel<IN, GS / 16>), grid, block, 0, stream, w, packed, scale, zero, chunks, sym); \
    return true
  switch (gs) {
    PMI_RTN16(16);
    PMI_RTN16(32);
    PMI_RTN16(64);
    PMI_RTN16(128);
    PMI_RTN16(256);
    PMI_RTN16(512);
    PMI_RTN16(1024);
    default: return false;
  }
#undef PMI_RTN16
}

// Kernel layout (group size gs) -> tiled layout of the tiled-weight GEMM.
// Output chunk i (16 bytes) of block (panel p, unit u): tile j = (i / 64) % 4,
// lane L = i % 64 = n + 16 h, row 64 p + 4 n + j (zero past N); its byte b
// holds columns c = 128 u + (b < 8 ? 8 h + b : 32 + 8 h + b - 8) in the low
// nibble and c + 64 in the high nibble. In the kernel layout column k of a row
// lies in the gs-wide tile starting at k0 = k - k % gs, byte k0 / 2 + k % (gs/2),
// low nibble for k % gs < gs / 2, high nibble otherwise. One thread per chunk.
__device__ __forceinline__ uint32_t kernel_nibble(const uint8_t* __restrict__ row, int k, int gs) {
  const int k0 = k - k % gs, j = k - k0, hg = gs >> 1;
  const uint8_t b = row[(k0 >> 1) + (j < hg ? j : j - hg)];
  return j < hg ? (b & 0xFu) : (b >> 4);
}

__global__ void tile_kernel(const uint8_t* __restrict__ wk, uint8_t* __restrict__ wt, int64_t N,
                            int64_t K, int gs) {
  const int64_t U = K >> 7;
  const int64_t chunks = (N + 63) / 64 * U * 256;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < chunks;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int L = (int)(i & 63), j = (int)((i >> 6) & 3);
    const int64_t pu = i >> 8;
    const int64_t u = pu % U, p = pu / U;
    const int n = L & 15, h = L >> 4;
    const int64_t row = 64 * p + 4 * n + j;
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    if (row < N) {
      const uint8_t* src = wk + row * (K >> 1);
      if (gs == 128) {
        // the unit is one group: its bytes carry columns c and c + 64 already
        const uint32_t* a = reinterpret_cast<const uint32_t*>(src + 64 * u + 8 * h);
        const uint32_t* b = reinterpret_cast<const uint32_t*>(src + 64 * u + 32 + 8 * h);
        w[0] = a[0], w[1] = a[1], w[2] = b[0], w[3] = b[1];
      } else if (gs == 64) {
        // k-steps 0 and 1 are the low and high nibbles of the first group's
        // bytes 8 h .., k-steps 2 and 3 those of the second's
        const uint32_t* a = reinterpret_cast<const uint32_t*>(src + 64 * u + 8 * h);
        const uint32_t* b = reinterpret_cast<const uint32_t*>(src + 64 * u + 32 + 8 * h);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          w[k] = (a[k] & 0x0F0F0F0Fu) | ((b[k] & 0x0F0F0F0Fu) << 4);
          w[2 + k] = ((a[k] >> 4) & 0x0F0F0F0Fu) | (b[k] & 0xF0F0F0F0u);
        }
      } else if (gs == 32) {
        // k-step t: nibble h / 2 of bytes 8 (h % 2) .. of group t's 16
        uint32_t r[4][2];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint32_t* a = reinterpret_cast<const uint32_t*>(src + 64 * u + 16 * t + 8 * (h & 1));
          r[t][0] = (a[0] >> (4 * (h >> 1))) & 0x0F0F0F0Fu;
          r[t][1] = (a[1] >> (4 * (h >> 1))) & 0x0F0F0F0Fu;
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          w[k] = r[0][k] | (r[2][k] << 4);
          w[2 + k] = r[1][k] | (r[3][k] << 4);
        }
      } else {
#pragma unroll
        for (int bb = 0; bb < 16; ++bb) {
          const int c = (int)(128 * u) + (bb < 8 ? 8 * h + bb : 32 + 8 * h + bb - 8);
          const uint32_t v = kernel_nibble(src, c, gs) | (kernel_nibble(src, c + 64, gs) << 4);
          w[bb >> 2] |= v << (8 * (bb & 3));
        }
      }
    }
    reinterpret_cast<u32x4*>(wt)[i] = u32x4{w[0], w[1], w[2], w[3]};
  }
}

int grid_for(int64_t work, int per_thread = 1) {
  int64_t blocks = (work / per_thread + kBlock - 1) / kBlock;
  if (blocks < 1) blocks = 1;
  if (blocks > 65536) blocks = 65536;
  return (int)blocks;
}

}  // namespace

hipError_t launch_repack(const uint8_t* packed, uint8_t* out, const int32_t* perm, int64_t N,
                         int64_t K, int64_t gs, hipStream_t stream) {
  const int64_t chunks = N * (K / 32);
  if (!perm && gs % 32 == 0 && chunks < (1ll << 31) && (uintptr_t)packed % 16 == 0 && (uintptr_t)out % 16 == 0) {
    const uint32_t per_tile = (uint32_t)(gs / 32);
    hipLaunchKernelGGL(repack16_kernel, dim3((unsigned)((chunks + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream,
                       packed, out, (uint32_t)chunks, per_tile, udiv_magic(per_tile));
    return hipGetLastError();
  }
  hipLaunchKernelGGL(repack_kernel, dim3(grid_for(N * (K / 8))), dim3(kBlock), 0, stream, packed,
                     out, perm, N, K, gs);
  return hipGetLastError();
}

hipError_t launch_tile(const uint8_t* w_kernel, uint8_t* w_tiled, int64_t N, int64_t K, int64_t gs,
                       hipStream_t stream) {
  hipLaunchKernelGGL(tile_kernel, dim3(grid_for((N + 63) / 64 * (K / 128) * 256)), dim3(kBlock), 0,
                     stream, w_kernel, w_tiled, N, K, (int)gs);
  return hipGetLastError();
}

hipError_t launch_zeros_to_u8(const float* zeros, uint8_t* out, int32_t* bad, int64_t count,
                              hipStream_t stream) {
  hipLaunchKernelGGL(zeros_to_u8_kernel, dim3(grid_for(count)), dim3(kBlock), 0, stream, zeros,
                     out, bad, count);
  return hipGetLastError();
}

hipError_t launch_perm_u16(const int32_t* perm, uint16_t* out, int32_t* bad, int64_t K,
                           hipStream_t stream) {
  hipLaunchKernelGGL(perm_u16_kernel, dim3(grid_for(K)), dim3(kBlock), 0, stream, perm, out, bad,
                     K);
  return hipGetLastError();
}

hipError_t launch_sz_group_major(const float* scales, const void* zeros, int zero_u8, int strict,
                                 float* scales_gm, uint8_t* zeros_gm, int32_t* bad, int64_t N,
                                 int64_t G, hipStream_t stream) {
  const int64_t gy = (G + 31) / 32;
  hipLaunchKernelGGL(sz_group_major_kernel, dim3((unsigned)((N + 31) / 32), (unsigned)(gy < 65535 ? gy : 65535)),
                     dim3(kBlock), 0, stream, scales, zeros, zero_u8, strict, scales_gm, zeros_gm, bad, N, G);
  return hipGetLastError();
}

hipError_t launch_awq_to_storage(const int32_t* qweight, const int32_t* qzeros, const void* scales,
                                 uint8_t* packed, float* scale, float* zero, int64_t N, int64_t K,
                                 int64_t gs, hipStream_t stream) {
  hipLaunchKernelGGL(awq_to_storage_kernel, dim3(grid_for((K / 32) * (N / 8))), dim3(kBlock), 0,
                     stream, qweight, packed, N, K);
  if (hipError_t e = hipGetLastError()) return e;
  const int64_t G = K / gs;
  hipLaunchKernelGGL(awq_sz_to_rows_kernel, dim3(grid_for(G * (N / 8))), dim3(kBlock), 0, stream,
                     qzeros, (const f16*)scales, scale, zero, N, G);
  return hipGetLastError();
}

hipError_t launch_storage_to_awq(const uint8_t* packed, const float* scale, const void* zero,
                                 int zero_u8, int32_t* qweight, int32_t* qzeros, void* scales,
                                 int32_t* bad, int64_t N, int64_t K, int64_t gs,
                                 hipStream_t stream) {
  hipLaunchKernelGGL(storage_to_awq_kernel, dim3(grid_for((K / 32) * (N / 8))), dim3(kBlock), 0,
                     stream, packed, qweight, N, K);
  if (hipError_t e = hipGetLastError()) return e;
  const int64_t G = K / gs;
  hipLaunchKernelGGL(awq_sz_from_rows_kernel, dim3(grid_for(G * (N / 8))), dim3(kBlock), 0, stream,
                     scale, zero, zero_u8, qzeros, (f16*)scales, bad, N, G);
  return hipGetLastError();
}

hipError_t launch_dequant(const uint8_t* w, int layout, const float* scales, const void* zeros,
                          int zero_u8, const int32_t* idx, void* out, int out_dtype, int64_t N,
                          int64_t K, int64_t gs, hipStream_t stream) {
  const int64_t chunks = N * (K / 8);
  if (layout == PMI_LAYOUT_STORAGE && !idx && gs % 8 == 0 && chunks < (1ll << 31) - 4 * kBlock &&
      (uintptr_t)w % 4 == 0 && (uintptr_t)out % 16 == 0) {
    const uint32_t pg = (uint32_t)(gs / 8), m = udiv_magic(pg);
    const dim3 grid((unsigned)((chunks + 4 * kBlock - 1) / (4 * kBlock))), block(kBlock);
#define PMI_DEQUANT8(OUT)                                                                           \
  if (zero_u8)                                                                                      \
    hipLaunchKernelGGL((dequant8_kernel<OUT, true>), grid, block, 0, stream, w, scales, zeros, out, \
                       (uint32_t)chunks, pg, m);                                                    \
  else                                                                                              \
    hipLaunchKernelGGL((dequant8_kernel<OUT, false>), grid, block, 0, stream, w, scales, zeros, out, \
                       (uint32_t)chunks, pg, m)
    switch (out_dtype) {
      case PMI_F16: PMI_DEQUANT8(PMI_F16); break;
      case PMI_BF16: PMI_DEQUANT8(PMI_BF16); break;
      default: PMI_DEQUANT8(PMI_F32);
    }
#undef PMI_DEQUANT8
    return hipGetLastError();
  }
  const dim3 grid(grid_for(N * K)), block(kBlock);
  switch (out_dtype) {
    case PMI_F16:
      hipLaunchKernelGGL(dequant_kernel<PMI_F16>, grid, block, 0, stream, w, layout, scales, zeros,
                         zero_u8, idx, out, N, K, gs);
      break;
    case PMI_BF16:
      hipLaunchKernelGGL(dequant_kernel<PMI_BF16>, grid, block, 0, stream, w, layout, scales,
                         zeros, zero_u8, idx, out, N, K, gs);
      break;
    default:
      hipLaunchKernelGGL(dequant_kernel<PMI_F32>, grid, block, 0, stream, w, layout, scales, zeros,
                         zero_u8, idx, out, N, K, gs);
  }
  return hipGetLastError();
}

hipError_t launch_rtn(const void* w, int w_dtype, uint8_t* packed, float* scale, float* zero,
                      int64_t N, int64_t K, int64_t gs, int sym, hipStream_t stream) {
  const int64_t chunks = N * (K / 16);
  if (gs >= 16 && K % 16 == 0 && chunks < (1ll << 31) - kBlock && (uintptr_t)w % 16 == 0 &&
      (uintptr_t)packed % 8 == 0) {
    const uint32_t n = (uint32_t)chunks;
    const bool done = w_dtype == PMI_F32   ? launch_rtn16<PMI_F32>(w, packed, scale, zero, n, gs, sym, stream)
                      : w_dtype == PMI_F16 ? launch_rtn16<PMI_F16>(w, packed, scale, zero, n, gs, sym, stream)
                                           : launch_rtn16<PMI_BF16>(w, packed, scale, zero, n, gs, sym, stream);
    if (done) return hipGetLastError();
  }
  const int64_t units = N * (K / gs);
  const int waves_per_block = 4;
  const dim3 grid((unsigned)((units + waves_per_block - 1) / waves_per_block));
  const dim3 block(64 * waves_per_block);
  switch (w_dtype) {
    case PMI_F32:
      hipLaunchKernelGGL(rtn_kernel<PMI_F32>, grid, block, 0, stream, w, packed, scale, zero, N, K,
                         gs, sym);
      break;
    case PMI_F16:
      hipLaunchKernelGGL(rtn_kernel<PMI_F16>, grid, block, 0, stream, w, packed, scale, zero, N, K,
                         gs, sym);
      break;
    default:
      hipLaunchKernelGGL(rtn_kernel<PMI_BF16>, grid, block, 0, stream, w, packed, scale, zero, N,
                         K, gs, sym);
  }
  return hipGetLastError();
}

}  // namespace pmi
