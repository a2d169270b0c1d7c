// Big-tile GEMM: INT4 W4A16 for many activation rows (prefill), gfx950
// (v_mfma_f32_16x16x32_f16 / _bf16).
//
// Work. A group of four waves owns MT 16-row activation tiles x 256 weight
// rows (a band of four 64-row panels), wave w the 64 rows of panel w against
// every activation row, over 128-column units of K. Each B operand (8 weights
// of a lane) is formed once and feeds MT MFMAs; each A operand read from LDS
// feeds four. Per unit and wave that is 16 MT MFMAs against 16 MT folds (fma
// x 4 lanes of accumulators), 176 instructions to form the B operands and 4 MT
// LDS reads. The layout before this one (eight waves of 32 rows x 128) read
// each A operand for two MFMAs only, which kept the LDS pipe as busy as the
// matrix cores: 4096 x 28672 x 4096 went from 937 to 745-765 us.
//
// Two groups per CU. A wave alternates between forming B operands (VALU) and
// MFMAs, so a SIMD needs two waves to keep both pipes busy. With KG = 1 a
// workgroup is one group and two workgroups share a CU (80 KiB of LDS and 256
// VGPRs each); where the output has no more tiles than the chip has CUs,
// KG = 2 makes a workgroup of two groups that take alternate units of one tile
// and add their accumulators through LDS at the end. Where the tiles fill
// less than half of the CUs, K is also split over workgroups (`splits`), whose
// fp32 partial tiles a second launch adds in split order.
//
// Staging. Everything goes global -> LDS by buffer_load ... lds, no registers
// in between: the unit's activation rows (128 columns, 16-byte chunk c of row r
// at chunk c ^ (r % 16), so the 16 rows of an A read fall in 16 bank groups),
// double-buffered; the wave's own 4 KiB of codes, single-buffered (they are
// read into registers at the head of a unit, and the copies of the next unit's
// follow). One s_barrier per unit. The copies are issued from inline asm: the
// compiler, which cannot tell the two activation slots apart, would otherwise
// drain them before every A read. They write LDS only (no register), and each
// wave waits for its own (vmcnt(0)) before the barrier that publishes them.
//
// Fold. Weight tiles go two at a time: the eight MFMAs of a pair run beside the
// fold (y += s * sum x (q - z), fp32) of the pair before it, interleaved by
// sched_group_barrier. Raised wave priority during the MFMAs lets the other
// wave's B operands fill the gaps (4096 x 28672 x 4096: 773 -> 747 us).
//
// Group sizes. KSG = 32-column k-steps per scale group inside a unit: 4 (group
// sizes that are multiples of 128), 2 (64) and 1 (32), whose scales and zero
// points are staged in LDS as well (fewer activation rows make room: MT = 7
// and 6). Few rows take MT = 4 (bgemm_config).
//
// bf16 (BF). gfx950 has no packed bf16 subtract: B is 128 + q (exact) and a
// group's sum starts from -(128 + z) * sum x instead of 0; the row sums
// come from a pass over x ahead of the launch (bgemm_row_sums_kernel).
//
// Sources of the codes: the tiled copy (one contiguous 4 KiB block per panel and
// unit), or (RM) the row-major kernel layout, 64 bytes per row and unit, for
// callers without the copy.
//
// Numerics (fp16): those of the tiled GEMM. B = q - z exact (v_perm_b32 under a
// 0x64 exponent byte, one packed subtract); the products x (q - z) are exact in
// fp32; y += s * sum x (q - z) per group in fp32, the reference's w = (q - z) * s
// with fp32 accumulation (pare/kernels/matmul_int4.py:145-176).
// bf16: products x (128 + q) are exact as well, but a group's sum and its start are up
// to 143 |x| a term and cancel, as they do in the GEMV and the tiled GEMM's bf16
// variant: each of their roundings is 2^-24 of that. Below the rounding of y to bf16
// (1.7e-3) unless a column is some 10^4 times the others: against 64 bits, 64 x 512 x
// 4096, N(0, 1) activations, or those with a mean of 100, 1.65e-3 and 1.72e-3, the
// rounding itself; with two columns of 1e3 / 1e4 / 1e5 whose codes equal their zero
// points 1.66e-3 / 1.71e-3 / 4.1e-3 (the GEMV 1.66e-3 / 1.76e-3 / 6.0e-3).
#include <atomic>

#include "pmi_common.h"
#include "pmi_launch.h"

namespace pmi {
namespace {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct BgemmArgs {
  const uint16_t* x;     // fp16 or bf16 [M, K]
  const uint8_t* w;      // tiled weights, or kernel layout [N, K/2] (RM)
  const float* s_gm;     // fp32 [G, N]
  const uint8_t* z_gm;   // u8 [G, N]
  const float* sums;     // BF: row sums of x per scale group of a unit, [.., sums_ld]
  uint16_t* y;           // [M, N]
  float* part;           // splits > 1: partial tiles
  int M, N, K, gs;
  int n_panels, n_bands, grid_m, splits;
  int chunk;             // workgroups per XCD
  int sums_ld;
  int glu;               // fp16, tiled, 128-column groups: y [M, N / 2] = silu(gate) * up
};

template <int MT, int KSG, bool BF>
struct Shape {
  static constexpr int kRows = 16 * MT;
  static constexpr int kX = kRows * 256;                  // one activation slot
  static constexpr int kGU = 4 / KSG;                     // scale groups per unit
  static constexpr bool kSzLds = KSG < 4 || BF;           // scales and zero points in LDS
  static constexpr int kSz = kSzLds ? kGU * 1280 : 0;     // 256 rows x (4 + 1) bytes a group
  // row sums, in whole 64-lane copies (a copy's last lanes may hold nothing)
  static constexpr int kXs = BF ? (kGU * kRows * 4 + 255) / 256 * 256 : 0;
  static constexpr int kW = 2 * kX;                       // offset of the codes
  static constexpr int kS = kW + 4 * 4096;                // offset of the s/z slots
  static constexpr int kR = kS + 2 * kSz;                 // offset of the row-sum slots
  static constexpr int kGroup = kR + 2 * kXs;             // LDS of one four-wave group
  static_assert(kGroup <= 80 * 1024, "two groups fit the LDS of a CU");
};

// Buffer descriptor in SGPRs (untyped dwords, no swizzle) for the copies
// below.
PMI_DEV u32x4 descriptor(const void* p, uint32_t bytes) {
  const uint64_t a = (uint64_t)p;
  u32x4 d = {(uint32_t)a, (uint32_t)(a >> 32) & 0xFFFFu, bytes, 0x00020000u};
#pragma unroll
  for (int i = 0; i < 4; ++i) d[i] = __builtin_amdgcn_readfirstlane(d[i]);
  return d;
}

// 16 (or 4) bytes per lane from a buffer to LDS address base + 16 (4) * lane.
// base is uniform. No register but m0 is written, which is reserved (a clobber list
// may not name it): the compiler sets it right ahead of each of its own uses, and
// has none in this kernel. The caller waits with wait_vmcnt<0>.
PMI_DEV void dma16(u32x4 r, uint32_t base, int voff, int soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(base),
               "v"(voff), "s"(r), "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory");
#else
  (void)r, (void)base, (void)voff, (void)soff;
#endif
}
PMI_DEV void dma4(u32x4 r, uint32_t base, int voff, int soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(base),
               "v"(voff), "s"(r), "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory");
#else
  (void)r, (void)base, (void)voff, (void)soff;
#endif
}

template <bool BF>
PMI_DEV f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (BF)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Rows m .. m + 3 (v[j][e]: row m + e, column row0 + j) to y.
template <bool BF>
PMI_DEV void store_rows(uint16_t* __restrict__ y, const f32x4* v, int m, int M, int N, int row0) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (m + e >= M) continue;
    u32x2 o;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      uint32_t v0, v1;
      if constexpr (BF) {
        v0 = f32_to_bf16_rne(v[2 * q][e]);
        v1 = f32_to_bf16_rne(v[2 * q + 1][e]);
      } else {
        v0 = __builtin_bit_cast(uint16_t, f32_to_f16_rne(v[2 * q][e]));
        v1 = __builtin_bit_cast(uint16_t, f32_to_f16_rne(v[2 * q + 1][e]));
      }
      o[q] = v0 | (v1 << 16);
    }
    *reinterpret_cast<u32x2*>(y + (size_t)(m + e) * N + row0) = o;
  }
}

// The same rows of a gate/up weight in pmi_matmul_w4a16_gate_up_silu's row order
// (v[0], v[1] gate, v[2], v[3] up of output columns col, col + 1): silu(gate) * up
// with the roundings of the plain matmul followed by pmi_silu_mul_f16.
PMI_DEV void store_rows_glu(uint16_t* __restrict__ y, const f32x4* v, int m, int M, int ld, int col) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (m + e >= M) continue;
    uint32_t h[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) h[j] = __builtin_bit_cast(uint16_t, f32_to_f16_rne(v[j][e]));
    *reinterpret_cast<uint32_t*>(y + (size_t)(m + e) * ld + col) = glu_pair(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
  }
}

template <int MT, int KSG, bool BF, int KG, bool RM>
__global__ __launch_bounds__(256 * KG, 2) void w4a16_bgemm_kernel(BgemmArgs a) {
  using S = Shape<MT, KSG, BF>;
  constexpr int GU = S::kGU;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_all[];

  const int tid = threadIdx.x, l = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kgrp = KG == 1 ? 0 : wave >> 2, wv = wave & 3;
  // Workgroup 8 k + x runs on XCD x and takes entry x chunk + k of the list
  // (activation block, split, band), band fastest: the bands that share
  // activation rows share an XCD's L2. A placement preference only.
  const int x8 = blockIdx.x % 8, k8 = blockIdx.x / 8;
  const int L = x8 * a.chunk + k8;
  if (k8 >= a.chunk || L >= a.n_bands * a.splits * a.grid_m) return;  // padding (uniform)
  const int band = L % a.n_bands, rest = L / a.n_bands;
  const int sp = rest % a.splits, mb = rest / a.splits;
  const int M = a.M, N = a.N, K = a.K;
  const int U = K >> 7;
  const int u_lo = (int)((int64_t)U * sp / a.splits), u_hi = (int)((int64_t)U * (sp + 1) / a.splits);
  const int m0 = S::kRows * mb;
  const int p = band * 4 + wv;
  const int pc = p < a.n_panels ? p : a.n_panels - 1;

  uint8_t* lds = lds_all + kgrp * S::kGroup;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  // Rows past M lie past the descriptor's end and read as zeros.
  const int rows = M - m0 < S::kRows ? M - m0 : S::kRows;
  const u32x4 dx = descriptor(a.x + (int64_t)m0 * K, (uint32_t)rows * K * 2);
  const u32x4 dw = descriptor(a.w, RM ? (uint32_t)N * (K >> 1) : (uint32_t)a.n_panels * 64 * (K >> 1));
  const int groups = K / a.gs;
  const u32x4 ds = descriptor(a.s_gm, (uint32_t)groups * N * 4);
  const u32x4 dz = descriptor(a.z_gm, (uint32_t)groups * N);
  const __amdgpu_buffer_rsrc_t rs = rsrc(a.s_gm, (int64_t)groups * N * 4);
  const __amdgpu_buffer_rsrc_t rz = rsrc(a.z_gm, (int64_t)groups * N);

  // Lane values that a unit needs once are worked out there, from an opaque
  // copy of the lane id: kept across the MFMAs they would spill.
  auto lane = [&]() {
    int v = l;
    asm volatile("" : "+v"(v));
    return v;
  };
  // Unit u (its first scale group: g) to slot b.
  auto copy_x = [&](int u, int b) {
    const int q = lane();
    const int row0 = 4 * MT * wv + (q >> 4);
    // chunk (q % 16) ^ (row % 16) of row row0 + 4 i
    const int r4 = (4 * MT * wv) & 15;
    const int base = row0 * K * 2;
#pragma unroll
    for (int i = 0; i < MT; ++i)
      dma16(dx, lds0 + b * S::kX + (wv * MT + i) * 1024,
            base + i * 8 * K + ((((q & 15) ^ (q >> 4)) << 4) ^ (((r4 + 4 * i) & 12) << 4)), u * 256);
  };
  auto copy_w = [&](int u) {
    const int q = lane();
    const uint32_t base = lds0 + S::kW + wv * 4096;
    if constexpr (RM) {
      // tile j: 16-byte chunk c of row 4 n + j at (16 c + n) * 16
      int r0 = 64 * p + 4 * (q & 15);
      r0 = r0 < N ? r0 : N - 4;
      const int v = r0 * (K >> 1) + 16 * (q >> 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) dma16(dw, base + j * 1024, v + j * (K >> 1), u * 64);
    } else {
      const int so = (pc * U + u) * 4096;
#pragma unroll
      for (int j = 0; j < 4; ++j) dma16(dw, base + j * 1024, 16 * q, so + j * 1024);
    }
  };
  // Scales and zero points of the band's 256 rows, wave w the unit's group w,
  // and the rows' sums (BF).
  auto copy_sz = [&](int u, int g, int b) {
    if constexpr (S::kSzLds) {
      const int q = lane();
      if (wv < GU) {
        int r0 = 256 * band + 4 * q;
        r0 = r0 < N ? r0 : N - 4;
        const uint32_t base = lds0 + S::kS + b * S::kSz + wv * 1280;
        dma16(ds, base, r0 * 4, (g + wv) * N * 4);
        dma4(dz, base + 1024, r0, (g + wv) * N);
      }
      if constexpr (BF) {
        constexpr int n = GU * S::kRows;  // floats: GU runs of kRows, at most two per lane of a group
        const u32x4 dr = descriptor(a.sums + (int64_t)u * GU * a.sums_ld, (uint32_t)GU * a.sums_ld * 4);
#pragma unroll
        for (int k = 0; k < (n + 255) / 256; ++k) {
          const int f0 = (4 * k + wv) * 64;  // this wave's first float
          if (f0 < n) {
            int f = f0 + q;
            f = f < n ? f : n - 1;
            const int gg = f / S::kRows;
            dma4(dr, lds0 + S::kR + b * S::kXs + f0 * 4, (gg * a.sums_ld + m0 + f - gg * S::kRows) * 4, 0);
          }
        }
      }
    }
  };
  f32x4 s_next = {};  // fp16, group sizes of 128 and more: the next unit's
  uint32_t z_next = 0;
  auto load_sz = [&](int g) {
    if constexpr (!S::kSzLds) {
      int r0 = 64 * p + 4 * (lane() & 15);
      r0 = r0 < N ? r0 : N - 4;
      s_next = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, r0 * 4, g * N * 4, 0));
      z_next = __builtin_amdgcn_raw_buffer_load_b32(rz, r0, g * N, 0);
    }
  };

  f32x4 acc[MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

  // group of unit u: u / units-per-group, stepped without a division
  const int upg = KSG == 4 ? a.gs >> 7 : 1;
  int u = u_lo + kgrp, g, ug;
  if constexpr (KSG == 4) {
    g = u / upg;
    ug = u - g * upg;
  } else {
    g = GU * u;
    ug = 0;
  }
  {
    const bool in = u < u_hi;
    load_sz(in ? g : 0);
    if (in) {
      copy_w(u);
      copy_sz(u, g, 0);
      copy_x(u, 0);
    }
  }
  const int steps = (u_hi - u_lo + KG - 1) / KG;  // the same for both groups: they share the barriers
  for (int s = 0; s < steps; ++s, u += KG) {
    wait_vmcnt<0>();
    barrier_only();
    const int slot = s & 1;
    if (KG > 1 && u >= u_hi) continue;  // the shorter group's last step (uniform per wave)

    // codes to registers; their LDS and the other slots may then be refilled
    const uint8_t* wb = lds + S::kW + wv * 4096;
    u32x4 w[4];
    u32x2 w32[4][4];  // RM, 32-column groups: one 8-byte piece per k-step
    {
      const int q = lane();
      if constexpr (RM && KSG == 1) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < 4; ++t)
            w32[j][t] = *reinterpret_cast<const u32x2*>(wb + j * 1024 + t * 256 + 16 * (q & 15) + 8 * ((q >> 4) & 1));
#pragma unroll
        for (int j = 0; j < 4; ++j)
          asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(w32[j][0]), "+v"(w32[j][1]), "+v"(w32[j][2]), "+v"(w32[j][3])::"memory");
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (RM) {
            const int o = j * 1024 + 256 * (q >> 5) + 16 * (q & 15) + 8 * ((q >> 4) & 1);
            const u32x2 lo = *reinterpret_cast<const u32x2*>(wb + o);
            const u32x2 hi = *reinterpret_cast<const u32x2*>(wb + o + 512);
            w[j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
          } else {
            w[j] = *reinterpret_cast<const u32x4*>(wb + j * 1024 + 16 * q);
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3])::"memory");
      }
    }
    f32x4 sc[GU];
    uint32_t zq[GU];
    if constexpr (S::kSzLds) {
      const int q = lane();
      const uint8_t* sb = lds + S::kS + slot * S::kSz + 256 * wv + 16 * (q & 15);
      const uint8_t* zb = lds + S::kS + slot * S::kSz + 1024 + 64 * wv + 4 * (q & 15);
#pragma unroll
      for (int gg = 0; gg < GU; ++gg) {
        sc[gg] = *reinterpret_cast<const f32x4*>(sb + gg * 1280);
        zq[gg] = *reinterpret_cast<const uint32_t*>(zb + gg * 1280);
      }
    } else {
      sc[0] = s_next;
      zq[0] = z_next;
    }
    const bool more = u + KG < u_hi;
    if constexpr (KSG == 4) {
#pragma unroll
      for (int n = 0; n < KG; ++n)
        if (++ug == upg) ug = 0, ++g;
    } else {
      g += GU * KG;
    }
    load_sz(more ? g : 0);
    if (more) {
      copy_w(u + KG);
      copy_sz(u + KG, g, slot ^ 1);
      copy_x(u + KG, slot ^ 1);
    }

    // A operand of k-step t: row n of each tile, chunk (4 t + h) ^ n
    int ao[4];
    {
      const int q = lane();
      const int o = ((q & 15) << 8) + (((q & 15) ^ (q >> 4)) << 4);
#pragma unroll
      for (int t = 0; t < 4; ++t) ao[t] = o ^ (64 * t);
    }
    const uint8_t* xb = lds + slot * S::kX;
    u32x4 A[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) A[t] = *reinterpret_cast<const u32x4*>(xb + ao[t]);
    f32x4 xs[BF ? GU : 1];
    const uint8_t* rb = lds + S::kR + slot * S::kXs;
    int ro = 0;
    if constexpr (BF) {
      ro = (lane() >> 4) << 4;
#pragma unroll
      for (int gg = 0; gg < GU; ++gg) xs[gg] = *reinterpret_cast<const f32x4*>(rb + ro + gg * S::kRows * 4);
    }

    u32x4 B[4][4];
    float zf[GU][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint32_t z = (zq[t / KSG] >> (8 * j)) & 0xFFu;
        uint32_t w0, w1;
        if constexpr (RM && KSG == 1) {
          const int sh = 4 * (lane() >> 5);
          w0 = w32[j][t][0] >> sh, w1 = w32[j][t][1] >> sh;
        } else {
          // tiled and 128-column groups: k-steps (0, 1) low nibbles, (2, 3) high;
          // row-major 64-column groups: low and high nibbles alternate
          const int piece = RM && KSG == 2 ? t >> 1 : t & 1, high = RM && KSG == 2 ? t & 1 : t >> 1;
          w0 = w[j][2 * piece], w1 = w[j][2 * piece + 1];
          if (high) w0 >>= 4, w1 >>= 4;
        }
        w0 &= 0x0F0F0F0Fu, w1 &= 0x0F0F0F0Fu;
        if constexpr (BF) {
          B[j][t] = __builtin_bit_cast(u32x4, b_operand_bf16(w0, w1));
          if (t % KSG == 0) zf[t / KSG][j] = -(128.f + (float)z);
        } else {
          B[j][t] = __builtin_bit_cast(u32x4, b_operand(w0, w1, as_f16x2(neg_magic_zero_x2(z))));
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    // step (i, q, gg): activation tile i, weight tiles 2 q and 2 q + 1, scale group gg
    f32x4 cg[2][2];
    int pi = 0, pq = 0, pg = 0;  // the step whose fold is pending
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int gg = 0; gg < GU; ++gg) {
          const int buf = ((2 * i + q) * GU + gg) & 1;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            if constexpr (BF) {
#pragma unroll
              for (int e = 0; e < 4; ++e) cg[buf][j][e] = xs[gg][e] * zf[gg][2 * q + j];
            }
          }
          if (BF && q == 1 && i + 1 < MT)
            xs[gg] = *reinterpret_cast<const f32x4*>(rb + ro + (gg * S::kRows + 16 * (i + 1)) * 4);
#pragma unroll
          for (int t = gg * KSG; t < (gg + 1) * KSG; ++t) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
              cg[buf][j] = mfma<BF>(A[t], B[2 * q + j][t], !BF && t == gg * KSG ? zero4 : cg[buf][j]);
            if (q == 1 && i + 1 < MT) A[t] = *reinterpret_cast<const u32x4*>(xb + ao[t] + (i + 1) * 4096);
          }
          if (i + q + gg > 0) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                acc[pi][2 * pq + j][e] = fmaf(sc[pg][2 * pq + j], cg[buf ^ 1][j][e], acc[pi][2 * pq + j][e]);
          }
          pi = i, pq = q, pg = gg;
          // MFMAs first (the pending sums' last ones are still in flight), then
          // two folds to each
          if constexpr (KSG == 4 && !BF) {
            __builtin_amdgcn_sched_group_barrier(0x8, 3, 0);
#pragma unroll
            for (int n = 0; n < 4; ++n) {
              __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
              __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
              if (q) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc[MT - 1][2 + j][e] = fmaf(sc[GU - 1][2 + j], cg[(2 * MT * GU - 1) & 1][j][e], acc[MT - 1][2 + j][e]);
    __builtin_amdgcn_s_setprio(0);
  }

  const int t256 = tid & 255;
  constexpr int H = KG == 1 ? MT : (MT + 1) / 2;  // activation tiles that group 0 finishes
  if constexpr (KG == 2) {
    // each group hands the other the tiles that one finishes
    __syncthreads();
    f32x4* ex = reinterpret_cast<f32x4*>(lds_all);
    if (kgrp == 1) {
#pragma unroll
      for (int i = 0; i < H; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) ex[(4 * i + j) * 256 + t256] = acc[i][j];
    } else {
#pragma unroll
      for (int i = H; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) ex[(4 * i + j) * 256 + t256] = acc[i][j];
    }
    __syncthreads();
    if (kgrp == 0) {
#pragma unroll
      for (int i = 0; i < H; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += ex[(4 * i + j) * 256 + t256];
    } else {
#pragma unroll
      for (int i = H; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += ex[(4 * i + j) * 256 + t256];
    }
  }

  if (a.splits > 1) {
    // partial tile of split sp: [4 i + j][thread] x 16 bytes, for the combine
    float* part = a.part + ((size_t)(mb * a.n_bands + band) * a.splits + sp) * (MT * 4 * 256 * 4);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (KG == 2 && (i < H) != (kgrp == 0)) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) reinterpret_cast<f32x4*>(part)[(4 * i + j) * 256 + t256] = acc[i][j];
    }
    return;
  }

  // lane (n, h): activation rows m0 + 16 i + 4 h + e, weight rows row0 .. row0 + 3
  const int row0 = 64 * p + 4 * (l & 15);
  if (p >= a.n_panels || row0 >= N) return;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    if (KG == 2 && (i < H) != (kgrp == 0)) continue;
    const int m = m0 + 16 * i + 4 * (l >> 4);
    if constexpr (!BF && !RM && KSG == 4) {
      if (a.glu) {
        store_rows_glu(a.y, acc[i], m, M, N / 2, 32 * p + 2 * (l & 15));
        continue;
      }
    }
    store_rows<BF>(a.y, acc[i], m, M, N, row0);
  }
}

// Split K: y = the partial tiles added in split order, one thread per four
// activation rows x four weight rows. A launch of its own: the last workgroup
// of a tile adding them alone read up to 1 MiB by itself (8 splits: 27 us for
// 1024 x 4096 at M = 128, of which the products are a quarter).
template <int MT, bool BF>
__global__ __launch_bounds__(256) void bgemm_combine_kernel(const float* __restrict__ part,
                                                            uint16_t* __restrict__ y, int M, int N,
                                                            int n_bands, int splits) {
  const int t = threadIdx.x, l = t & 63;
  const int i = blockIdx.x % MT, tl = blockIdx.x / MT;
  const int band = tl % n_bands, mb = tl / n_bands;
  const int row0 = 256 * band + 64 * (t >> 6) + 4 * (l & 15);
  const int m = 16 * (MT * mb + i) + 4 * (l >> 4);
  if (row0 >= N || m >= M) return;
  constexpr int kPart = MT * 4 * 256;  // f32x4 per partial tile
  const f32x4* src = reinterpret_cast<const f32x4*>(part) + (size_t)tl * splits * kPart + 4 * i * 256 + t;
  f32x4 v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = src[j * 256];
  for (int q = 1; q < splits; ++q)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += src[(size_t)q * kPart + j * 256];
  store_rows<BF>(y, v, m, M, N, row0);
}

// sums[k / cols][m] = sum of the bf16 row x[m] over columns k .. k + cols - 1
// (cols 32, 64 or 128: lanes = cols / 8 neighbouring lanes), 8 columns per thread;
// K % 128 == 0, so a run of lanes lies in one row. 1003 x 4096: 8.3 us with a wave
// per row, 5.3 with a thread per 8 columns.
__global__ __launch_bounds__(256) void bgemm_row_sums_kernel(const uint16_t* __restrict__ x,
                                                             float* __restrict__ sums, uint32_t n,
                                                             uint32_t chunks, uint32_t chunks_m, int lanes,
                                                             int ld) {
  const uint32_t i0 = blockIdx.x * 256 + threadIdx.x, i = i0 < n ? i0 : n - 1;
  const u32x4 d = *reinterpret_cast<const u32x4*>(x + (size_t)i * 8);
  float v = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    v += __builtin_bit_cast(float, d[k] << 16) + __builtin_bit_cast(float, d[k] & 0xFFFF0000u);
  for (int o = lanes >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o);
  const uint32_t m = udiv(i, chunks, chunks_m), c = i - m * chunks;
  if (i0 < n && c % lanes == 0) sums[(size_t)(c / lanes) * ld + m] = v;
}

template <int MT, int KSG, bool BF, int KG, bool RM>
hipError_t launch_one(const BgemmArgs& a, int grid, size_t lds, hipStream_t stream) {
  static std::atomic<uint64_t> allowed{0};
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  const uint64_t bit = 1ull << (dev & 63);
  const void* fn = reinterpret_cast<const void*>(&w4a16_bgemm_kernel<MT, KSG, BF, KG, RM>);
  if (!(allowed.load() & bit)) {
    if (hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        e != hipSuccess)
      return e;
    allowed.fetch_or(bit);
  }
  hipLaunchKernelGGL((w4a16_bgemm_kernel<MT, KSG, BF, KG, RM>), dim3(grid), dim3(256 * KG), lds, stream, a);
  return hipGetLastError();
}

template <int MT, int KSG, bool BF>
hipError_t launch_shape(const BgemmArgs& a, const BgemmConfig& c, bool rm, hipStream_t stream) {
  const size_t lds = (size_t)c.kg * Shape<MT, KSG, BF>::kGroup;
  hipError_t e;
  if (c.kg == 2)
    e = rm ? launch_one<MT, KSG, BF, 2, true>(a, c.grid, lds, stream)
           : launch_one<MT, KSG, BF, 2, false>(a, c.grid, lds, stream);
  else
    e = rm ? launch_one<MT, KSG, BF, 1, true>(a, c.grid, lds, stream)
           : launch_one<MT, KSG, BF, 1, false>(a, c.grid, lds, stream);
  if (e != hipSuccess || a.splits == 1) return e;
  hipLaunchKernelGGL((bgemm_combine_kernel<MT, BF>), dim3(MT * a.n_bands * a.grid_m), dim3(256), 0, stream,
                     a.part, a.y, a.M, a.N, a.n_bands, a.splits);
  return hipGetLastError();
}

// MT: the most activation tiles whose LDS fits twice on a CU, or 4 (bgemm_config).
template <int MT, int KSG, bool BF>
hipError_t launch_mt(const BgemmArgs& a, const BgemmConfig& c, bool rm, hipStream_t stream) {
  if (c.mt == 4) return launch_shape<4, KSG, BF>(a, c, rm, stream);
  return launch_shape<MT, KSG, BF>(a, c, rm, stream);
}

}  // namespace

BgemmConfig bgemm_config(int64_t M, int64_t N, int64_t K, int64_t gs, bool bf16) {
  BgemmConfig c{};
  c.ok = false;
  if (M < 1 || N < 4 || N % 4 != 0 || K % 128 != 0 || K < 128 || K % gs != 0) return c;
  if (gs != 32 && gs != 64 && gs % 128 != 0) return c;
  if (M * K * 2 >= (1ll << 31) || ((N + 63) / 64) * 64 * (K / 2) >= (1ll << 31)) return c;
  c.mt = gs == 32 ? 6 : (gs == 64 || bf16) ? 7 : 8;
  // Up to 64 rows, and where 128 rows take two of the taller tiles: tiles of 64
  // rows, whose products and folds are not spent on rows that are not there (us,
  // tall tiles / these): bf16 14336 x 4096 at M = 32 / 64 / 120 26.5 / 27.7 / 43.2
  // against 21.6 / 22.4 / 34.1; 28672 x 4096 at M = 113 66.0 against 49.2; gs 64 at
  // M = 40 / 128 31.7 / 47.4 against 26.9 / 38.4; gs 32, 4096 x 14336 at M = 100 40.5
  // against 33.4.
  if (M <= 64 || (M > 16 * c.mt && M <= 128)) c.mt = 4;
  const int64_t bands = ((N + 63) / 64 + 3) / 4;
  const int64_t gm = (M + 16 * c.mt - 1) / (16 * c.mt);
  const int64_t cus = device_cu_count(), tiles = bands * gm, units = K / 128;
  c.n_bands = (int)bands;
  c.grid_m = (int)gm;
  // One workgroup of two groups per CU up to one tile per CU; past that two
  // workgroups of one group.
  c.kg = tiles <= cus && units > 1 ? 2 : 1;
  // Fewer tiles than half the CUs: split K, at least kMinUnits units a split.
  constexpr int kMinUnits = 4;
  int64_t splits = 1;
  if (2 * tiles <= cus) {
    splits = cus / tiles;
    if (splits > units / kMinUnits) splits = units / kMinUnits;
    if (splits > 16) splits = 16;
    if (splits < 1) splits = 1;
  }
  c.splits = (int)splits;
  c.ws_split = splits > 1 ? (size_t)tiles * splits * c.mt * 4 * 256 * 16 : 0;
  c.sums_ld = (int)(gm * 16 * c.mt);
  c.ws_sums = bf16 ? ws_align((size_t)(K / (gs < 128 ? gs : 128)) * c.sums_ld * 4) : 0;
  const int64_t chunk = (tiles * splits + 7) / 8;
  if (8 * chunk >= (1ll << 31)) return c;
  c.chunk = (int)chunk;
  c.grid = (int)(8 * chunk);
  c.ok = true;
  return c;
}

bool bgemm_glu_supported(int64_t M, int64_t N, int64_t K, int64_t gs) {
  if (M <= 64 || N % 64 != 0 || gs % 128 != 0) return false;
  const BgemmConfig c = bgemm_config(M, N, K, gs);
  return c.ok && c.splits == 1 && (int64_t)c.n_bands * c.grid_m * 4 >= 3 * (int64_t)device_cu_count();
}

hipError_t launch_bgemm(const void* x, const uint8_t* w_tiled, const uint8_t* w_kernel, const float* scales_gm,
                        const uint8_t* zeros_gm, void* y, int64_t M, int64_t N, int64_t K, int64_t gs,
                        bool bf16, void* workspace, size_t ws_bytes, size_t ws_offset, hipStream_t stream,
                        bool glu) {
  BgemmConfig c = bgemm_config(M, N, K, gs, bf16);
  if (!c.ok || (glu && !bgemm_glu_supported(M, N, K, gs))) return hipErrorInvalidValue;
  BgemmArgs a{};
  a.glu = glu;
  size_t off = ws_offset;
  if (bf16) {
    if (!workspace || ws_bytes < off + c.ws_sums) return hipErrorInvalidValue;
    float* sums = (float*)((uint8_t*)workspace + off);
    off += c.ws_sums;
    const uint32_t n = (uint32_t)(M * (K / 8)), chunks = (uint32_t)(K / 8);
    hipLaunchKernelGGL(bgemm_row_sums_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, (const uint16_t*)x,
                       sums, n, chunks, udiv_magic(chunks), (int)((gs < 128 ? gs : 128) / 8), c.sums_ld);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    a.sums = sums;
  }
  if (c.splits > 1 && (!workspace || ws_bytes < off + c.ws_split)) {
    c.splits = 1;  // no room for the partial tiles
    c.chunk = (c.n_bands * c.grid_m + 7) / 8;
    c.grid = 8 * c.chunk;
  }
  const bool rm = w_tiled == nullptr;
  a.x = (const uint16_t*)x;
  a.w = rm ? w_kernel : w_tiled;
  a.s_gm = scales_gm;
  a.z_gm = zeros_gm;
  a.y = (uint16_t*)y;
  a.part = (float*)((uint8_t*)workspace + off);
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.gs = (int)gs;
  a.n_panels = (int)((N + 63) / 64);
  a.n_bands = c.n_bands;
  a.grid_m = c.grid_m;
  a.splits = c.splits;
  a.chunk = c.chunk;
  a.sums_ld = c.sums_ld;
  if (gs == 32) return bf16 ? launch_mt<6, 1, true>(a, c, rm, stream) : launch_mt<6, 1, false>(a, c, rm, stream);
  if (gs == 64) return bf16 ? launch_mt<7, 2, true>(a, c, rm, stream) : launch_mt<7, 2, false>(a, c, rm, stream);
  return bf16 ? launch_mt<7, 4, true>(a, c, rm, stream) : launch_mt<8, 4, false>(a, c, rm, stream);
}

}  // namespace pmi
