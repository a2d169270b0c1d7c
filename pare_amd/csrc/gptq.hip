// GPTQ producer kernels (pare/schemes/gptq.py:156-263): the sequential column
// loop of one 128-column block, the per-group scale/zero of the dynamic-group
// (desc_act) variant, the final un-permute + INT4 pack, and the diagonal blocks
// of the inverse Hessian's factor. The rest of the factor and the lazy update of
// the columns right of a block are GEMMs driven by the host.
//
// Rows are independent in GPTQ: row n's codes depend only on W[n, :] and the
// shared factor C.
#include "../../include/pare_amd.h"
#include "pmi_common.h"
#include "pmi_launch.h"

namespace pmi {
namespace {

constexpr int kRows = 16;       // rows of W per workgroup, 16 lanes each
constexpr int kThreads = 256;
constexpr int kBlk = 128;       // GPTQ block (gptq.py:42)
constexpr int kSlots = 8;       // columns of a block per lane

// f(0), ..., f(N - 1) with compile-time arguments.
template <int I>
struct Index {
  static constexpr int value = I;
};
template <int N, int I = 0, typename F>
PMI_DEV void static_for(F&& f) {
  if constexpr (I < N) {
    f(Index<I>{});
    static_for<N, I + 1>(f);
  }
}

// scale[n, g], zero[n, g] from W[n, c0 : c0 + cols] (row stride ldw), one
// wave per row.
__global__ void group_params_kernel(const float* __restrict__ w, int64_t ldw, int64_t N,
                                    int64_t c0, int64_t cols, int sym, float* __restrict__ scale,
                                    float* __restrict__ zero, int64_t G, int64_t g) {
  const int lane = threadIdx.x & 63;
  const int64_t n = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (n >= N) return;
  const float* row = w + n * ldw + c0;
  float mn = __builtin_inff(), mx = -__builtin_inff();
  for (int64_t c = lane; c < cols; c += 64) {
    mn = fminf(mn, row[c]);
    mx = fmaxf(mx, row[c]);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o, 64));
    mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  }
  float s, z;
  scale_zero_from_minmax(mn, mx, sym, s, z);
  if (lane == 0) {
    scale[n * G + g] = s;
    zero[n * G + g] = z;
  }
}

// a / b correctly rounded, from y = the refined reciprocal of b (Markstein): one
// remainder step in place of a division sequence, which is most of the column
// loop's dependent chain. Exact while nothing leaves the range of normal numbers on
// the way; the kernel below says what it checks for that.
PMI_DEV float reciprocal(float b) {
  float y = __builtin_amdgcn_rcpf(b);
  y = fmaf(fmaf(-b, y, 1.0f), y, y);
  return fmaf(fmaf(-b, y, 1.0f), y, y);
}
PMI_DEV float quotient(float a, float b, float y) {
  const float q = a * y;
  return fmaf(fmaf(-b, q, a), y, q);
}

// Lane L's value in every lane of its row of 16.
template <int L>
PMI_DEV float row_lane(float v) {
  const int i = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, 0x150 + L, 0xF, 0xF, false));
}

// One GPTQ block, columns b0 .. b0 + count - 1 of the permuted W [N, K]:
// per column j, q = clamp(rint(w / s + z), 0, 15) with the scale/zero of group
// colg[j]; e = (w - (q - z) s) / C[j, j]; every later column of the block
// gets w -= e * C[j, later], in order of j (one rounded product and one
// subtraction per step, as gptq.py:241-249 computes it). Writes the codes to
// qt [K, N] (processed column order, column-major so stores coalesce) and the
// errors to et [count, N] for the host's lazy update.
//
// Sixteen lanes share a row of W, lane t holding columns t, t + 16, ... in
// registers; a column's value, scale, zero point and C[j, j] reach the other
// lanes by DPP, each works out q and e for itself and updates its own columns.
// 16 rows per workgroup give one workgroup per CU at N = 4096; the chain of a
// column (about 25 dependent instructions) times 128 columns bounds the launch.
// 4096 rows, count 128: 148 us with a lane per row (32 workgroups), 24.9 this way.
// Quotients come from reciprocals while |s| and |C[j, j]| lie in [2^-40, 2^60] and
// every |w - (q - z) s| is 0 or in [2^-62, 2^60): then |w / s| < 2^107, 2^-122 < |e| <
// 2^100 and the remainders are exact. A workgroup that meets anything else
// (infinities, NaN, zero or denormal scales, overflowing updates) runs its rows
// again with divisions. The checks cost 1.0 of the 24.9 us.
// The updates also reach the columns at and before j, which nothing reads any
// more.
__global__ __launch_bounds__(kThreads) void gptq_block_kernel(
    const float* __restrict__ w, const float* __restrict__ c, const int32_t* __restrict__ colg,
    const float* __restrict__ scale, const float* __restrict__ zero, uint8_t* __restrict__ qt,
    float* __restrict__ et, int64_t N, int64_t K, int64_t G, int64_t b0, int count) {
  __shared__ float cl[(kBlk + 1) * kBlk];  // C[b0 + j][b0 + k] at [j][k]; the last row is padding
  __shared__ float el[kBlk * kRows];       // errors [j][row]
  __shared__ uint8_t ql[kBlk * kRows];     // codes [j][row]
  const int tid = threadIdx.x, t = tid & 15, r = tid >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * kRows;
  const int64_t n = n0 + r < N ? n0 + r : N - 1;  // rows past the end repeat the last one

  float wr[kSlots], s[kSlots], z[kSlots];
  auto load = [&]() {
#pragma unroll
    for (int m = 0; m < kSlots; ++m) {
      const int k = 16 * m + t < count ? 16 * m + t : t;
      const int64_t g = min(max((int64_t)colg[b0 + k], (int64_t)0), G - 1);
      wr[m] = w[n * K + b0 + k];
      s[m] = scale[n * G + g];
      z[m] = zero[n * G + g];
    }
  };
  auto magnitude = [](float v) { return __builtin_bit_cast(uint32_t, v) & 0x7FFFFFFFu; };
  constexpr uint32_t kLo = (127 - 62) << 23, kDenLo = (127 - 40) << 23, kHi = (127 + 60) << 23;
  load();
  for (int i = tid; i < kBlk * kBlk / 4; i += kThreads) {
    const int j = i / (kBlk / 4), k = 4 * (i % (kBlk / 4));
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (j < count && k < count)
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = c[(b0 + j) * K + b0 + k + q];
    *reinterpret_cast<f32x4*>(cl + j * kBlk + k) = v;
  }
  if (tid < kBlk) cl[kBlk * kBlk + tid] = 0.f;
  __syncthreads();

  // least and largest magnitude of the numerators of e (less one: 0 is in order)
  uint32_t lo = ~0u, hi = 0;
  auto columns = [&](auto divide) {
    constexpr bool kDivide = decltype(divide)::value != 0;
    for (int m0 = 0; 16 * m0 < count; ++m0) {
      // slot 0 holds columns 16 m0 + t
      const float inv_s = kDivide ? 0.f : reciprocal(s[0]);
      float es = 0.f, qs = 0.f;
      auto step = [&](auto lane) {
        constexpr int L = decltype(lane)::value;
        const float* crow = cl + (16 * m0 + L) * kBlk + 16 * m0 + t;
        float cv[kSlots];
#pragma unroll
        for (int m = 0; m < kSlots; ++m) cv[m] = crow[16 * m];
        const float d = row_lane<L>(cv[0]), sj = row_lane<L>(s[0]), zj = row_lane<L>(z[0]);
        const float wj = row_lane<L>(wr[0]);
        const float ws = kDivide ? wj / sj : quotient(wj, sj, row_lane<L>(inv_s));
        const float q = fminf(fmaxf(rintf(ws + zj), 0.0f), 15.0f);
        const float num = wj - (q - zj) * sj;
        const float e = kDivide ? num / d : quotient(num, d, reciprocal(d));
        if constexpr (!kDivide) {
          const uint32_t u = magnitude(num);
          lo = min(lo, u - 1u), hi = max(hi, u);
        }
        es = t == L ? e : es;
        qs = t == L ? q : qs;
#pragma unroll
        for (int m = 0; m < kSlots; ++m) {
          const float p = e * cv[m];
          wr[m] = wr[m] - p;
        }
      };
      static_for<16>(step);
      el[(16 * m0 + t) * kRows + r] = es;
      ql[(16 * m0 + t) * kRows + r] = (uint8_t)(int)qs;
#pragma unroll
      for (int m = 0; m + 1 < kSlots; ++m) wr[m] = wr[m + 1], s[m] = s[m + 1], z[m] = z[m + 1];
    }
  };
  bool off = false;
#pragma unroll
  for (int m = 0; m < kSlots; ++m) off |= magnitude(s[m]) - kDenLo > kHi - kDenLo;
  if (tid < count) off |= magnitude(cl[tid * kBlk + tid]) - kDenLo > kHi - kDenLo;
  columns(Index<0>{});
  off |= lo < kLo - 1u || hi >= kHi;
  if (__syncthreads_or(off)) {  // (uniform; the first pass's results are overwritten)
    load();
    columns(Index<1>{});
  }
  __syncthreads();
  for (int i = tid; i < count * kRows; i += kThreads) {
    const int j = i / kRows, row = i % kRows;
    if (n0 + row >= N) continue;
    et[(int64_t)j * N + n0 + row] = el[i];
    qt[(b0 + j) * N + n0 + row] = ql[i];
  }
}

// ---- the factor of the inverse Hessian -------------------------------------
// Cholesky factor of one n x n block (n <= 128) of a row-major fp64 matrix, its
// lower triangle in and out (the strict upper triangle is not touched), and the
// inverse of the factor to inv [128, 128] (lower triangular, zeros elsewhere,
// rows and columns past n those of the identity). A pivot that is not positive
// sets *info and counts as 1.
//
// One workgroup: thread (ty, tx) holds rows ty + 32 r and columns tx + 16 c in
// registers. Step j publishes column j of the block and row j of the inverse in
// LDS (double-buffered: one barrier per step) and every thread applies the
// rank-1 update to its elements. Columns of the block are finished (and written
// out) in the order in which columns of the inverse start, so one array holds
// the inverse left of the current 16 columns and the block right of them (two
// arrays spilled). The 128 steps are a serial chain whose issue on one CU bounds
// it: 72 us a block (97 with a square root and a division per step and barriers that
// waited for the stores); with 4 x 8 contiguous elements per thread, one published
// vector and every element updated at every step, 122.
constexpr int kDiag = 128;

__global__ __launch_bounds__(512) void chol_diag_kernel(double* __restrict__ a, int64_t ld, int n,
                                                        double* __restrict__ inv, int32_t* __restrict__ info) {
  __shared__ double col[2][kDiag], row[2][kDiag];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  double Z[4][8];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int i = ty + 32 * r, k = tx + 16 * c;
      // the upper triangle mirrors the lower one (it is updated, never used)
      const int hi = k <= i ? i : k, lo = k <= i ? k : i;
      Z[r][c] = hi < n ? a[hi * ld + lo] : (i == k ? 1.0 : 0.0);
    }
  bool bad = false;
  static_for<8>([&](auto cc) {
    constexpr int c0 = decltype(cc)::value;  // columns 16 c0 .. 16 c0 + 15 of this round
    constexpr int rj = c0 / 2;               // their rows are slot rj of threads ty == j % 32
    double X0[4];                            // the inverse's columns tx + 16 c0
#pragma unroll
    for (int r = 0; r < 4; ++r) X0[r] = ty + 32 * r == tx + 16 * c0 ? 1.0 : 0.0;
#pragma unroll 1
    for (int jl = 0; jl < 16; ++jl) {
      const int j = 16 * c0 + jl, b = j & 1;
      const bool mine = ty == (j & 31);  // holds row j
      if (tx == jl)
#pragma unroll
        for (int r = rj; r < 4; ++r) col[b][ty + 32 * r] = Z[r][c0];
      if (mine) {
#pragma unroll
        for (int c = 0; c < c0; ++c) row[b][tx + 16 * c] = Z[rj][c];
        row[b][tx + 16 * c0] = X0[rj];
      }
      // the LDS writes are done; the factor's stores stay in flight
      wait_lgkm0();
      barrier_only();
      double d = col[b][j];
      if (!(d > 0.0)) bad = true, d = 1.0;
      // 1 / sqrt(d): the approximation, then two steps of y += y (1 - d y^2)
      // (1/2 + 3/8 (1 - d y^2)), each cubing the error
      double li = __builtin_amdgcn_rsq(d);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const double e = fma(-d * li, li, 1.0);
        li = fma(li * e, fma(0.375, e, 0.5), li);
      }
      // rows above the round's are finished
      double lr[4];
#pragma unroll
      for (int r = rj; r < 4; ++r) {
        lr[r] = col[b][ty + 32 * r] * li;
        if (r == rj) lr[r] = ty + 32 * r > j ? lr[r] : 0.0;
      }
      if (tx == jl) {
#pragma unroll
        for (int r = rj; r < 4; ++r) {
          const int i = ty + 32 * r;
          if (i >= j && i < n) a[i * ld + j] = i > j ? lr[r] : d * li;
        }
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        if (c >= c0) {
          double lc = col[b][tx + 16 * c] * li;
          if (c == c0) lc = tx > jl ? lc : 0.0;
#pragma unroll
          for (int r = rj; r < 4; ++r) Z[r][c] = fma(-lr[r], lc, Z[r][c]);
        }
        if (c <= c0) {
          const double x = row[b][tx + 16 * c] * li;
          if (c == c0) {
            if (mine) X0[rj] = x;
#pragma unroll
            for (int r = rj; r < 4; ++r) X0[r] = fma(-lr[r], x, X0[r]);
          } else {
            if (mine) Z[rj][c] = x;
#pragma unroll
            for (int r = rj; r < 4; ++r) Z[r][c] = fma(-lr[r], x, Z[r][c]);
          }
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) Z[r][c0] = X0[r];
  });
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int i = ty + 32 * r, k = tx + 16 * c;
      inv[i * kDiag + k] = k <= i ? Z[r][c] : 0.0;
    }
  if (bad && threadIdx.x == 0) *info = 1;
}

// packed[n, :] (storage layout, original column order) from the codes qt
// [K, N] in processed order: original column k was processed at step
// inv_perm[k] (identity when inv_perm is null). One thread per (n, 8 columns).
__global__ void gptq_pack_kernel(const uint8_t* __restrict__ qt, const int32_t* __restrict__ inv_perm,
                                 uint8_t* __restrict__ packed, int64_t N, int64_t K) {
  const int64_t words = K >> 3;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < words * N;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t wd = idx / N, n = idx - wd * N;
    uint32_t v = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t k = wd * 8 + i;
      const int64_t p = inv_perm ? (int64_t)inv_perm[k] : k;
      const int64_t j = (p >= 0 && p < K) ? p : k;
      v |= ((uint32_t)qt[j * N + n] & 0xFu) << (4 * i);
    }
    *reinterpret_cast<uint32_t*>(packed + n * (K >> 1) + wd * 4) = v;
  }
}

}  // namespace

hipError_t launch_gptq_group_params(const float* w, int64_t ldw, int64_t N, int64_t c0,
                                    int64_t cols, int sym, float* scale, float* zero, int64_t G,
                                    int64_t g, hipStream_t stream) {
  const int waves = 4;
  hipLaunchKernelGGL(group_params_kernel, dim3((unsigned)((N + waves - 1) / waves)),
                     dim3(64 * waves), 0, stream, w, ldw, N, c0, cols, sym, scale, zero, G, g);
  return hipGetLastError();
}

hipError_t launch_gptq_block(const float* w, const float* c, const int32_t* colg,
                             const float* scale, const float* zero, uint8_t* qt, float* et,
                             int64_t N, int64_t K, int64_t G, int64_t b0, int count,
                             hipStream_t stream) {
  hipLaunchKernelGGL(gptq_block_kernel, dim3((unsigned)((N + kRows - 1) / kRows)), dim3(kThreads), 0,
                     stream, w, c, colg, scale, zero, qt, et, N, K, G, b0, count);
  return hipGetLastError();
}

hipError_t launch_chol_diag(double* a, int64_t ld, int n, double* inv, int32_t* info, hipStream_t stream) {
  hipLaunchKernelGGL(chol_diag_kernel, dim3(1), dim3(512), 0, stream, a, ld, n, inv, info);
  return hipGetLastError();
}

hipError_t launch_gptq_pack(const uint8_t* qt, const int32_t* inv_perm, uint8_t* packed, int64_t N,
                            int64_t K, hipStream_t stream) {
  int64_t blocks = ((K / 8) * N + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(gptq_pack_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, qt, inv_perm,
                     packed, N, K);
  return hipGetLastError();
}

}  // namespace pmi
