// fp32 linear: Y[M, N] = X[M, K] . W[N, K]^T (+ bias[N]) on the fp32 matrix cores.
//
// Semantics: src/stateful_llm_compiler/backends/triton_linear.py:10-84 (IEEE
// fp32 products, fp32 accumulation, bias added in fp32) and the reference
// executor's F.linear (execution.py:694-705).
//
// v_mfma_f32_16x16x4_f32 multiplies fp32 operands exactly as an FMA does and
// accumulates in fp32 at twice the VALU's FMA rate (157 TFLOP/s against 79).
// One lane holds one k of one row per operand, and any assignment of k's to
// lanes is a valid one as long as both operands use the same: lane (row c,
// group g) takes the 16-byte chunk g of a 64-byte row segment, and the four
// MFMAs of the segment use elements 0..3 of the chunks, so every operand read
// is a 16-byte one and none is transposed.
//
//  * Prefill rows: a ring of LDS stages (as the 16-bit ring kernel in
//    linear.hip): producer waves stream X and W k-tiles of 32 floats (128-byte
//    rows, 16-byte chunks XOR-swizzled by row) with direct-to-LDS loads,
//    consumer waves only read LDS and issue MFMAs.  A k-tile keeps a SIMD's
//    matrix core busy for several times the cycles of its LDS reads, so two or
//    three stages cover the memory latency and two workgroups share a CU (one
//    fills the matrix cores while the other meets at its barrier: M4096 N4864
//    K896 320 us with four stages and one workgroup per CU, 281 with two).
//    W rows are the A operand, X rows the B operand: a lane then holds four
//    consecutive features of one row and stores them with one 16-byte store.
//  * Few rows: W streams from HBM once.  Up to 16 rows with N up to 20 per CU
//    run on 4 x 4 blocks (linear_f32_few_kernel), the rest on 16-feature
//    workgroups whose waves split K (linear_f32_rows_kernel).
//
// Measured, against one FMA chain per thread on 16 x 16 LDS tiles: M4096
// N4864 K896 2125 -> 281-285 us (127 TFLOP/s; a large library product reaches
// 153 on this card), M4096 N896 K4864 2268 -> 286, M250 N4864 K896 57 -> 28,
// M48 N896 K4864 179 -> 19, M8 N896 K4864 176 -> 9, M8 N151936 K896 336 -> 129
// (4.2 TB/s).
#include "common.hpp"

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mfma4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, int64_t bytes) {
  const uint64_t address = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(address));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(address >> 32));
  void* uniform = reinterpret_cast<void*>((static_cast<uint64_t>(hi) << 32) | lo);
  const int clamped = bytes > 0x7fffffff ? 0x7fffffff : static_cast<int>(bytes);
  return __builtin_amdgcn_make_buffer_rsrc(uniform, 0, __builtin_amdgcn_readfirstlane(clamped),
                                           0x00020000);
}
__device__ __forceinline__ f32x4_t load4(__amdgpu_buffer_rsrc_t rsrc, int offset) {
  return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, 0));
}
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t rsrc, unsigned char* lds,
                                          int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      rsrc, (__attribute__((address_space(3))) void*)lds, 16, voffset, soffset, 0, 0);
}

constexpr int kBK = 32;         // floats of K per ring tile
constexpr int kRow = kBK * 4;   // bytes of one tile row

__device__ __forceinline__ int lds_offset(int row, int chunk) {
  return row * kRow + ((chunk ^ (row & 7)) << 4);
}

// BM x BN output tile, CWM x CWN consumer waves, PW producer waves, S stages.
// K is a multiple of kBK.
template <int BM, int BN, int CWM, int CWN, int PW, int S>
__global__ __launch_bounds__((CWM * CWN + PW) * 64) void linear_f32_ring_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ y, int M, int N, int K, int64_t x_rs, int64_t y_rs, int n_tiles,
    int wide_store) {
  constexpr int CW = CWM * CWN;
  constexpr int TM = BM / CWM, TN = BN / CWN;   // consumer wave tile
  constexpr int FM = TM / 16, FN = TN / 16;
  constexpr int XB = BM * kRow;
  constexpr int kStage = (BM + BN) * kRow;
  constexpr int kOps = (BM + BN) / 8 / PW;      // 1 KB loads per producer wave and tile
  static_assert(((BM + BN) / 8) % PW == 0, "loads split evenly over the producers");
  static_assert((S - 2) * kOps <= 63, "the wait count fits vmcnt");
  __shared__ __attribute__((aligned(16))) unsigned char ring[S * kStage];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  // Consecutive workgroup ids go round-robin to the 8 XCDs: gather them per
  // XCD, then run groups of 8 M-tiles N-tile by N-tile, so that the tiles one
  // XCD holds at a time share rows in its L2.
  int m0, n0;
  {
    constexpr int kXcds = 8, kGroupM = 8;
    const int total = static_cast<int>(gridDim.x);
    const int m_tiles = total / n_tiles;
    const int per = total / kXcds;
    const int id = blockIdx.x;
    const int t = id < per * kXcds ? (id % kXcds) * per + id / kXcds : id;
    const int span = kGroupM * n_tiles;
    const int first_m = (t / span) * kGroupM;
    const int gm = m_tiles - first_m < kGroupM ? m_tiles - first_m : kGroupM;
    m0 = (first_m + (t % span) % gm) * BM;
    n0 = ((t % span) / gm) * BN;
  }
  const int ktiles = K / kBK;

  if (wave >= CW) {
    const int pw = wave - CW;
    const int64_t x_rows = M - m0 < BM ? M - m0 : BM;
    const int64_t w_rows = N - n0 < BN ? N - n0 : BN;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(x + m0 * x_rs, ((x_rows - 1) * x_rs + K) * 4);
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(w + static_cast<int64_t>(n0) * K, w_rows * K * 4);
    const __amdgpu_buffer_rsrc_t rnone = make_rsrc(x, 0);
    // Load i of this wave covers ring rows 8 * (pw + PW * i) .. + 7 of the
    // stacked X and W tile; lane L fills row L / 8, chunk L % 8.
    int voff[kOps];
    bool is_x[kOps];
#pragma unroll
    for (int i = 0; i < kOps; ++i) {
      const int row = 8 * (pw + PW * i) + lane / 8;
      const int chunk = (lane % 8) ^ (row & 7);
      is_x[i] = 8 * (pw + PW * i) < BM;
      voff[i] = is_x[i] ? static_cast<int>(row * x_rs * 4) + chunk * 16
                        : (row - BM) * K * 4 + chunk * 16;
    }
    auto issue = [&](int kt) {
      unsigned char* dst = ring + (kt % S) * kStage;
      const bool live = kt < ktiles;
      const int kb = __builtin_amdgcn_readfirstlane(live ? kt * kRow : 0);
#pragma unroll
      for (int i = 0; i < kOps; ++i) {
        // Past the last tile: an empty range, so every wait counts the same loads.
        if (is_x[i])
          lds_dma16(live ? rx : rnone, dst + (pw + PW * i) * 1024, voff[i], kb);
        else
          lds_dma16(live ? rw : rnone, dst + (pw + PW * i) * 1024, voff[i], kb);
      }
    };
#pragma unroll
    for (int t = 0; t < S - 1; ++t) issue(t);
    for (int kt = 0; kt < ktiles; ++kt) {
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"((S - 2) * kOps) : "memory");
      issue(kt + S - 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }

  const int c = lane & 15;
  const int g = lane >> 4;
  const int wm = wave / CWN;
  const int wn = wave % CWN;
  f32x4_t acc[FN][FM];
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto fragments = [&](int kt, int kk, f32x4_t (&a)[FN], f32x4_t (&b)[FM]) {
    const unsigned char* xs = ring + (kt % S) * kStage;
#pragma unroll
    for (int j = 0; j < FN; ++j)
      a[j] = *reinterpret_cast<const f32x4_t*>(xs + XB + lds_offset(wn * TN + j * 16 + c, kk * 4 + g));
#pragma unroll
    for (int i = 0; i < FM; ++i)
      b[i] = *reinterpret_cast<const f32x4_t*>(xs + lds_offset(wm * TM + i * 16 + c, kk * 4 + g));
  };
  auto multiply = [&](const f32x4_t (&a)[FN], const f32x4_t (&b)[FM]) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[j][i] = mfma4(a[j][e], b[i][e], acc[j][i]);
  };
  f32x4_t a0[FN], b0[FM], a1[FN], b1[FM];
  for (int kt = 0; kt < ktiles; ++kt) {
    __syncthreads();  // tile kt landed; the stage read before may be refilled
    fragments(kt, 0, a0, b0);
    fragments(kt, 1, a1, b1);
    multiply(a0, b0);
    multiply(a1, b1);
  }
  // Lane (row c of the X fragment, features 4g .. 4g + 3 of the W fragment).
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int n = n0 + wn * TN + j * 16 + 4 * g;
    if (n >= N) continue;
    f32x4_t bv = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (bias != nullptr) {
#pragma unroll
      for (int r = 0; r < 4; ++r) bv[r] = n + r < N ? bias[n + r] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = m0 + wm * TM + i * 16 + c;
      if (m >= M) continue;
      const f32x4_t v = bias != nullptr ? acc[j][i] + bv : acc[j][i];
      float* out = y + m * y_rs + n;
      if (wide_store) {
        *reinterpret_cast<f32x4_t*>(out) = v;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) out[r] = v[r];
      }
    }
  }
}

// 16 features by 16 * MB rows per workgroup (grid y: row blocks), KW waves
// over K, U 16-float k-steps per batch of loads with the next batch in flight.
// K % 4 == 0.
template <int MB, int KW, int U>
__global__ __launch_bounds__(KW * 64) void linear_f32_rows_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ y, int rows, int N, int K, int64_t x_rs, int64_t y_rs) {
  __shared__ float partial[KW][MB][64][4];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c = lane & 15;
  const int g = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int m0 = blockIdx.y * (16 * MB);
  const int M = min(16 * MB, rows - m0);
  x += m0 * x_rs;
  y += m0 * y_rs;
  const int steps = (K + 15) / 16;
  const int per_wave = (steps + KW - 1) / KW;
  const int s_begin = wave * per_wave;
  const int s_end = min(s_begin + per_wave, steps);
  const int w_rows = min(16, N - n0);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(w + static_cast<int64_t>(n0) * K,
                                              static_cast<int64_t>(w_rows) * K * 4);
  const __amdgpu_buffer_rsrc_t rx =
      make_rsrc(x, ((static_cast<int64_t>(M) - 1) * x_rs + K) * 4);
  const int w_off = c * K * 4 + g * 16;  // rows past N / M read zero
  int x_off[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) x_off[i] = static_cast<int>((i * 16 + c) * x_rs * 4) + g * 16;

  f32x4_t acc[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32x4_t wa[U], xa[U][MB], wb[U], xb[U][MB];
  const f32x4_t zero = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int s0, f32x4_t (&wr)[U], f32x4_t (&xr)[U][MB]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u;
      const bool ok = s < s_end && s * 16 + g * 4 < K;
      wr[u] = ok ? load4(rw, w_off + s * 64) : zero;
#pragma unroll
      for (int i = 0; i < MB; ++i) xr[u][i] = ok ? load4(rx, x_off[i] + s * 64) : zero;
    }
  };
  auto multiply = [&](const f32x4_t (&wr)[U], const f32x4_t (&xr)[U][MB]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < MB; ++i) acc[i] = mfma4(xr[u][i][e], wr[u][e], acc[i]);
  };
  int s0 = s_begin;
  fetch(s0, wa, xa);
  while (s0 < s_end) {
    fetch(s0 + U, wb, xb);
    multiply(wa, xa);
    s0 += U;
    if (s0 >= s_end) break;
    fetch(s0 + U, wa, xa);
    multiply(wb, xb);
    s0 += U;
  }
  // Lane (feature c, rows 4g .. 4g + 3 of block i).
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) partial[wave][i][lane][r] = acc[i][r];
  __syncthreads();
  for (int idx = tid; idx < MB * 256; idx += KW * 64) {
    const int i = idx / 256, l = (idx / 4) % 64, r = idx % 4;
    float sum = 0.0f;
#pragma unroll
    for (int v = 0; v < KW; ++v) sum += partial[v][i][l][r];
    const int n = n0 + (l & 15);
    const int m = i * 16 + 4 * (l >> 4) + r;
    if (n < N && m < M) {
      if (bias != nullptr) sum += bias[n];
      y[m * y_rs + n] = sum;
    }
  }
}

// M <= 4 * RG rows (RG <= 4), 4 * FG features per workgroup: the 16-feature
// form above leaves most CUs without a workgroup at a hidden-sized N, and one
// MFMA of 16 x 16 spends as long on 4 features as on 16.  v_mfma_f32_4x4x1_f32
// multiplies 16 independent 4 x 4 blocks at the same rate: block b takes the
// k's of the 16-byte chunk b, so lane (block l / 4, row l % 4) reads chunk
// l / 4 of W row (X row) l % 4, and the blocks' sums are added at the end.
template <int FG, int RG, int KW, int U>
__global__ __launch_bounds__(KW * 64) void linear_f32_few_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ y, int M, int N, int K, int64_t x_rs, int64_t y_rs) {
  __shared__ float partial[KW][FG * RG * 16];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int r4 = lane & 3;
  const int chunk = lane >> 2;
  const int n0 = blockIdx.x * (4 * FG);
  const int steps = (K + 63) / 64;
  const int per_wave = (steps + KW - 1) / KW;
  const int s_begin = wave * per_wave;
  const int s_end = min(s_begin + per_wave, steps);
  const int w_rows = min(4 * FG, N - n0);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(w + static_cast<int64_t>(n0) * K,
                                              static_cast<int64_t>(w_rows) * K * 4);
  const __amdgpu_buffer_rsrc_t rx =
      make_rsrc(x, ((static_cast<int64_t>(M) - 1) * x_rs + K) * 4);
  int w_off[FG], x_off[RG];  // rows past N / M read zero
#pragma unroll
  for (int f = 0; f < FG; ++f) w_off[f] = (4 * f + r4) * K * 4 + chunk * 16;
#pragma unroll
  for (int i = 0; i < RG; ++i) x_off[i] = static_cast<int>((4 * i + r4) * x_rs * 4) + chunk * 16;

  f32x4_t acc[FG][RG];
#pragma unroll
  for (int f = 0; f < FG; ++f)
#pragma unroll
    for (int i = 0; i < RG; ++i) acc[f][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32x4_t wa[U][FG], xa[U][RG], wb[U][FG], xb[U][RG];
  const f32x4_t zero = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int s0, f32x4_t (&wr)[U][FG], f32x4_t (&xr)[U][RG]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u;
      const bool ok = s < s_end && s * 64 + chunk * 4 < K;
#pragma unroll
      for (int f = 0; f < FG; ++f) wr[u][f] = ok ? load4(rw, w_off[f] + s * 256) : zero;
#pragma unroll
      for (int i = 0; i < RG; ++i) xr[u][i] = ok ? load4(rx, x_off[i] + s * 256) : zero;
    }
  };
  auto multiply = [&](const f32x4_t (&wr)[U][FG], const f32x4_t (&xr)[U][RG]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int f = 0; f < FG; ++f)
#pragma unroll
          for (int i = 0; i < RG; ++i)
            acc[f][i] = __builtin_amdgcn_mfma_f32_4x4x1f32(xr[u][i][e], wr[u][f][e], acc[f][i], 0, 0, 0);
  };
  int s0 = s_begin;
  fetch(s0, wa, xa);
  while (s0 < s_end) {
    fetch(s0 + U, wb, xb);
    multiply(wa, xa);
    s0 += U;
    if (s0 >= s_end) break;
    fetch(s0 + U, wa, xa);
    multiply(wb, xb);
    s0 += U;
  }
  // Lane (block l / 4, feature l % 4) holds rows 0..3: add the 16 blocks.
#pragma unroll
  for (int f = 0; f < FG; ++f)
#pragma unroll
    for (int i = 0; i < RG; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[f][i][r];
        v += __shfl_xor(v, 4, 64);
        v += __shfl_xor(v, 8, 64);
        v = slc::sum_xor32(slc::sum_xor16(v));
        if (lane < 4) partial[wave][((f * RG + i) * 4 + r) * 4 + lane] = v;
      }
  __syncthreads();
  for (int idx = tid; idx < FG * RG * 16; idx += KW * 64) {
    float sum = 0.0f;
#pragma unroll
    for (int v = 0; v < KW; ++v) sum += partial[v][idx];
    const int n = n0 + (idx / (RG * 16)) * 4 + (idx & 3);
    const int m = ((idx / 16) % RG) * 4 + ((idx >> 2) & 3);
    if (n < N && m < M) {
      if (bias != nullptr) sum += bias[n];
      y[m * y_rs + n] = sum;
    }
  }
}

template <int BM, int BN, int CWM, int CWN, int PW, int S>
int launch_ring(const float* x, const float* w, const float* bias, float* y, int M, int N, int K,
                int64_t x_rs, int64_t y_rs, hipStream_t stream) {
  const int n_tiles = (N + BN - 1) / BN, m_tiles = (M + BM - 1) / BM;
  const int wide = N % 4 == 0 && y_rs % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
  hipLaunchKernelGGL((linear_f32_ring_kernel<BM, BN, CWM, CWN, PW, S>),
                     dim3(static_cast<unsigned>(n_tiles) * m_tiles), dim3((CWM * CWN + PW) * 64), 0,
                     stream, x, w, bias, y, M, N, K, x_rs, y_rs, n_tiles, wide);
  return slc_host::check_launch("slc_hip_linear(f32 ring)");
}

template <int MB, int KW, int U>
int launch_rows(const float* x, const float* w, const float* bias, float* y, int M, int N, int K,
                int64_t x_rs, int64_t y_rs, hipStream_t stream) {
  hipLaunchKernelGGL((linear_f32_rows_kernel<MB, KW, U>),
                     dim3((N + 15) / 16, (M + 16 * MB - 1) / (16 * MB)), dim3(KW * 64), 0, stream, x,
                     w, bias, y, M, N, K, x_rs, y_rs);
  return slc_host::check_launch("slc_hip_linear(f32 rows)");
}

template <int FG, int KW, int U>
int launch_few(const float* x, const float* w, const float* bias, float* y, int M, int N, int K,
               int64_t x_rs, int64_t y_rs, hipStream_t stream) {
  const dim3 grid((N + 4 * FG - 1) / (4 * FG));
#define SLC_FEW(RG)                                                                             \
  hipLaunchKernelGGL((linear_f32_few_kernel<FG, RG, KW, U>), grid, dim3(KW * 64), 0, stream, x, w, \
                     bias, y, M, N, K, x_rs, y_rs)
  if (M <= 4) {
    SLC_FEW(1);
  } else if (M <= 8) {
    SLC_FEW(2);
  } else {
    SLC_FEW(4);
  }
#undef SLC_FEW
  return slc_host::check_launch("slc_hip_linear(f32 few rows)");
}

}  // namespace

namespace slc_host {

int linear_f32(const float* x, const float* w, const float* bias, float* y, int M, int N, int K,
               int64_t x_rs, int64_t y_rs, hipStream_t s) {
  const uint64_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w);
  if ((bits & 15) != 0 || K % 4 != 0 || x_rs % 4 != 0 || x_rs < K || 128 * x_rs * 4 >= (int64_t{1} << 31) ||
      int64_t{128} * K * 4 >= (int64_t{1} << 31))
    return SLC_ERR_UNSUPPORTED;
  const int64_t cus = device_cu_count();
  const int64_t blocks16 = ceil_div(N, 16) * ceil_div(M, 16);
  // Short K leaves these kernels little but their start and their epilogue: the
  // generic kernel takes K below 64 (K32: 16 rows N4864 10.5 us here, 2.8 there;
  // 4096 rows N16384 K4 588 | 137) except large grids of whole k-tiles (4096 rows
  // N4864 K32 0.4 of its time), and up to 92 many rows past the ring's k-tiles.
  if (K < 64 && (K % kBK != 0 || M <= 16 || blocks16 <= 8 * cus)) return SLC_ERR_UNSUPPORTED;
  if (K < 96 && K % kBK != 0 && M > 16 && blocks16 > 2 * cus) return SLC_ERR_UNSUPPORTED;
  if (M <= 16) {
    // One round of workgroups of 4, 8 or 20 features each, while that covers N
    // and K is long enough for the sums over the waves at the end, which grow
    // with the features and rows (16 rows N4864: K256 10.8 us, the generic kernel
    // 8.4, 16-feature workgroups 4.2; K384 11.3 | 11.5 | 5.5, with three times the
    // error; 16 rows N1500 K128 6.6 | 4.9 | 3.3; 8 rows N4864 K128 6.5 | 5.1 | 3.3).
    const int rows = M <= 4 ? 0 : (M <= 8 ? 1 : 2);
    constexpr int kLeast[3][3] = {{64, 96, 128}, {96, 128, 256}, {128, 256, 384}};
    if (N <= 4 * cus && K >= kLeast[0][rows])
      return launch_few<1, 16, 2>(x, w, bias, y, M, N, K, x_rs, y_rs, s);
    if (N > 4 * cus && N <= 8 * cus && K >= kLeast[1][rows])
      return launch_few<2, 16, 1>(x, w, bias, y, M, N, K, x_rs, y_rs, s);
    if (N > 8 * cus && N <= 20 * cus && K >= kLeast[2][rows])
      return launch_few<5, 8, 1>(x, w, bias, y, M, N, K, x_rs, y_rs, s);
    return launch_rows<1, 4, 4>(x, w, bias, y, M, N, K, x_rs, y_rs, s);
  }
  if (K % kBK != 0 || blocks16 <= 2 * cus) {
    if (M > 65535 * 16) return SLC_ERR_UNSUPPORTED;
    if (blocks16 <= cus) return launch_rows<1, 16, 4>(x, w, bias, y, M, N, K, x_rs, y_rs, s);
    return launch_rows<2, 16, 2>(x, w, bias, y, M, N, K, x_rs, y_rs, s);
  }
  // The matrix cores bound the kernel, so the tile is the one whose grid
  // leaves the fewest of them idle: rounds of the grid over the CUs times what
  // a CU takes for one tile (microseconds at K = 896 with the CUs full: 3.4 ns
  // per output of the two large tiles, 4.1 and 5.4 of the smaller ones, which
  // read more per product).
  auto cost = [&](int64_t bm, int64_t bn, double us) {
    return static_cast<double>(ceil_div(ceil_div(M, bm) * ceil_div(N, bn), cus)) * us;
  };
  const double c128 = cost(128, 128, 56), c64x128 = cost(64, 128, 28), c64 = cost(64, 64, 17),
               c32 = cost(32, 32, 5.5);
  if (c32 < c64 && c32 < c64x128 && c32 < c128)
    return launch_ring<32, 32, 2, 2, 1, 6>(x, w, bias, y, M, N, K, x_rs, y_rs, s);
  if (c64 < c64x128 && c64 < c128)
    return launch_ring<64, 64, 2, 2, 1, 3>(x, w, bias, y, M, N, K, x_rs, y_rs, s);
  if (c64x128 <= c128) return launch_ring<64, 128, 2, 2, 1, 2>(x, w, bias, y, M, N, K, x_rs, y_rs, s);
  return launch_ring<128, 128, 2, 4, 2, 2>(x, w, bias, y, M, N, K, x_rs, y_rs, s);
}

}  // namespace slc_host
