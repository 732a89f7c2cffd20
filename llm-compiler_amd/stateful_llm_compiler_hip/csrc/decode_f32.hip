// fp32 decode attention on the fp32 matrix cores (head_dim 64 or 128, up to 16
// query heads per KV head).
//
// Semantics: src/stateful_llm_compiler/execution.py:281-327, fp32 throughout.
// With fp32 tensors the reference's rounding of the probabilities changes
// nothing, so one single-pass kernel serves both softmax orders.
//
// What bounds it: HBM.  Every K and V byte is read once for all the query heads
// of its KV head (one wave per query head and token before: each row read seven
// times, one token per wave and round trip).
//  * S^T[token, head] = K . Q^T on v_mfma_f32_16x16x4_f32: lane (token c, group
//    g) loads the 16-byte chunks 4 kk + g of its row straight into the A
//    operand and the MFMAs take the chunks' elements in turn (Q holds the same
//    dims).
//  * O[head, dim] += P . V: accumulator element r of lane (head c, group g) is
//    token 4g + r, which is k-slot g of the A operand, so the probabilities
//    never move; V rows are loaded 16 bytes per lane (row 4g + r, dims 4c ..
//    4c + 3) and the MFMAs' columns are dims 4c + e.
//  * A score's products are summed in chains of two MFMAs added in pairs: with
//    two chains the result was up to 1.44 times as far from float64 as one wave
//    per head with its sums across lanes (L64 D128 2.03e-7 against 1.40e-7, now
//    1.35e-7; L300 D64 2.1e-7, 2.0e-7, now 1.7e-7; L32768 3.4e-7, 16e-7, now
//    3.1e-7).  It costs 1 to 5 % of the time.
//  * Sequences are split over about two workgroups per CU; partials merge in
//    the last workgroup of each (batch, KV head), as in decode_kernel.hpp.
// Measured against the wave-per-head kernel (graphs of back-to-back calls, every
// sequence at its full length): B27 L9241 2237 -> 57 us (4.5 TB/s of K and V), B1
// L32768 7371 -> 28, B16 L30000 D128 12262 -> 204 (4.8 TB/s), B6 L247 35 -> 8.4.
#include "common.hpp"
#include "decode_kernel.hpp"

namespace {

__device__ __forceinline__ f32x4_t mfma4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kTokens = 16;               // tokens per wave and step
constexpr int kAheadF32 = 2;              // steps in flight per wave
constexpr int kSweepF32 = kWaves * kTokens;

// MK: mask element type (0 = none, else an slc_dtype tag + 1).
template <int D, int MK>
__global__ __launch_bounds__(kThreads) void decode_attention_f32_kernel(
    const float* __restrict__ query, const float* __restrict__ key_buffer,
    const float* __restrict__ value_buffer, const void* __restrict__ lengths, int lengths_dtype,
    const void* __restrict__ mask, float* __restrict__ output, float* __restrict__ part_o,
    float* __restrict__ part_ml, int q_heads, int kv_heads, int groups, int64_t capacity,
    int64_t mask_len, int64_t q_sb, int64_t q_sh, int64_t kv_sb, int64_t kv_ss, int64_t kv_sh,
    int64_t m_sb, int64_t m_ss, int64_t o_sb, int64_t o_sh, float scale, int chunk_tokens,
    int nchunks, int* __restrict__ counters) {
  constexpr int KK = D / 16;  // 16-byte chunks of K per lane
  constexpr int VH = D / 64;  // 64-dim halves of a V row
  __shared__ float sm_m[kWaves][kMaxGroups], sm_l[kWaves][kMaxGroups];
  __shared__ float sm_o[kWaves][kMaxGroups][D];
  const int chunk = blockIdx.x, kvh = blockIdx.y;
  const int64_t b = blockIdx.z;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c = lane & 15, g = lane >> 4;

  f32x4_t qv[KK];
  {
    const float* qp = query + b * q_sb + (kvh * groups + min(c, groups - 1)) * q_sh;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qv[kk] = *reinterpret_cast<const f32x4_t*>(qp + 16 * kk + 4 * g);
  }
  int64_t end64 = slc::load_length(lengths, b, lengths_dtype);
  end64 = end64 < 0 ? 0 : end64;
  end64 = end64 < mask_len ? end64 : mask_len;
  end64 = end64 < capacity ? end64 : capacity;
  // One sequence's length: uniform, and below 2^30 as a chunk's end is (the
  // host checks).
  const int seq_end = __builtin_amdgcn_readfirstlane(static_cast<int>(end64));
  const int first = chunk * chunk_tokens;
  const int end = min(seq_end, first + chunk_tokens);

  const float* kbase = key_buffer + b * kv_sb + kvh * kv_sh;
  const float* vbase = value_buffer + b * kv_sb + kvh * kv_sh;
  const int row_bytes = static_cast<int>(kv_ss * 4);
  const int k_off = c * row_bytes + 16 * g;
  const int v_off = 4 * g * row_bytes + 16 * c;

  struct Step {
    f32x4_t k[KK], v[4][VH];
    float mk[MK == 0 ? 1 : 4];
  };
  auto load = [&](int t0, Step& s) {
    const int rows = min(kTokens, end - t0);  // rows past the end read zero
    const int bytes = rows > 0 ? (rows - 1) * row_bytes + D * 4 : 0;
    const int64_t at = rows > 0 ? static_cast<int64_t>(t0) * kv_ss : 0;
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(kbase + at, bytes), rv = make_rsrc(vbase + at, bytes);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      s.k[kk] = __builtin_bit_cast(f32x4_t, buffer_load16(rk, k_off + kk * 64));
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int h = 0; h < VH; ++h)
        s.v[r][h] = __builtin_bit_cast(f32x4_t, buffer_load16(rv, v_off + r * row_bytes + h * 256));
    if constexpr (MK != 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = t0 + 4 * g + r;
        s.mk[r] = t < end ? slc::load_as_f32(mask, b * m_sb + t * m_ss, MK - 1) : 0.0f;
      }
    }
  };

  float m_run = -INFINITY, l_part = 0.0f;
  f32x4_t acc[VH][4];
#pragma unroll
  for (int h = 0; h < VH; ++h)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[h][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](int t0, const Step& s) {
    // Chains of two MFMAs, added in pairs: a long chain rounds its partial sums
    // one after the other.
    f32x4_t st = f32x4_t{0.f, 0.f, 0.f, 0.f}, part[2 * KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      part[2 * kk] = mfma4(s.k[kk][1], qv[kk][1], mfma4(s.k[kk][0], qv[kk][0], st));
      part[2 * kk + 1] = mfma4(s.k[kk][3], qv[kk][3], mfma4(s.k[kk][2], qv[kk][2], st));
    }
#pragma unroll
    for (int n = KK; n > 0; n /= 2)
#pragma unroll
      for (int i = 0; i < n; ++i) part[i] = part[2 * i] + part[2 * i + 1];
    st = part[0];
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = st[r] * scale;
      if constexpr (MK != 0) v += s.mk[r];
      st[r] = t0 + 4 * g + r < end ? v : -INFINITY;
      mx = fmaxf(mx, st[r]);
    }
    mx *= kLog2e;
    if (__any(mx > m_run + kRescaleThreshold)) {
      mx = slc::max_xor32(slc::max_xor16(mx));
      const float m_new = fmaxf(m_run, mx);
      const float alpha = weight_exp2<float>(m_run - (m_new == -INFINITY ? 0.0f : m_new));
      l_part *= alpha;
      m_run = m_new;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float a = __shfl(alpha, 4 * g + r, 64);  // accumulator rows are heads
#pragma unroll
        for (int h = 0; h < VH; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[h][e][r] *= a;
      }
    }
    const float m_use = m_run == -INFINITY ? 0.0f : m_run;
    // As weight_exp2; only waves with a result below 2^-126 (a masked token's
    // counts) pay for the scaling.
    float x[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = fmaf(st[r], kLog2e, -m_use);
    if (__any(fminf(fminf(x[0], x[1]), fminf(x[2], x[3])) < -126.0f)) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int r = 0; r < 4; ++r) st[r] = exp2f(x[r]);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) st[r] = fast_exp2(x[r]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) l_part += st[r];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int h = 0; h < VH; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[h][e] = mfma4(st[r], s.v[r][h][e], acc[h][e]);
  };

  Step steps[kAheadF32];
  const int start = first + wave * kTokens;
#pragma unroll
  for (int i = 0; i < kAheadF32; ++i) {
    load(start + i * kSweepF32, steps[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int t0 = start; t0 < end; t0 += kAheadF32 * kSweepF32) {
#pragma unroll
    for (int i = 0; i < kAheadF32; ++i) {
      compute(t0 + i * kSweepF32, steps[i]);
      load(t0 + (i + kAheadF32) * kSweepF32, steps[i]);
    }
  }

  // Combine the waves: sums over the lane groups, then weights per wave.
  const float l_run = slc::sum_xor32(slc::sum_xor16(l_part));
  if (g == 0) {
    sm_m[wave][c] = m_run;
    sm_l[wave][c] = l_run;
  }
#pragma unroll
  for (int h = 0; h < VH; ++h)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int r = 0; r < 4; ++r) sm_o[wave][4 * g + r][64 * h + 4 * c + e] = acc[h][e][r];
  __syncthreads();
  for (int idx = tid; idx < groups * D; idx += kThreads) {
    const int head = idx / D, d = idx % D;
    const int qh = kvh * groups + head;
    float mmax = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) mmax = fmaxf(mmax, sm_m[w][head]);
    const float mu = mmax == -INFINITY ? 0.0f : mmax;
    float lsum = 0.0f, osum = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float f = weight_exp2<float>(sm_m[w][head] - mu);
      lsum += f * sm_l[w][head];
      osum += f * sm_o[w][head][d];
    }
    if (nchunks == 1) {
      output[b * o_sb + qh * o_sh + d] = osum / lsum;
    } else {
      const int64_t p = (b * q_heads + qh) * nchunks + chunk;
      publish(part_o + p * D + d, osum);
      if (d == 0) {
        publish(part_ml + 2 * p, mmax);
        publish(part_ml + 2 * p + 1, lsum);
      }
    }
  }
  if (nchunks == 1) return;
  merge_if_last<float, D>(part_o, part_ml, output, counters, nullptr, b, kvh, q_heads, kv_heads,
                          groups, o_sb, o_sh, nchunks, LenAdvance{});
}

}  // namespace

namespace slc_host {

bool decode_f32_eligible(int64_t head_dim, int64_t groups) {
  return (head_dim == 64 || head_dim == 128) && groups <= kMaxGroups;
}

int64_t decode_f32_chunks(int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t head_dim,
                          int64_t mask_len) {
  // Two workgroups for each of MI355X's 256 CUs, at least two sweeps of tokens
  // each, and partials of at most 8 MiB (what the no-allocation entry point
  // holds).  The count is a constant, as in choose_chunk: it sizes the caller's
  // workspace, which is asked for without a device.
  int64_t n = std::min<int64_t>(512 / std::max<int64_t>(1, batch * kv_heads),
                                ceil_div(mask_len, 2 * kSweepF32));
  n = std::min<int64_t>(n, 64);
  if (n > 1 && partial_bytes(batch, q_heads, head_dim, n) > (int64_t{8} << 20)) n = 1;
  return std::max<int64_t>(n, 1);
}

int decode_attention_f32(const float* query, const float* kb, const float* vb, const void* lengths,
                         int lengths_dtype, const void* mask, int mask_dtype, float* output,
                         void* workspace, int64_t workspace_bytes, int* counters,
                         int64_t num_counters, int64_t batch, int64_t q_heads, int64_t kv_heads,
                         int64_t head_dim, int64_t capacity, int64_t mask_len, const int64_t* st,
                         float scale, hipStream_t stream) {
  const uint64_t bits = reinterpret_cast<uintptr_t>(query) | reinterpret_cast<uintptr_t>(kb) |
                        reinterpret_cast<uintptr_t>(vb);
  const int64_t strides = st[0] | st[1] | st[2] | st[3] | st[4];
  const int64_t groups = q_heads / kv_heads;
  if (!decode_f32_eligible(head_dim, groups) || mask_len < 1 || (bits & 15) != 0 ||
      (strides & 3) != 0 || st[3] < head_dim || st[3] >= (int64_t{1} << 24) ||
      mask_len >= (int64_t{1} << 30))
    return SLC_ERR_UNSUPPORTED;
  int64_t n = decode_f32_chunks(batch, q_heads, kv_heads, head_dim, mask_len);
  // Without room for the partials one workgroup takes a whole sequence.
  if (workspace == nullptr || workspace_bytes < partial_bytes(batch, q_heads, head_dim, n) ||
      counters == nullptr || num_counters < counter_count(batch, kv_heads))
    n = 1;
  const int64_t chunk = ceil_div(ceil_div(mask_len, n), kSweepF32) * kSweepF32;
  n = ceil_div(mask_len, chunk);
  float* part_o = static_cast<float*>(workspace);
  float* part_ml = n > 1 ? part_o + batch * q_heads * n * head_dim : nullptr;
  const dim3 grid(static_cast<unsigned>(n), static_cast<unsigned>(kv_heads),
                  static_cast<unsigned>(batch));
#define SLC_F32_K(D, MK)                                                                         \
  hipLaunchKernelGGL((decode_attention_f32_kernel<D, MK>), grid, dim3(kThreads), 0, stream, query, \
                     kb, vb, lengths, lengths_dtype, mask, output, part_o, part_ml,              \
                     static_cast<int>(q_heads), static_cast<int>(kv_heads),                      \
                     static_cast<int>(groups), capacity, mask_len, st[0], st[1], st[2], st[3],   \
                     st[4], st[5], st[6], st[7], st[8], scale, static_cast<int>(chunk),          \
                     static_cast<int>(n), counters)
#define SLC_F32_D(D)                 \
  if (mask == nullptr) {             \
    SLC_F32_K(D, 0);                 \
  } else if (mask_dtype == SLC_F32) { \
    SLC_F32_K(D, SLC_F32 + 1);       \
  } else if (mask_dtype == SLC_F16) { \
    SLC_F32_K(D, SLC_F16 + 1);       \
  } else {                           \
    SLC_F32_K(D, SLC_BF16 + 1);      \
  }
  mark_kernel_begin(stream);
  for (int rep = timed_repeats(); rep > 0; --rep) {
    if (head_dim == 64) {
      SLC_F32_D(64)
    } else {
      SLC_F32_D(128)
    }
  }
  mark_kernel_end(stream);
#undef SLC_F32_D
#undef SLC_F32_K
  return check_launch("slc_hip_decode_attention(f32)");
}

}  // namespace slc_host
