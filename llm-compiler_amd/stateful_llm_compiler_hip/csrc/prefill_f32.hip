// fp32 prefill attention on the fp32 matrix cores (head_dim 64).
//
// Semantics: src/stateful_llm_compiler/execution.py:707-739 and
// backends/triton_prefill_attention.py:10-150, fp32 throughout:
//   out[b,h,q,:] = sum_k softmax_k(scale * q.k + mask[b,q,k]) v[b,k,h/g,:]
// With fp32 tensors the two softmax orders differ only in where the division
// by the row sum falls (the reference's rounding of the probabilities to the
// tensor type changes nothing), so one kernel serves both.
//
// What bounds it: the matrix cores.  v_mfma_f32_16x16x4_f32 does 64 FLOP per
// cycle and SIMD, so a wave's 128 MFMAs on a 64-key tile take 4096 cycles
// against about 1500 of VALU (softmax, and the sums that keep the error below
// one chain's) and 1024 of LDS reads for its workgroup: memory and LDS hide
// behind them with two workgroups per CU.
//  * A workgroup is 4 waves of 16 queries each of one query head; 64-key K and
//    V tiles (16 KB each) are double-buffered in LDS, filled by direct loads.
//  * S^T[key, query] = K . Q^T: lane (row c, group g) reads the 16-byte chunk
//    4 kk + g of key c (chunks XOR-swizzled by key, so the 16 keys of a read
//    fall on different banks) and the MFMAs take its elements in turn; Q holds
//    the same dims in registers.
//  * O^T[dim, query] += V^T . P^T: accumulator element r of lane (query c,
//    group g) is key 4g + r, which is exactly k-slot g of the r-th MFMA's B
//    operand, so the probabilities never move; V is read one float per lane
//    (dims 16 db + c of key 4g + r; the four groups' 64-byte segments are
//    swizzled onto different banks).
//  * Key tiles that the mask's classes rule out are not visited, tiles of the
//    causal pattern are masked from the indices, and only the rest read their
//    mask, element by element (any strides), under the score MFMAs.
//  * A score is eight chains of two MFMAs added in pairs, and a tile's sums over
//    its keys are added to the running ones once: a single chain of 64 products
//    and one over all keys were up to 1.44 times as far from float64 as one wave
//    per query with its sums across lanes (16 tokens 1.21e-7 against 0.84e-7,
//    now 0.81e-7; 200 tokens 2.3e-7 against 1.8e-7, now 1.4e-7; 1000 tokens
//    3.3e-7, 3.2e-7, now 1.6e-7).  It costs 8 to 11 % of the time.
// Measured against one wave per query: B8 T512 padded causal mask 2930 -> 58
// us, B6 T1000 causal 3670 -> 117 us (92 TFLOP/s of the causal products; a
// large fp32 library product reaches 153 on this card), B1 T64 29 -> 6.4.
#include <algorithm>

#include "common.hpp"

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kRescaleThreshold = 8.0f;
constexpr int kD = 64;
constexpr int kKeys = 64;
constexpr int kWaves = 4;
constexpr int kQueries = 16 * kWaves;
constexpr int kRow = kD * 4;             // bytes of one K or V row
constexpr int kTile = kKeys * kRow;      // 16 KB
constexpr int kMaxClassTiles = 1024;     // key tiles the class list covers

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
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t rsrc, unsigned char* lds,
                                          int voffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      rsrc, (__attribute__((address_space(3))) void*)lds, 16, voffset, 0, 0, 0);
}

struct Strides {
  int64_t q_sb, q_sh, q_st, k_sb, k_sh, k_st, v_sb, v_sh, v_st, m_sb, m_sq, m_sk, o_sb, o_sh, o_st;
};

template <bool MASK>
__global__ __launch_bounds__(kWaves * 64, 2) void prefill_attention_f32_kernel(
    const float* __restrict__ query, const float* __restrict__ key, const float* __restrict__ value,
    const void* __restrict__ mask, int mask_dtype, const unsigned char* __restrict__ tile_class,
    float* __restrict__ output, int tokens, int groups, int causal, Strides s, float scale) {
  __shared__ __attribute__((aligned(16))) unsigned char ring[2][2 * kTile];
  // The key tiles this block visits, in order; bit 15: the mask is read.
  __shared__ uint16_t live_tiles[MASK ? kMaxClassTiles : 1];
  __shared__ int live_count;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c = lane & 15;
  const int g = lane >> 4;
  // Grid (heads, batch, query blocks), last query blocks first: under a causal
  // pattern those are the heaviest.
  const int qblk = static_cast<int>(gridDim.z) - 1 - static_cast<int>(blockIdx.z);
  const int h = blockIdx.x;
  const int kvh = h / groups;
  const int64_t b = blockIdx.y;
  const int q0 = qblk * kQueries;
  const int key_end = causal ? min(q0 + kQueries, tokens) : tokens;
  const int all_tiles = (key_end + kKeys - 1) / kKeys;
  const bool classed = MASK && tile_class != nullptr;
  if constexpr (MASK) {
    if (classed) {
      if (wave == 0) {
        const int64_t key_tiles = (tokens + kKeys - 1) / kKeys;
        const unsigned char* row = tile_class + (b * key_tiles + qblk) * key_tiles;
        int count = 0;
        for (int base = 0; base < all_tiles; base += 64) {
          const int t = base + lane;
          const int cls = t < all_tiles ? row[t] : 0;
          const uint64_t live = __ballot(cls != 0);
          const int before = __builtin_amdgcn_mbcnt_hi(
              static_cast<uint32_t>(live >> 32),
              __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(live), 0));
          if (cls != 0) live_tiles[count + before] = static_cast<uint16_t>(t | (cls == 2 ? 0x8000 : 0));
          count += __popcll(live);
        }
        if (lane == 0) live_count = count;
      }
      __syncthreads();
    }
  }
  const int ntiles = classed ? __builtin_amdgcn_readfirstlane(live_count) : all_tiles;
  auto entry = [&](int i) {
    return classed ? __builtin_amdgcn_readfirstlane(static_cast<int>(live_tiles[i]))
                   : i | (MASK ? 0x8000 : 0);
  };

  const float* kbase = key + b * s.k_sb + kvh * s.k_sh;
  const float* vbase = value + b * s.v_sb + kvh * s.v_sh;
  // This wave's quarter of a tile: load n covers rows 4 * (4 * wave + n) .. + 3,
  // lane L row L / 16, chunk position L % 16.
  int koff[4], voff[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int row = 4 * (4 * wave + n) + lane / 16;
    const int pos = lane % 16;
    koff[n] = static_cast<int>(row * s.k_st * 4) + ((pos ^ (row & 15)) << 4);
    voff[n] = static_cast<int>(row * s.v_st * 4) + ((pos ^ (((row >> 2) & 3) << 2)) << 4);
  }
  auto issue = [&](int i) {
    if (i >= ntiles) return;
    unsigned char* dst = ring[i & 1];
    const int k0 = ((classed ? entry(i) & 0x7fff : i)) * kKeys;
    const int64_t rows = min(kKeys, tokens - k0);
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(kbase + k0 * s.k_st, ((rows - 1) * s.k_st + kD) * 4);
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vbase + k0 * s.v_st, ((rows - 1) * s.v_st + kD) * 4);
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      lds_dma16(rk, dst + (4 * wave + n) * 1024, koff[n]);
      lds_dma16(rv, dst + kTile + (4 * wave + n) * 1024, voff[n]);
    }
  };

  const int my_query = q0 + 16 * wave + c;
  const int q_row = min(my_query, tokens - 1);
  f32x4_t qv[4];
  {
    const float* qp = query + b * s.q_sb + h * s.q_sh + q_row * s.q_st;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) qv[kk] = *reinterpret_cast<const f32x4_t*>(qp + 16 * kk + 4 * g);
  }
  int k_read[4], v_read[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) k_read[kk] = c * kRow + (((4 * kk + g) ^ c) << 4);
#pragma unroll
  for (int db = 0; db < 4; ++db) v_read[db] = kTile + 4 * g * kRow + (db ^ g) * 64 + c * 4;
  const int64_t mask_row = MASK ? b * s.m_sb + static_cast<int64_t>(q_row) * s.m_sq : 0;

  float m_run = -INFINITY, l_part = 0.0f;
  f32x4_t acc[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  issue(0);
  for (int i = 0; i < ntiles; ++i) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's loads of tile i
    __syncthreads();  // every wave's; and every wave is done with the other buffer
    issue(i + 1);
    const int e = entry(i);
    const int k0 = (e & 0x7fff) * kKeys;
    const bool read_mask = MASK && (e & 0x8000) != 0;
    const bool causal_tile = causal || (MASK && !read_mask);
    const unsigned char* tile = ring[i & 1];

    float mv[16];
    if constexpr (MASK) {
      if (read_mask) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int k = min(k0 + 16 * (j >> 2) + 4 * g + (j & 3), tokens - 1);
          mv[j] = slc::load_as_f32(mask, mask_row + k * s.m_sk, mask_dtype);
        }
      }
    }
    // Eight chains of two MFMAs per score, added in pairs: one chain of sixteen
    // rounds 64 partial sums one after the other.
    f32x4_t st[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      f32x4_t part[8];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const f32x4_t ka = *reinterpret_cast<const f32x4_t*>(tile + k_read[kk] + 16 * kb * kRow);
        const f32x4_t z = f32x4_t{0.f, 0.f, 0.f, 0.f};
        part[2 * kk] = mfma4(ka[1], qv[kk][1], mfma4(ka[0], qv[kk][0], z));
        part[2 * kk + 1] = mfma4(ka[3], qv[kk][3], mfma4(ka[2], qv[kk][2], z));
      }
      st[kb] = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) st[kb][r] *= scale;
    if constexpr (MASK) {
      if (read_mask) {
#pragma unroll
        for (int j = 0; j < 16; ++j) st[j >> 2][j & 3] += mv[j];
      }
    }
    const bool full = k0 + kKeys <= tokens && (!causal_tile || k0 + kKeys <= q0 + 16 * wave);
    if (!full) {
      asm volatile("" ::: "memory");  // keep this a branch
      int last = tokens - 1 - k0 - 4 * g;
      if (causal_tile) last = min(last, my_query - k0 - 4 * g);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) st[kb][r] = 16 * kb + r <= last ? st[kb][r] : -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, st[kb][r]);
    mx *= kLog2e;
    if (__any(mx > m_run + kRescaleThreshold)) {
      mx = slc::max_xor32(slc::max_xor16(mx));
      const float m_new = fmaxf(m_run, mx);
      const float alpha = exp2f(m_run - (m_new == -INFINITY ? 0.0f : m_new));
      l_part *= alpha;
#pragma unroll
      for (int db = 0; db < 4; ++db) acc[db] = acc[db] * alpha;
      m_run = m_new;
    }
    const float m_use = m_run == -INFINITY ? 0.0f : m_run;
    // Probabilities below 2^-126 stay subnormal numbers (exp2f), which only
    // tiles that have one pay for; masked scores count.
    float mn = st[0][0];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) mn = fminf(mn, st[kb][r]);
    if (__any(fmaf(mn, kLog2e, -m_use) < -126.0f)) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) st[kb][r] = exp2f(fmaf(st[kb][r], kLog2e, -m_use));
    } else {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) st[kb][r] = __builtin_amdgcn_exp2f(fmaf(st[kb][r], kLog2e, -m_use));
    }
    // The tile's own sums first, then one addition each to the running ones.
    float l_tile = 0.0f;
    f32x4_t pv[4];
#pragma unroll
    for (int db = 0; db < 4; ++db) pv[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) l_tile += st[kb][r];
    l_part += l_tile;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int db = 0; db < 4; ++db) {
          const float v = *reinterpret_cast<const float*>(tile + v_read[db] + (16 * kb + r) * kRow);
          pv[db] = mfma4(v, st[kb][r], pv[db]);
        }
#pragma unroll
    for (int db = 0; db < 4; ++db) acc[db] = acc[db] + pv[db];
  }

  // The row sum over the 4 lane groups; an empty row is 0 * inf = NaN, as the
  // reference's softmax over an all -inf row.
  const float inv = 1.0f / slc::sum_xor32(slc::sum_xor16(l_part));
  if (my_query < tokens) {
    float* op = output + b * s.o_sb + h * s.o_sh + static_cast<int64_t>(my_query) * s.o_st;
#pragma unroll
    for (int db = 0; db < 4; ++db)
      *reinterpret_cast<f32x4_t*>(op + 16 * db + 4 * g) = acc[db] * inv;
  }
}

}  // namespace

namespace slc_host {

int prefill_attention_f32(const float* query, const float* key, const float* value, const void* mask,
                          int mask_dtype, const unsigned char* tile_class, float* output,
                          int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t tokens,
                          int64_t head_dim, int causal, const int64_t* st, float scale,
                          hipStream_t stream) {
  const uint64_t bits = reinterpret_cast<uintptr_t>(query) | reinterpret_cast<uintptr_t>(key) |
                        reinterpret_cast<uintptr_t>(value) | reinterpret_cast<uintptr_t>(output);
  int64_t strides = st[12] | st[13] | st[14];
  for (int i = 0; i < 9; ++i) strides |= st[i];
  const int64_t blocks = ceil_div(tokens, kQueries);
  const bool ok = head_dim == kD && (bits & 15) == 0 && (strides & 3) == 0 && st[5] >= kD &&
                  st[8] >= kD && kKeys * std::max(st[5], st[8]) * 4 < (int64_t{1} << 31) &&
                  blocks <= 0x7fff;  // a tile index and its mask flag share 16 bits
  if (!ok) return SLC_ERR_UNSUPPORTED;
  const Strides s{st[0], st[1], st[2],  st[3],  st[4],  st[5],  st[6], st[7],
                  st[8], st[9], st[10], st[11], st[12], st[13], st[14]};
  // The tile list holds up to kMaxClassTiles key tiles; longer masks are read
  // in full.
  const unsigned char* classes = blocks <= kMaxClassTiles ? tile_class : nullptr;
  const dim3 grid(static_cast<unsigned>(q_heads), static_cast<unsigned>(batch),
                  static_cast<unsigned>(blocks));
  const int groups = static_cast<int>(q_heads / kv_heads);
  if (mask != nullptr)
    hipLaunchKernelGGL(prefill_attention_f32_kernel<true>, grid, dim3(kWaves * 64), 0, stream, query,
                       key, value, mask, mask_dtype, classes, output, static_cast<int>(tokens),
                       groups, causal, s, scale);
  else
    hipLaunchKernelGGL(prefill_attention_f32_kernel<false>, grid, dim3(kWaves * 64), 0, stream, query,
                       key, value, mask, mask_dtype, classes, output, static_cast<int>(tokens),
                       groups, causal, s, scale);
  return check_launch("slc_hip_prefill_attention(f32)");
}

}  // namespace slc_host
