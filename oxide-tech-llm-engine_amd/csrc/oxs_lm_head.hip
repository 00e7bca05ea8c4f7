// oxs_lm_head.hip — the LM head that feeds the sampler, in the reference CUDA
// backend's GGUF formats (Q8_0 weights x q8_1 activations), on gfx950.
//
// The reference's batched decode quantizes the final hidden states to q8_1
// and projects them with launch_cuda_mmvq_q8_0
// (oxide-backend-cuda/src/lib.rs:4013-4035). Here:
// - quantize_q8_1_kernel: one 32-lane group per q8_1 block, amax and sum by
//   the same xor butterfly, so the stored sum is the reference's bit for bit;
// - pack_q8_0_kernel: a one-time repack of the GGUF rows into tiles of 32
//   tokens x one 32-wide k block, with the quants in the order the matrix
//   cores read them (one 16-byte load per lane per block) and the 32 scales
//   permuted to the rows each lane's accumulators hold;
// - mmvq_q8_0_kernel: per wavefront 32 tokens x 32 or 64 batch columns. Each k
//   block is one v_mfma_i32_32x32x32_i8 per 32 columns, giving the exact integer
//   dot of every (token, column) pair; the float accumulation then follows the reference
//   kernel exactly (four accumulators by b % 4, fmaf(d_w * d_x, dot, acc),
//   then (A0 + A2) + (A1 + A3)), so y is the reference's to the last bit.
//
// Bound: HBM (34 bytes per 32 weights, read once; activations and y are small
// beside them) and, as the batch grows, the VALU's operations per
// (token, column, block) that the reference's float order needs (convert the
// integer dot, fused multiply-add; the scale product is a second matrix
// instruction).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/oxide_sampler.h"

namespace oxs_lm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kQ81Bytes = 36;       // {f16 d, f16 sum, int8 qs[32]} (common_types.cuh:8-11)
constexpr int kQ80Bytes = 34;       // {f16 d, int8 qs[32]} (common_types.cuh:13-16)
constexpr int kPackedBlock = 1088;  // 32 tokens x one k block: 64 lanes x 16 quant bytes, then 32 f16 scales
constexpr int kGroupsPerBlock = 4;  // token groups (wavefronts) per workgroup
constexpr int kThreads = 256;

__device__ __forceinline__ float half_to_float(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }

__device__ __forceinline__ uint16_t float_to_half(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }

// Row i of the 32 x 32 MFMA output held in register r of a lane in half g
// (lanes 32g .. 32g + 31): 8 (r / 4) + 4 g + r % 4.
__device__ __forceinline__ uint32_t out_row(uint32_t r, uint32_t g) { return 8u * (r >> 2) + 4u * g + (r & 3u); }

// quantize_f32_to_q8_1_cuda_kernel (norms_rope.cu:2-29): eight 32-lane groups
// per workgroup, one q8_1 block each.
__global__ __launch_bounds__(kThreads) void quantize_q8_1_kernel(const float* __restrict__ x, uint32_t nblocks,
                                                                 uint8_t* __restrict__ y) {
  const uint32_t lane = threadIdx.x & 31u;
  const uint32_t blk = blockIdx.x * (kThreads / 32) + (threadIdx.x >> 5);
  if (blk >= nblocks) return;  // the whole 32-lane group leaves together
  const float v = x[(size_t)blk * 32 + lane];
  float amax = fabsf(v), sum = v;
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) {
    amax = fmaxf(amax, __shfl_xor(amax, o, 32));
    sum += __shfl_xor(sum, o, 32);
  }
  const float d = amax / 127.0f;
  const float id = d > 0.0f ? 1.0f / d : 0.0f;
  uint8_t* out = y + (size_t)blk * kQ81Bytes;
  out[4 + lane] = (uint8_t)(int8_t)roundf(v * id);
  if (lane == 0) {
    *(uint16_t*)out = float_to_half(d);
    *(uint16_t*)(out + 2) = float_to_half(sum);
  }
}

// One wavefront per (token group, k block): lane l writes quant bytes
// [16 (l / 32), +16) of token 32 tg + l % 32 at offset 16 l; lanes 0..31 write
// the scales, position p holding token out_row(p % 16, p / 16). Tokens past m
// are zero.
__global__ __launch_bounds__(kThreads) void pack_q8_0_kernel(const uint8_t* __restrict__ w, uint32_t m, uint32_t nb,
                                                             uint64_t pieces, uint8_t* __restrict__ out) {
  const uint64_t gid = (uint64_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  if (gid >= pieces) return;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t tg = (uint32_t)(gid / nb), b = (uint32_t)(gid % nb);
  uint8_t* dst = out + gid * kPackedBlock;
  {
    const uint32_t t = tg * 32u + (lane & 31u), g = lane >> 5;
    uint32_t q[4] = {0u, 0u, 0u, 0u};
    if (t < m) {
      const uint8_t* src = w + ((size_t)t * nb + b) * kQ80Bytes + 2 + 16 * g;  // 2-byte aligned
#pragma unroll
      for (int i = 0; i < 16; ++i) q[i / 4] |= (uint32_t)src[i] << (8 * (i % 4));
    }
    *(uint4*)(dst + 16 * lane) = make_uint4(q[0], q[1], q[2], q[3]);
  }
  if (lane < 32) {
    const uint32_t t = tg * 32u + out_row(lane & 15u, lane >> 4);
    uint16_t s = 0;
    if (t < m) {
      const uint8_t* src = w + ((size_t)t * nb + b) * kQ80Bytes;
      s = (uint16_t)(src[0] | (src[1] << 8));
    }
    *(uint16_t*)(dst + 1024 + 2 * lane) = s;
  }
}

// mmvq_q8_0_cuda_kernel (quant_gemv_standard.cu:425-513) for 32 * TILES
// columns x 32 * WAVES tokens per workgroup; each of its wavefronts owns one
// group of 32 tokens and all of the columns, so the weights are read once per
// column block. With several column blocks, the workgroups of one token range
// sit 8 apart in launch order: workgroups go round-robin over the 8 XCDs, so
// they run on the same XCD at about the same time and the later ones read the
// weights from that XCD's L2 instead of HBM.
// - Weights go straight to registers, PF groups of four k blocks ahead: a
//   block's registers are reloaded as soon as its last matrix instruction has
//   read them.
// - The activations of a group are staged once per workgroup in LDS
//   (double-buffered, one barrier per group): quants as
//   [k block][half g][column][16 bytes], scales as [column][k block].
// - The scale products d_w * d_x of a 32 x 32 tile are one more matrix
//   instruction: an outer product of the two half scales (k = 0 of eight, the
//   others zero). A product of two halves has at most 22 significant bits, so
//   its f32 value is exact, as the reference's is. It takes 16 vector
//   instructions per tile and k block off the VALU, which bound this kernel.
// Wavefronts past the last token group recompute the last one and store
// nothing.
//
// Bound: HBM up to 32 columns (128256 x 4096: 97.4 us at 5 columns, 5.8 TB/s;
// 105 at 32), then the issue of converts and FMAs, which two wavefronts per SIMD
// overlap with the loads (64 columns: 122 us, 4.8 TB/s; 128: 208). The kernel
// before it (32 columns per wavefront, scale products on the VALU, weights one
// group ahead) took 119, 125, 215 and 397 us. Measured and left out: 64 columns
// with four wavefronts per workgroup (they spill; 181 us), two groups staged per
// barrier (123).
constexpr int kGroupBlocks = 4;   // k blocks per group (one per accumulator)

typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

// One half scale as the only nonzero entry of a lane's four (w: the half in
// the low 16 bits, zero above).
__device__ __forceinline__ v4h lone_half(uint32_t w) {
  const uint64_t v = w;
  return __builtin_bit_cast(v4h, v);
}

// A 32-bit byte offset whose widening stays next to the load that uses it, so
// that the load takes a scalar base and this offset.
__device__ __forceinline__ uint32_t local_offset(uint32_t o) {
  asm("" : "+v"(o));
  return o;
}
__device__ __forceinline__ uint64_t local_offset(uint64_t o) { return o; }

// WAVES: token groups (wavefronts) per workgroup
template <int TILES, int PF, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void mmvq_q8_0_kernel(float* __restrict__ y,
                                                                  const uint8_t* __restrict__ wp,
                                                                  const uint8_t* __restrict__ x, uint32_t m,
                                                                  uint32_t nb, uint32_t batch, uint32_t ncb,
                                                                  uint32_t vec_out) {
  constexpr int kMmThreads = 64 * WAVES;
  constexpr int COLS = 32 * TILES;
  constexpr int PLANE = COLS + 1;  // 16-byte entries per (block, half) plane; the odd one spreads the banks
  constexpr int XW = COLS * kGroupBlocks * 9;  // dwords of x per group
  constexpr int XR = (XW + kMmThreads - 1) / kMmThreads;
  // per group: quants as [k block][half g][column][16 bytes], then the scales
  // as [k block][column] pairs {half scale, 0}, as the matrix instruction
  // takes them; after the two buffers, zeros for lanes 32..63's scales
  constexpr int XD = kGroupBlocks * 2 * PLANE * 4;
  constexpr int XG = XD + kGroupBlocks * COLS * 2;
  __shared__ __align__(16) uint32_t s_x[2 * XG + (XG - XD)];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  // token block tb and column block cb: in each run of 8 * ncb workgroups,
  // workgroup 8 c + i holds token block i of the run and column block c
  uint32_t tb, cb;
  {
    const uint32_t per = 8u * ncb, full = (gridDim.x / per) * per;
    if (blockIdx.x < full) {
      const uint32_t run = blockIdx.x / per, r = blockIdx.x - run * per;
      tb = run * 8u + (r & 7u);
      cb = r >> 3;
    } else {
      const uint32_t r = blockIdx.x - full;
      tb = (full / per) * 8u + r / ncb;
      cb = r - (r / ncb) * ncb;
    }
  }
  const uint32_t groups = (m + 31u) / 32u;
  const uint32_t tg = tb * WAVES + wave;
  const bool live = tg < groups;
  const uint32_t g = lane >> 5, j = lane & 31u;
  const uint32_t c0 = cb * COLS;
  const uint32_t ngroups = nb / kGroupBlocks;

  // staging: dword i of a group's COLS x 36 dwords, for i = tid, tid + kMmThreads, ...:
  // consecutive lanes read consecutive dwords of a column's 144 bytes
  // (offsets from the column block; 32 bits for 64 columns, which the host
  // takes only where they suffice)
  using XOff = std::conditional_t<TILES == 1, uint64_t, uint32_t>;
  const uint8_t* xc = x + (size_t)c0 * nb * kQ81Bytes;
  XOff x_src[XR];
  uint32_t x_dst[XR], x_and[XR], xr[XR];
#pragma unroll
  for (int i = 0; i < XR; ++i) {
    const uint32_t w = min(tid + (uint32_t)i * kMmThreads, (uint32_t)XW - 1u);
    const uint32_t col = w / 36u, d = w - col * 36u, b = d / 9u, e = d - b * 9u;
    x_src[i] = (XOff)min(col, batch - 1u - c0) * nb * kQ81Bytes + d * 4u;  // + 144 per group
    x_dst[i] = e == 0u ? XD + (b * COLS + col) * 2u
                       : ((b * 2u + ((e - 1u) >> 2)) * PLANE + col) * 4u + ((e - 1u) & 3u);
    x_and[i] = e == 0u ? 0xffffu : 0xffffffffu;  // the scale's word without the sum beside it
  }
  auto stage_load = [&](uint32_t grp) {
    const uint8_t* p = xc + (size_t)min(grp, ngroups - 1u) * (kGroupBlocks * kQ81Bytes);
#pragma unroll
    for (int i = 0; i < XR; ++i) xr[i] = *(const uint32_t*)(p + local_offset(x_src[i]));  // 4-byte aligned
  };
  auto stage_store = [&](uint32_t buf) {  // (threads past the group's dwords repeat its last one)
#pragma unroll
    for (int i = 0; i < XR; ++i) s_x[buf * XG + x_dst[i]] = xr[i] & x_and[i];
  };

  // weights: this wavefront's tiles are contiguous; lane l's quants at 16 l,
  // token j's scale at position 16 ((j / 4) % 2) + 4 (j / 8) + j % 4
  const uint8_t* wg = wp + (size_t)(live ? tg : groups - 1u) * nb * kPackedBlock;
  const uint32_t q_off = 16u * lane;
  const uint32_t s_off = 1024u + 2u * (16u * ((j >> 2) & 1u) + 4u * (j >> 3) + (j & 3u));
  v4i wa[PF][kGroupBlocks];
  uint32_t ws[PF][kGroupBlocks];
  auto group_at = [&](uint32_t grp) {
    return wg + (size_t)min(grp, ngroups - 1u) * (kGroupBlocks * kPackedBlock);
  };
  auto weight_load = [&](int set, int q, const uint8_t* at) {
    wa[set][q] = *(const v4i*)(at + q * kPackedBlock + local_offset(q_off));
    ws[set][q] = *(const uint16_t*)(at + q * kPackedBlock + local_offset(s_off));
  };

  float acc[TILES][kGroupBlocks][16];
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int q = 0; q < kGroupBlocks; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][q][r] = 0.0f;
  const v16i zi = {};
  const v16f zf = {};

  stage_load(0);
#pragma unroll
  for (int s = 0; s < PF; ++s)
#pragma unroll
    for (int q = 0; q < kGroupBlocks; ++q) weight_load(s, q, group_at((uint32_t)s));
  // zeros: the scales' second words, which staging never writes, and lanes 32..63's scales
  for (uint32_t i = tid; i < 2u * kGroupBlocks * COLS; i += kMmThreads)
    s_x[(i / (kGroupBlocks * COLS)) * XG + XD + (i % (kGroupBlocks * COLS)) * 2u + 1u] = 0u;
  for (uint32_t i = tid; i < (uint32_t)(XG - XD); i += kMmThreads) s_x[2 * XG + i] = 0u;
  stage_store(0);
  __syncthreads();
  uint32_t buf = 0;
  // one group of four k blocks, from weight set s
  auto group = [&](auto sc, uint32_t grp) {
    constexpr int s = decltype(sc)::value;
    stage_load(grp + 1u);
    const uint8_t* next = group_at(grp + PF);
    const uint32_t* xg = s_x + buf * XG;
    const uint32_t* xq = xg + (g * PLANE + j) * 4u;
    const uint32_t* xd = (g ? s_x + 2 * XG : xg + XD) + 2u * j;
    // a tile's columns are read from LDS one tile ahead
    uint4 bq;
    uint64_t dx;
    auto tile_read = [&](int q, int t) {
      bq = *(const uint4*)(xq + (q * 2 * PLANE + 32 * t) * 4);
      dx = *(const uint64_t*)(xd + (q * COLS + 32 * t) * 2);
    };
    tile_read(0, 0);
#pragma unroll
    for (int q = 0; q < kGroupBlocks; ++q) {
      // the outer product's k = 0 entries are in lanes 0..31
      const v4h dw = lone_half(g ? 0u : ws[s][q]);
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
        const v4i bv = {(int)bq.x, (int)bq.y, (int)bq.z, (int)bq.w};
        const v16i d = __builtin_amdgcn_mfma_i32_32x32x32_i8(wa[s][q], bv, zi, 0, 0, 0);
        const v16f dd = __builtin_amdgcn_mfma_f32_32x32x8f16(dw, __builtin_bit_cast(v4h, dx), zf, 0, 0, 0);
        if (t + 1 < TILES) tile_read(q, t + 1);
        else if (q + 1 < kGroupBlocks) tile_read(q + 1, 0);
        if (t + 1 == TILES) weight_load(s, q, next);  // this block's registers, PF groups ahead
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          acc[t][q][r] = __builtin_fmaf(dd[r], (float)d[r], acc[t][q][r]);
          asm("" : "+v"(acc[t][q][r]));  // computed here: not put off to the end of the group
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    buf ^= 1u;
    stage_store(buf);
    __syncthreads();
  };
  // (No branch leaves the unrolled groups: with one, the wait before a
  // register's use would count the loads of the shortest path through the
  // loop, and the weights would be waited for almost as soon as issued.)
  uint32_t g0 = 0;
  for (; g0 + PF <= ngroups; g0 += PF) {
    group(std::integral_constant<int, 0>{}, g0);
    if constexpr (PF > 1) group(std::integral_constant<int, 1>{}, g0 + 1u);
    if constexpr (PF > 2) group(std::integral_constant<int, 2>{}, g0 + 2u);
    if constexpr (PF > 3) group(std::integral_constant<int, 3>{}, g0 + 3u);
  }
  if (g0 < ngroups) group(std::integral_constant<int, 0>{}, g0);
  if constexpr (PF > 2) {
    if (g0 + 1u < ngroups) group(std::integral_constant<int, 1>{}, g0 + 1u);
    if (g0 + 2u < ngroups) group(std::integral_constant<int, 2>{}, g0 + 2u);
  }
  if (!live) return;

  // (A0 + A2) + (A1 + A3); registers 4 q' .. 4 q' + 3 hold four consecutive tokens
  const bool vec = vec_out != 0u;  // m % 4 == 0 and y 16-byte aligned: float4 stores
#pragma unroll
  for (int t = 0; t < TILES; ++t) {
    const uint32_t col = c0 + 32u * t + j;
    if (col >= batch) continue;
    float* yrow = y + (size_t)col * m;
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * qq + e;
        v[e] = (acc[t][0][r] + acc[t][2][r]) + (acc[t][1][r] + acc[t][3][r]);
      }
      const uint32_t tok = tg * 32u + out_row(4u * qq, g);
      if (vec && tok + 3u < m) {
        *(float4*)(yrow + tok) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (tok + e < m) yrow[tok + e] = v[e];
      }
    }
  }
}

// The same product for batches of one or two columns, where a 32-column MFMA
// tile would be almost idle (128256 x 4096: 96.0 and 93.7 us against 97.4 for
// the MFMA kernel), and for three or four where that kernel's tokens per workgroup
// leave CUs idle (below). Each workgroup first stages the whole of x
// (NC columns x every k block) in LDS, then each wavefront walks its 32
// tokens with no further barrier: lane (j, g) takes 16 quant bytes of token j
// per block (the packed layout's MFMA order), four dot4 products per column,
// and the lane pair (j, j + 32) adds its halves into the block's exact
// integer dot. The float accumulation is the reference's, as above. Bound:
// HBM.
template <int NC>
__global__ __launch_bounds__(kThreads) void mmvq_q8_0_small_kernel(float* __restrict__ y,
                                                                   const uint8_t* __restrict__ wp,
                                                                   const uint8_t* __restrict__ x, uint32_t m,
                                                                   uint32_t nb, uint32_t batch) {
  extern __shared__ __align__(16) uint8_t s_small[];
  uint4* s_q = (uint4*)s_small;                              // [NC][nb][2] quant halves
  float* s_d = (float*)(s_small + (size_t)NC * nb * 32);     // [NC][nb] scales
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  for (uint32_t i = tid; i < NC * nb; i += kThreads) {
    const uint32_t c = i / nb, b = i - c * nb;
    const uint32_t* p = (const uint32_t*)(x + ((size_t)min(c, batch - 1u) * nb + b) * kQ81Bytes);
    s_d[i] = half_to_float((uint16_t)(p[0] & 0xffffu));
    s_q[2 * i] = make_uint4(p[1], p[2], p[3], p[4]);
    s_q[2 * i + 1] = make_uint4(p[5], p[6], p[7], p[8]);
  }
  __syncthreads();
  const uint32_t tg = blockIdx.x * kGroupsPerBlock + wave;
  if (tg >= (m + 31u) / 32u) return;
  const uint32_t g = lane >> 5, j = lane & 31u;
  // this token's scale: position 16 ((j / 4) % 2) + 4 (j / 8) + j % 4 of the permuted scales
  const uint32_t sp = 16u * ((j >> 2) & 1u) + 4u * (j >> 3) + (j & 3u);
  const uint8_t* wg = wp + (size_t)tg * nb * kPackedBlock;
  float acc[NC][4];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[c][q] = 0.0f;
  for (uint32_t b0 = 0; b0 < nb; b0 += 4) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t b = b0 + q;
      const uint8_t* blk = wg + (size_t)b * kPackedBlock;
      const uint4 wq = *(const uint4*)(blk + 16 * lane);
      const float dw = half_to_float(*(const uint16_t*)(blk + 1024 + 2 * sp));
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const uint4 xq = s_q[2 * (c * nb + b) + g];
        int dot = __builtin_amdgcn_sdot4((int)wq.x, (int)xq.x, 0, false);
        dot = __builtin_amdgcn_sdot4((int)wq.y, (int)xq.y, dot, false);
        dot = __builtin_amdgcn_sdot4((int)wq.z, (int)xq.z, dot, false);
        dot = __builtin_amdgcn_sdot4((int)wq.w, (int)xq.w, dot, false);
        dot += __shfl_xor(dot, 32);
        acc[c][q] = __builtin_fmaf(dw * s_d[c * nb + b], (float)dot, acc[c][q]);
      }
    }
  }
  const uint32_t tok = tg * 32u + j;
  if (g == 0 && tok < m) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if ((uint32_t)c < batch) y[(size_t)c * m + tok] = (acc[c][0] + acc[c][2]) + (acc[c][1] + acc[c][3]);
  }
}

}  // namespace oxs_lm

static int launch_status() { return hipGetLastError() == hipSuccess ? OXS_OK : OXS_ERR_HIP; }

extern "C" int oxs_quantize_q8_1(const float* x, uint32_t n, void* y_q8_1, void* stream) {
  const uint32_t nblocks = n / 32u;
  if (nblocks == 0) return OXS_OK;
  if (!x || !y_q8_1) return OXS_ERR_INVALID_ARGUMENT;
  if (((uintptr_t)x & 3u) || ((uintptr_t)y_q8_1 & 1u)) return OXS_ERR_INVALID_ARGUMENT;  // float loads, half stores
  const uint32_t per = oxs_lm::kThreads / 32;
  hipLaunchKernelGGL(oxs_lm::quantize_q8_1_kernel, dim3((nblocks + per - 1) / per), dim3(oxs_lm::kThreads), 0,
                     (hipStream_t)stream, x, nblocks, (uint8_t*)y_q8_1);
  return launch_status();
}

extern "C" size_t oxs_q8_0_packed_bytes(uint32_t m, uint32_t k) {
  if (k == 0 || k % 128u != 0) return 0;
  return (size_t)((m + 31u) / 32u) * (k / 32u) * oxs_lm::kPackedBlock;
}

extern "C" int oxs_pack_q8_0(const void* w, uint32_t m, uint32_t k, void* w_packed, void* stream) {
  if (k == 0 || k % 128u != 0) return OXS_ERR_UNSUPPORTED;
  if (m == 0) return OXS_OK;
  if (!w || !w_packed) return OXS_ERR_INVALID_ARGUMENT;
  if ((uintptr_t)w_packed & 15u) return OXS_ERR_INVALID_ARGUMENT;  // 16-byte stores
  const uint32_t nb = k / 32u;
  const uint64_t pieces = (uint64_t)((m + 31u) / 32u) * nb;
  const uint64_t per = oxs_lm::kThreads / 64;
  const uint64_t grid = (pieces + per - 1) / per;
  if (grid > 0x7fffffffull) return OXS_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(oxs_lm::pack_q8_0_kernel, dim3((uint32_t)grid), dim3(oxs_lm::kThreads), 0, (hipStream_t)stream,
                     (const uint8_t*)w, m, nb, pieces, (uint8_t*)w_packed);
  return launch_status();
}

extern "C" int oxs_mmvq_q8_0(float* y, const void* w_packed, const void* x_q8_1, uint32_t m, uint32_t k,
                             uint32_t batch, void* stream) {
  if (m == 0 || k == 0 || batch == 0) return OXS_OK;  // as launch_cuda_mmvq_q8_0's early return
  if (k % 128u != 0) return OXS_ERR_UNSUPPORTED;
  if (!y || !w_packed || !x_q8_1) return OXS_ERR_INVALID_ARGUMENT;
  // 16-byte weight loads, 4-byte activation loads, 4-byte stores
  if (((uintptr_t)w_packed & 15u) || ((uintptr_t)x_q8_1 & 3u) || ((uintptr_t)y & 3u)) return OXS_ERR_INVALID_ARGUMENT;
  const uint32_t vec_out = (m % 4u == 0u && ((uintptr_t)y & 15u) == 0u) ? 1u : 0u;
  const uint32_t groups = (m + 31u) / 32u;
  const uint32_t gx = (groups + oxs_lm::kGroupsPerBlock - 1) / oxs_lm::kGroupsPerBlock;
  const uint32_t nb = k / 32u;
  const uint32_t blocks256 = (groups + 7u) / 8u;  // workgroups of 256 tokens: one per CU at a time
  // Three or four columns take the small kernel where the MFMA kernel's second round of
  // workgroups is little used or its start is much of a short row, us for 3 columns
  // (MFMA / small): k = 128, m = 32000 5.0 / 3.8; above 256 workgroups k = 896, m =
  // 128256 25.4 / 21.7, 80000 21.1 / 16.4, k = 1536 35.7 / 34.4, 29.4 / 25.1, but k = 2048,
  // m = 128256 45.4 / 47.5; with less than half of the last round in use k = 2048, m =
  // 134000 59.0 / 52.4, 80000 37.1 / 32.0, k = 3072 51.9 / 46.4, and past 512
  // workgroups k = 4096, m = 134000 125 / 113; but k = 4096, m = 80000 76 / 85, and
  // past 512 full ones k = 1152, m = 262144 61 / 63.
  // Up to 256 workgroups MFMA wins from k = 512 on (50257 x 896 12.4 / 13.7).
  const bool half_round = blocks256 % 256u != 0u && blocks256 % 256u < 128u;
  const bool small4 =
      k <= 256u || (blocks256 > 256u && (k <= 1024u || (k <= 1536u && blocks256 <= 512u) ||
                                         (half_round && (k <= 3072u || blocks256 > 512u))));
  const uint32_t nc = batch <= 2u ? batch : 4u;  // columns that the small kernel stages
  if ((batch <= 2u || (batch <= 4u && small4)) && (size_t)nc * nb * 36u <= 65536u) {  // the whole of x fits in LDS
    const size_t lds = (size_t)nc * nb * 36u;
    const auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(gx), dim3(oxs_lm::kThreads), lds, (hipStream_t)stream, y,
                         (const uint8_t*)w_packed, (const uint8_t*)x_q8_1, m, nb, batch);
    };
    if (nc == 1u) go(oxs_lm::mmvq_q8_0_small_kernel<1>);
    else if (nc == 2u) go(oxs_lm::mmvq_q8_0_small_kernel<2>);
    else go(oxs_lm::mmvq_q8_0_small_kernel<4>);
    return launch_status();
  }
  // Columns and tokens per workgroup. 64 columns read the weights half as often
  // as 32 and 256 tokens stage x half as often as 128, but each needs enough
  // workgroups to occupy the 256 CUs, one per CU; the line lies between 125 and
  // 197 of them. Measured, us: 64 columns / 32 columns for a batch of 64 at
  // k = 4096, 125 workgroups (m = 32000) 45.0 / 39.5, 197 (m = 50257) 61.7 / 69.4;
  // 256 / 128 tokens at a batch of 5, 125 workgroups 30.3 / 25.6, 197 42.2 / 45.6.
  // Rows of up to 512 weights take 128 tokens again above one round of the CUs, where
  // a workgroup's start is much of its time: m = 128256, k = 512, batch 32 22.5 / 20.7, m = 200000
  // 37.1 / 31.7. (64 columns also need their offsets into x within 32 bits.)
  constexpr uint64_t kEnough = 160;
  const auto blocks = [&](uint32_t cols, uint32_t waves) {
    return (uint64_t)((groups + waves - 1u) / waves) * ((batch + cols - 1u) / cols);
  };
  const bool wide = batch > 32u && blocks(64u, 8u) >= kEnough && (uint64_t)64u * nb * oxs_lm::kQ81Bytes <= 0xffffffffull;
  const uint32_t cols = wide ? 64u : 32u;
  const uint64_t b32 = blocks(32u, 8u);
  const uint32_t waves = wide || (b32 >= kEnough && !(k <= 512u && b32 > 256u)) ? 8u : 4u;
  const uint64_t grid = blocks(cols, waves);
  // (the bound is on 128 tokens x 32 columns per workgroup whatever the launch takes)
  if ((uint64_t)gx * ((batch + 31u) / 32u) > 0x7fffffffull) return OXS_ERR_INVALID_ARGUMENT;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((uint32_t)grid), dim3(64u * waves), 0, (hipStream_t)stream, y,
                       (const uint8_t*)w_packed, (const uint8_t*)x_q8_1, m, nb, batch, (batch + cols - 1u) / cols,
                       vec_out);
  };
  if (wide) go(oxs_lm::mmvq_q8_0_kernel<2, 2, 8>);
  else if (waves == 8u) go(oxs_lm::mmvq_q8_0_kernel<1, 4, 8>);
  else go(oxs_lm::mmvq_q8_0_kernel<1, 4, 4>);
  return launch_status();
}
