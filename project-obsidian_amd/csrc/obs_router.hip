// obs_router.hip — MoE router: 8-bit gate logits and softmax/top-k.
//
// Replaces Model::gate_gpu (src/forward.rs:386-397) + dequant_matvec_8bit.metal
// and MoeRouter::route/route_dispatch (src/router.rs:25-83) + moe_routing_topk.metal.
//
// Logit reduction order (documented, reproduced by the CPU oracle): for each
// (token, expert row) one wave of 64 lanes; lane l owns the in/64 contiguous
// columns [l*in/64, (l+1)*in/64) and accumulates acc = fma(w_c, x_c, acc) in
// column order from 0; the lanes are combined by an xor butterfly with
// offsets 1, 2, 4, ..., 32 (wave_sum_asc in the decode kernels; the two
// kernels below add the same pairs as a tree over the lane partials).
//
// Selection (moe_routing_topk.metal:24-56): under the reference rule each
// logit is first rounded to f16 (dequant_matvec_8bit.metal:30 stores halves);
// m = max logit; e_i = exp(l_i - m)
// with the deterministic exp; S = sum e_i where lane l adds e_l, e_{l+64},
// e_{l+128}, e_{l+192} in that order and the lanes are combined by the xor
// butterfly; p_i = e_i / S; k rounds of argmax over p (lower id wins ties);
// wsum = serial sum of the selected p; if norm_topk and wsum > 0 the weights
// are p / wsum (under the reference rule f16(p) and f16(f16(p) / wsum)). All
// steps are correctly rounded operations, so the ids and weights are
// bit-identical to the oracle given the same logits.
#include "obs_internal.hpp"

#include <algorithm>

namespace {

using namespace obsd;

constexpr uint32_t ROUTE_FUSED_TOKENS = 8;

// ---- logits of many tokens, on the matrix cores (logits_by_rows: the line) ----
// A lane's partial of the reduction order above is a chain of in/64 fp32 fmas over
// consecutive columns. v_mfma_f32_16x16x1_4b_f32 is one such fma (correctly
// rounded, subnormals kept: checked bit for bit) for each (token, expert) of four
// independent 16 x 16 blocks, so a block takes one of the 64 chains and C = in/64
// instructions walk its columns in order: the logits keep every bit.
//
// A workgroup owns 16 experts and runs one tile of 16 tokens after another; wave w
// owns the chains [8w, 8w + 8) as two quads. Lane l = 16 b + r feeds chain 4q + b:
// its C columns of expert r, dequantized once into registers (fma(q, s, b)), and of
// token r, from LDS (read whole rows at a time by coalesced loads, the next tile's
// while this one is multiplied; the row padding spreads the 16-byte reads of 16
// rows over the banks). The chain sums are added as the butterfly adds them, a
// pairwise tree in chain order: a wave's 8 in registers, the 8 waves' in LDS.
//
// Bound by the fp32 matrix rate (256 FLOP/clock/CU): 6.8 us at 2,048 tokens x 128
// experts x 2,048; a tile on every CU costs 2.6-3 us, 2.1 of them matrix
// instructions. The vector units have half that rate, and a partial per lane and
// pair had to pass through LDS. Logits and top-k launches, 128 experts: 512 tokens
// 14.6 -> 12.3 us, 2,048 35.3 -> 24.2, 4,096 61.5 -> 36.0 (256 experts 113 -> 59).
// Workgroups of one XCD share token tiles, so a row of x is read into one L2.
constexpr uint32_t LG_TILE = 16, LG_WAVES = 8;
typedef float f32x16_lg __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_lg __attribute__((ext_vector_type(4)));  // (an array of uint4 structs went to scratch)

template <uint32_t C>
constexpr size_t lg_lds_bytes() {  // staged rows of 64 C bf16 + 16 bytes
  return LG_TILE * (64u * C + 8u) * sizeof(uint16_t);
}

// ONE_SCALE: group >= C, one scale and bias per chain; else one per packed word.
template <uint32_t C, bool ONE_SCALE>
__global__ void __launch_bounds__(64 * LG_WAVES, C <= 32u ? 4 : 2)
    gate_logits_mfma_kernel(const uint32_t* __restrict__ w8, const uint16_t* __restrict__ s,
                            const uint16_t* __restrict__ b, const uint16_t* __restrict__ x,
                            float* __restrict__ logits, uint32_t T, uint32_t n_exp, uint32_t group,
                            uint32_t slots) {
  constexpr uint32_t in = 64u * C, STRIDE = in + 8u, XL = C / 4u;  // XL: 16-byte pieces of a tile per thread
  extern __shared__ __attribute__((aligned(16))) uint16_t s_x[];   // [LG_TILE][STRIDE]
  __shared__ float s_part[LG_WAVES][LG_TILE * LG_TILE];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, r = lane & 15u, blk = lane >> 4;
  const uint32_t etiles = (n_exp + LG_TILE - 1u) / LG_TILE, ttiles = (T + LG_TILE - 1u) / LG_TILE;
  const uint32_t p = blockIdx.x / 8u, e0 = p % etiles * LG_TILE;
  uint32_t tile = blockIdx.x % 8u + 8u * (p / etiles);  // then every 8 * slots
  if (tile >= ttiles) return;  // uniform per workgroup
  u32x4_lg xr[XL];
  auto load_x = [&](uint32_t tl) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < XL; ++i) {
      const uint32_t c = tid + 64u * LG_WAVES * i, row = min(tl * LG_TILE + c / (in / 8u), T - 1u);
      xr[i] = *reinterpret_cast<const u32x4_lg*>(x + static_cast<uint64_t>(row) * in + 8u * (c % (in / 8u)));
    }
  };
  load_x(tile);
  float wv[2][C];
  {
    const uint32_t e = min(e0 + r, n_exp - 1u), groups = in / group;  // a repeated row: computed, not stored
#pragma unroll
    for (uint32_t q = 0; q < 2; ++q) {
      const uint32_t c0 = C * (4u * (2u * wave + q) + blk);  // the chain's first column
      const uint32_t* wp = w8 + (static_cast<uint64_t>(e) * in + c0) / 4u;
      const uint64_t g0 = static_cast<uint64_t>(e) * groups;
      uint32_t wb[C / 4u];
      if constexpr (C >= 16u) {
#pragma unroll
        for (uint32_t i = 0; i < C / 16u; ++i) {
          const uint4 v = reinterpret_cast<const uint4*>(wp)[i];
          wb[4 * i] = v.x; wb[4 * i + 1] = v.y; wb[4 * i + 2] = v.z; wb[4 * i + 3] = v.w;
        }
      } else {
        const uint2 v = *reinterpret_cast<const uint2*>(wp);
        wb[0] = v.x; wb[1] = v.y;
      }
      float sc = bf16_to_f32(s[g0 + c0 / group]), bi = bf16_to_f32(b[g0 + c0 / group]);
#pragma unroll
      for (uint32_t i = 0; i < C / 4u; ++i) {
        if (!ONE_SCALE) {
          sc = bf16_to_f32(s[g0 + (c0 + 4u * i) / group]);
          bi = bf16_to_f32(b[g0 + (c0 + 4u * i) / group]);
        }
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
          wv[q][4 * i + j] = __builtin_fmaf(static_cast<float>((wb[i] >> (8u * j)) & 0xffu), sc, bi);
      }
    }
  }
  // a tile's logits from the waves' partials
  auto finish = [&](uint32_t tl) __attribute__((always_inline)) {
    if (tid < LG_TILE * LG_TILE) {
      const uint32_t t = tl * LG_TILE + tid / LG_TILE;
      uint32_t e = e0 + tid % LG_TILE;
      asm("" : "+v"(e));  // the address is formed here: kept over the tiles it went to scratch
      const float v = ((s_part[0][tid] + s_part[1][tid]) + (s_part[2][tid] + s_part[3][tid])) +
                      ((s_part[4][tid] + s_part[5][tid]) + (s_part[6][tid] + s_part[7][tid]));
      if (t < T && e < n_exp) logits[static_cast<uint64_t>(t) * n_exp + e] = v;
    }
  };
  for (uint32_t first = tile; tile < ttiles; tile += 8u * slots) {  // uniform per workgroup
    if (tile != first) {
      __syncthreads();  // the tile before has been read, its partials are written
      finish(tile - 8u * slots);
    }
#pragma unroll
    for (uint32_t i = 0; i < XL; ++i) {
      const uint32_t c = tid + 64u * LG_WAVES * i;
      *reinterpret_cast<u32x4_lg*>(s_x + c / (in / 8u) * STRIDE + 8u * (c % (in / 8u))) = xr[i];
    }
    __syncthreads();
    load_x(tile + 8u * slots);  // (past the last tile: its last row, never used)
    f32x16_lg acc[2];  // acc[q][4 b + i]: chain 4 (2 wave + q) + b, token 4 blk + i, expert r
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.0f;
    const uint16_t* xp = s_x + r * STRIDE + C * (8u * wave + blk);
#pragma unroll
    for (uint32_t i = 0; i < C / 8u; ++i) {
      u32x4_lg v[2];
#pragma unroll
      for (uint32_t q = 0; q < 2; ++q) v[q] = *reinterpret_cast<const u32x4_lg*>(xp + 4u * C * q + 8u * i);
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j)
#pragma unroll
        for (uint32_t q = 0; q < 2; ++q) {
          const uint32_t d = j < 2u ? v[q].x : j < 4u ? v[q].y : j < 6u ? v[q].z : v[q].w;
          acc[q] = __builtin_amdgcn_mfma_f32_16x16x1f32(j & 1u ? bf16hi(d) : bf16lo(d), wv[q][8 * i + j], acc[q], 0, 0, 0);
        }
    }
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i)
      s_part[wave][(4u * blk + i) * LG_TILE + r] =
          ((acc[0][i] + acc[0][4 + i]) + (acc[0][8 + i] + acc[0][12 + i])) +
          ((acc[1][i] + acc[1][4 + i]) + (acc[1][8 + i] + acc[1][12 + i]));
  }
  __syncthreads();
  finish(tile - 8u * slots);
}

// ---- few tokens, and the one-launch router of up to 8 -------------------------
// The routing step of the one-launch router (obs_route): where the range's
// ids and weights go, and the per-range counters that elect the workgroup
// that routes (context memory, zero between launches); with NORM the RMSNorm
// weight and epsilon of the input rows.
struct RouteTail {
  uint32_t* cnt;
  int32_t* ids;
  float* weights;
  uint32_t k;
  int norm_topk, rule;
  const uint16_t* norm_w;
  float eps;
};

// WPL = packed words per lane (in = 64 lanes * 4 cols * WPL). A wave keeps one
// expert row dequantized in registers; the workgroup stages the activation rows
// in LDS once for its 4 waves. Each lane's partial sum of every (token, row) pair
// goes to LDS, and one thread per pair adds the 64 partials in the butterfly's
// order: a wave reduction per pair (DPP steps and lane reads, ~20 dependent
// instructions) had cost as much as the pair's fmas.
// The grid is 8 times the workgroups the logits need, and only those with
// blockIdx.x % 8 == 0 work: the dispatcher deals workgroups round-robin over the
// 8 XCDs, so they all run on one XCD and the logits pass through its L2 (plain
// stores, polled past the CU's vector cache), as the fused decode's exchanges do.
// Each working workgroup counts itself in cnt[0] once its logits are stored, and
// the last to do so resets the counter and routes the tokens (route_topk_kernel's
// per-token wave). NQ: logit slots per lane when routing.
// NORM: each workgroup normalises the rows as it stages them, in obs_rmsnorm's
// sequence, so a decode layer needs no launch for the norm.
// FUSED off: the logits of few tokens alone, workgroup (x, y) the rows 4x.. and
// the tokens 8y..
template <int WPL, int NQ, bool NORM, bool FUSED>
__global__ void __launch_bounds__(256) route_rows_kernel(const uint32_t* __restrict__ w8,
                                                         const uint16_t* __restrict__ s,
                                                         const uint16_t* __restrict__ b,
                                                         const uint16_t* __restrict__ x,
                                                         float* __restrict__ logits, uint32_t T, uint32_t in,
                                                         uint32_t n_exp, uint32_t group, RouteTail rt) {
  constexpr int C = 4 * WPL;  // columns per lane
  // lane partials, 68 floats per pair: a thread's 16-byte reads of its pair hit
  // distinct banks across 16 consecutive threads
  constexpr uint32_t PART_STRIDE = 68;
  __shared__ __attribute__((aligned(16))) float s_part[ROUTE_FUSED_TOKENS * 4 * PART_STRIDE];
  extern __shared__ __attribute__((aligned(16))) uint16_t s_x[];  // [T][in]
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = threadIdx.x / 64u;
  if (FUSED && blockIdx.x % 8u != 0u) return;  // uniform: the working workgroups are on XCD 0
  const uint32_t bx = FUSED ? blockIdx.x / 8u : blockIdx.x, e0 = bx * 4u + wave;
  if (!FUSED) {
    const uint32_t t0 = blockIdx.y * ROUTE_FUSED_TOKENS;
    x += static_cast<uint64_t>(t0) * in;
    logits += static_cast<uint64_t>(t0) * n_exp;
    T = min(ROUTE_FUSED_TOKENS, T - t0);
  }
  const uint32_t words = in / 4, groups = in / group;
  // dequantize this lane's C weights of the row once (exact: byte*scale has <= 16 bits)
  float wv[C];
  {
    const uint32_t e = min(e0, n_exp - 1u);  // a row past the last expert: computed, not stored
    const uint32_t* wr = w8 + static_cast<uint64_t>(e) * words + lane * WPL;
    const uint16_t* sr = s + static_cast<uint64_t>(e) * groups;
    const uint16_t* br = b + static_cast<uint64_t>(e) * groups;
#pragma unroll
    for (int j = 0; j < WPL; ++j) {
      const uint32_t word = wr[j];
      const uint32_t g = (lane * C + 4 * j) / group;
      const float sc = bf16_to_f32(sr[g]), bi = bf16_to_f32(br[g]);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        wv[4 * j + q] = __builtin_fmaf(static_cast<float>((word >> (8 * q)) & 0xffu), sc, bi);
    }
  }
  if constexpr (NORM) {
    for (uint32_t t = wave; t < T; t += 4u) {  // one wave per row, the lane's C columns
      uint4 xv[C / 8], nv[C / 8];
#pragma unroll
      for (int i = 0; i < C / 8; ++i) {
        xv[i] = reinterpret_cast<const uint4*>(x + static_cast<uint64_t>(t) * in + lane * C)[i];
        nv[i] = reinterpret_cast<const uint4*>(rt.norm_w + lane * C)[i];
      }
      float ss = 0.0f;
#pragma unroll
      for (int i = 0; i < C / 8; ++i) {
        const uint32_t d[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          ss = __builtin_fmaf(bf16lo(d[j]), bf16lo(d[j]), ss);
          ss = __builtin_fmaf(bf16hi(d[j]), bf16hi(d[j]), ss);
        }
      }
      const float inv = 1.0f / __builtin_sqrtf(wave_sum_asc(ss) / static_cast<float>(in) + rt.eps);
#pragma unroll
      for (int i = 0; i < C / 8; ++i) {
        const uint32_t d[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w}, g[4] = {nv[i].x, nv[i].y, nv[i].z, nv[i].w};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[j] = pack_bf16x2((bf16lo(d[j]) * inv) * bf16lo(g[j]), (bf16hi(d[j]) * inv) * bf16hi(g[j]));
        *reinterpret_cast<uint4*>(s_x + t * in + lane * C + 8 * i) = make_uint4(o[0], o[1], o[2], o[3]);
      }
    }
  } else {
    const uint32_t row_chunks = in / 8u;  // 16-byte chunks per activation row
    for (uint32_t c = threadIdx.x; c < T * row_chunks; c += 256u)
      *reinterpret_cast<uint4*>(s_x + 8u * c) = *reinterpret_cast<const uint4*>(x + 8u * static_cast<uint64_t>(c));
  }
  __syncthreads();
  // the lane partials (serial fma over the lane's columns) of every (token, row)
  // pair go to LDS, pair-major
  if (e0 < n_exp) {  // wave-uniform
    for (uint32_t t = 0; t < T; ++t) {
      const uint16_t* xr = s_x + t * in + lane * C;
      float xf[C];
#pragma unroll
      for (int c = 0; c < C; c += 8) {
        const uint4 xv = *reinterpret_cast<const uint4*>(xr + c);
        xf[c + 0] = bf16lo(xv.x); xf[c + 1] = bf16hi(xv.x); xf[c + 2] = bf16lo(xv.y); xf[c + 3] = bf16hi(xv.y);
        xf[c + 4] = bf16lo(xv.z); xf[c + 5] = bf16hi(xv.z); xf[c + 6] = bf16lo(xv.w); xf[c + 7] = bf16hi(xv.w);
      }
      float acc = 0.0f;
#pragma unroll
      for (int c = 0; c < C; ++c) acc = __builtin_fmaf(wv[c], xf[c], acc);
      s_part[(t * 4u + wave) * PART_STRIDE + lane] = acc;
    }
  }
  __syncthreads();
  // one thread per pair: its 64 lane partials summed in the xor-butterfly order
  // (at step off, lane l adds lane l ^ off; lane 0's value is the sum over
  // aligned blocks, pairwise in index order), as wave_sum_asc does in registers
  for (uint32_t pr = threadIdx.x; pr < T * 4u; pr += 256u) {
    const uint32_t t = pr / 4u, e = bx * 4u + pr % 4u;
    float v[64];
    const float4* src = reinterpret_cast<const float4*>(s_part + pr * PART_STRIDE);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float4 q = src[i];
      v[4 * i] = q.x; v[4 * i + 1] = q.y; v[4 * i + 2] = q.z; v[4 * i + 3] = q.w;
    }
#pragma unroll
    for (int off = 1; off < 64; off *= 2)
#pragma unroll
      for (int l = 0; l < 64; l += 2 * off) v[l] = v[l] + v[l + off];
    float* dst = logits + static_cast<uint64_t>(t) * n_exp + e;
    if (e < n_exp) {
      if (FUSED)  // to the XCD's L2, where the routing workgroup reads it
        __hip_atomic_store(reinterpret_cast<uint32_t*>(dst), __float_as_uint(v[0]), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WAVEFRONT);
      else
        *dst = v[0];
    }
  }
  if constexpr (FUSED) {
    // A thread's logit stores have reached the L2 once its memory counter is 0,
    // before the workgroup counts itself; the routing workgroup's loads
    // follow the count it read and skip its CU's vector cache.
    __shared__ uint32_t s_last;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();
    if (threadIdx.x == 0) {
      const uint32_t before = __hip_atomic_fetch_add(rt.cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_last = before + 1u == gridDim.x / 8u ? 1u : 0u;
      if (s_last) __hip_atomic_store(rt.cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (s_last == 0u) return;  // uniform per workgroup
    for (uint32_t t = wave; t < T; t += 4u) {  // uniform per wave
      const uint32_t* lg = reinterpret_cast<const uint32_t*>(logits + static_cast<uint64_t>(t) * n_exp);
      float l[NQ];
#pragma unroll
      for (int j = 0; j < NQ; ++j)
        l[j] = __uint_as_float(__hip_atomic_load(lg + min(lane + 64u * j, n_exp - 1u), __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT));
      int32_t id;
      float w;
      if (rt.k == 8)
        route_wave_top8<NQ>(l, n_exp, rt.norm_topk, rt.rule, lane, &id, &w);
      else
        route_wave<NQ>(l, n_exp, rt.k, rt.norm_topk, rt.rule, lane, &id, &w);
      if (lane < rt.k) {
        rt.ids[static_cast<uint64_t>(t) * rt.k + lane] = id;
        rt.weights[static_cast<uint64_t>(t) * rt.k + lane] = w;
      }
    }
  }
}

// One wave per token (route_wave); n_exp <= 64 * NQ, k <= 64.
template <int NQ>
__global__ void __launch_bounds__(256) route_topk_kernel(const float* __restrict__ logits, int32_t* __restrict__ ids,
                                                         float* __restrict__ weights, uint32_t T, uint32_t n_exp,
                                                         uint32_t k, int norm_topk, int rule) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t t = blockIdx.x * 4 + threadIdx.x / 64;
  if (t >= T) return;  // wave-uniform: every lane of a wave shares t
  const float* lg = logits + static_cast<uint64_t>(t) * n_exp;
  float l[NQ];
#pragma unroll
  for (int j = 0; j < NQ; ++j) l[j] = lg[min(lane + 64u * j, n_exp - 1u)];
  int32_t id;
  float w;
  if (k == 8)
    route_wave_top8<NQ>(l, n_exp, norm_topk, rule, lane, &id, &w);
  else
    route_wave<NQ>(l, n_exp, k, norm_topk, rule, lane, &id, &w);
  if (lane < k) {
    ids[static_cast<uint64_t>(t) * k + lane] = id;
    weights[static_cast<uint64_t>(t) * k + lane] = w;
  }
}

}  // namespace

namespace obs {

int check_router_shape(obs_ctx* ctx, const char* who, uint32_t in, uint32_t n_exp, uint32_t group) {
  if (n_exp == 0 || n_exp > 256)
    return set_error(ctx, OBS_E_SHAPE, "%s: n_exp must be in [1, 256] (got %u)", who, n_exp);
  if (group == 0 || group % 4 != 0 || in % group != 0)
    return set_error(ctx, OBS_E_SHAPE, "%s: in (%u) must be a multiple of group (%u), group a multiple of 4", who, in, group);
  if (in != 512 && in != 1024 && in != 2048 && in != 4096)
    return set_error(ctx, OBS_E_SHAPE, "%s: in must be 512, 1024, 2048 or 4096 (got %u)", who, in);
  // a lane's contiguous span must not straddle groups in a way the per-word
  // scale lookup cannot express: 4 | group makes every word single-group.
  return OBS_OK;
}

// Whether T tokens' logits take the kernel of few tokens: while its workgroups (4
// experts x 8 tokens each) fit the GPU at once, two to a CU up to in = 2048 and one
// at 4096. The matrix kernel has a tile's instructions in one workgroup whatever the
// number of tokens. Measured, us, matrix kernel | this one, 128 experts: in = 2048
// 64 tokens 6.5 | 5.0, 128 (512 workgroups) 6.5 | 5.7, 160 6.6 | 6.8; in = 4096 64
// tokens (256 workgroups) 10.3 | 8.6, 72 10.3 | 12.0; 256 experts: in = 2048 64
// tokens 6.5 | 5.7, 72 6.5 | 6.8; in = 4096 32 tokens 10.3 | 8.5, 48 10.3 | 12.1.
// (At 512 and 1,024 columns it stays ahead to twice as many.)
bool logits_by_rows(const obs_ctx* ctx, uint32_t T, uint32_t in, uint32_t n_exp) {
  const uint64_t wgs = ((n_exp + 3u) / 4u) * ((static_cast<uint64_t>(T) + ROUTE_FUSED_TOKENS - 1u) / ROUTE_FUSED_TOKENS);
  return wgs <= static_cast<uint64_t>(ctx->num_cus) * (in <= 2048u ? 2u : 1u);
}

// The matrix kernel's staged tiles are more than 64 KB from in = 2048 on: its
// limit is raised once per context, at creation.
int router_init(obs_ctx* ctx) {
  const struct {
    const void* fn;
    size_t lds;
  } ks[] = {{reinterpret_cast<const void*>(&gate_logits_mfma_kernel<32u, true>), lg_lds_bytes<32u>()},
            {reinterpret_cast<const void*>(&gate_logits_mfma_kernel<32u, false>), lg_lds_bytes<32u>()},
            {reinterpret_cast<const void*>(&gate_logits_mfma_kernel<64u, true>), lg_lds_bytes<64u>()},
            {reinterpret_cast<const void*>(&gate_logits_mfma_kernel<64u, false>), lg_lds_bytes<64u>()}};
  for (const auto& k : ks)
    OBS_HIP_TRY(ctx, hipFuncSetAttribute(k.fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(k.lds)));
  return OBS_OK;
}

// One workgroup per CU (two up to in = 2048, by LDS and registers), each running
// its share of the token tiles.
int launch_gate_logits(obs_ctx* ctx, const uint32_t* w8, const uint16_t* s, const uint16_t* b,
                       const uint16_t* x, float* logits, uint32_t T, uint32_t in, uint32_t n_exp,
                       uint32_t group) {
  if (logits_by_rows(ctx, T, in, n_exp)) {
    const dim3 grid((n_exp + 3) / 4, (T + ROUTE_FUSED_TOKENS - 1u) / ROUTE_FUSED_TOKENS);
    const size_t lds = sizeof(uint16_t) * ROUTE_FUSED_TOKENS * in;
    const RouteTail none{};
#define OBS_LOGITS(WPL)                                                                                     \
  OBS_LAUNCH(ctx, "q8_gate_logits", (route_rows_kernel<WPL, 1, false, false><<<grid, 256, lds, ctx->stream>>>( \
                                        w8, s, b, x, logits, T, in, n_exp, group, none)))
    switch (in) {
      case 512: OBS_LOGITS(2); break;
      case 1024: OBS_LOGITS(4); break;
      case 2048: OBS_LOGITS(8); break;
      default: OBS_LOGITS(16); break;
    }
#undef OBS_LOGITS
    return OBS_OK;
  }
  const uint32_t ttiles = (T + LG_TILE - 1u) / LG_TILE, etiles = (n_exp + LG_TILE - 1u) / LG_TILE;
  const uint32_t resident = static_cast<uint32_t>(ctx->num_cus) * (in <= 2048u ? 2u : 1u);
  const uint32_t slots = std::min((ttiles + 7u) / 8u, std::max(1u, resident / (8u * etiles)));
  const uint32_t grid = 8u * slots * etiles;
#define OBS_LOGITS2(C, ONE)                                                                                      \
  OBS_LAUNCH(ctx, "q8_gate_logits",                                                                              \
             (gate_logits_mfma_kernel<C, ONE><<<grid, 64 * LG_WAVES, lg_lds_bytes<C>(), ctx->stream>>>(          \
                 w8, s, b, x, logits, T, n_exp, group, slots)))
#define OBS_LOGITS(C) \
  if (group >= C) OBS_LOGITS2(C, true); else OBS_LOGITS2(C, false)
  switch (in) {  // C = in / 64; group divides in, a power of two, so it divides C or is a multiple of it
    case 512: OBS_LOGITS(8u); break;
    case 1024: OBS_LOGITS(16u); break;
    case 2048: OBS_LOGITS(32u); break;
    default: OBS_LOGITS(64u); break;
  }
#undef OBS_LOGITS
#undef OBS_LOGITS2
  return OBS_OK;
}

int launch_route_topk(obs_ctx* ctx, const float* logits, int32_t* ids, float* w, uint32_t T,
                      uint32_t n_exp, uint32_t k, int norm_topk, int rule) {
  if (n_exp <= 64)
    OBS_LAUNCH(ctx, "route_topk", route_topk_kernel<1><<<(T + 3) / 4, 256, 0, ctx->stream>>>(logits, ids, w, T, n_exp, k, norm_topk, rule));
  else if (n_exp <= 128)
    OBS_LAUNCH(ctx, "route_topk", route_topk_kernel<2><<<(T + 3) / 4, 256, 0, ctx->stream>>>(logits, ids, w, T, n_exp, k, norm_topk, rule));
  else
    OBS_LAUNCH(ctx, "route_topk", route_topk_kernel<4><<<(T + 3) / 4, 256, 0, ctx->stream>>>(logits, ids, w, T, n_exp, k, norm_topk, rule));
  return OBS_OK;
}

// The router step (logits, then routing). One launch for up to 8 tokens on a
// device whose workgroups b share an XCD by b % 8 (the exchange stays in one
// L2); otherwise the two launches.
template <int NQ>
int launch_route_fused(obs_ctx* ctx, const uint32_t* w8, const uint16_t* s, const uint16_t* b, const uint16_t* x,
                       float* logits, uint32_t T, uint32_t in, uint32_t n_exp, uint32_t group, const RouteTail& rt) {
  const dim3 grid(8u * ((n_exp + 3) / 4), 1);
  const size_t lds = sizeof(uint16_t) * T * in;  // at most 64 KB (8 tokens, in = 4096)
#define OBS_ROUTE2(WPL, NORM)                                                                         \
  OBS_LAUNCH(ctx, "route_fused", (route_rows_kernel<WPL, NQ, NORM, true><<<grid, 256, lds, ctx->stream>>>( \
                                     w8, s, b, x, logits, T, in, n_exp, group, rt)))
#define OBS_ROUTE1(WPL) \
  if (rt.norm_w) OBS_ROUTE2(WPL, true); else OBS_ROUTE2(WPL, false)
  switch (in) {
    case 512: OBS_ROUTE1(2); break;
    case 1024: OBS_ROUTE1(4); break;
    case 2048: OBS_ROUTE1(8); break;
    default: OBS_ROUTE1(16); break;
  }
#undef OBS_ROUTE1
#undef OBS_ROUTE2
  return OBS_OK;
}

bool route_one_launch(const obs_ctx* ctx, uint32_t T) {
  return T <= ROUTE_FUSED_TOKENS && ctx->xcd_map_ok;
}

int launch_route(obs_ctx* ctx, const uint32_t* w8, const uint16_t* s, const uint16_t* b, const uint16_t* x,
                 float* logits, int32_t* ids, float* w, uint32_t T, uint32_t in, uint32_t n_exp, uint32_t group,
                 uint32_t k, int norm_topk, int rule, const uint16_t* norm_w, float eps) {
  if (route_one_launch(ctx, T)) {
    const RouteTail rt{ctx->route_cnt, ids, w, k, norm_topk, rule, norm_w, eps};
    if (n_exp <= 64) return launch_route_fused<1>(ctx, w8, s, b, x, logits, T, in, n_exp, group, rt);
    if (n_exp <= 128) return launch_route_fused<2>(ctx, w8, s, b, x, logits, T, in, n_exp, group, rt);
    return launch_route_fused<4>(ctx, w8, s, b, x, logits, T, in, n_exp, group, rt);
  }
  const int rc = launch_gate_logits(ctx, w8, s, b, x, logits, T, in, n_exp, group);
  if (rc) return rc;
  return launch_route_topk(ctx, logits, ids, w, T, n_exp, k, norm_topk, rule);
}

}  // namespace obs

extern "C" {

int obs_q8_gate_logits(obs_ctx* ctx, const uint32_t* w8, const uint16_t* scales, const uint16_t* biases,
                       const uint16_t* x, float* logits, uint32_t T, uint32_t in, uint32_t n_exp,
                       uint32_t group) {
  if (!ctx) return OBS_E_INVALID;
  if (!w8 || !scales || !biases || !x || !logits)
    return obs::set_error(ctx, OBS_E_INVALID, "obs_q8_gate_logits: null pointer");
  int rc = obs::check_router_shape(ctx, "obs_q8_gate_logits", in, n_exp, group);
  if (rc) return rc;
  if (!obs::aligned(x, 16) || !obs::aligned(w8, 16))
    return obs::set_error(ctx, OBS_E_ALIGN, "obs_q8_gate_logits: x and w8 must be 16-byte aligned");
  if (T == 0) return OBS_OK;
  return obs::launch_gate_logits(ctx, w8, scales, biases, x, logits, T, in, n_exp, group);
}

int obs_route(obs_ctx* ctx, const uint32_t* w8, const uint16_t* scales, const uint16_t* biases, const uint16_t* x,
              float* logits, int32_t* ids, float* weights, uint32_t T, uint32_t in, uint32_t n_exp, uint32_t group,
              uint32_t k, int norm_topk, int rule) {
  if (!ctx) return OBS_E_INVALID;
  if (!w8 || !scales || !biases || !x || !logits || !ids || !weights)
    return obs::set_error(ctx, OBS_E_INVALID, "obs_route: null pointer");
  int rc = obs::check_router_shape(ctx, "obs_route", in, n_exp, group);
  if (rc) return rc;
  if (k == 0 || k > n_exp || k > 64)
    return obs::set_error(ctx, OBS_E_SHAPE, "obs_route: k must be in [1, min(n_exp, 64)] (got %u)", k);
  if (rule != OBS_ROUTE_REF && rule != OBS_ROUTE_F32)
    return obs::set_error(ctx, OBS_E_INVALID, "obs_route: unknown rule %d", rule);
  if (!obs::aligned(x, 16) || !obs::aligned(w8, 16))
    return obs::set_error(ctx, OBS_E_ALIGN, "obs_route: x and w8 must be 16-byte aligned");
  if (T == 0) return OBS_OK;
  return obs::launch_route(ctx, w8, scales, biases, x, logits, ids, weights, T, in, n_exp, group, k, norm_topk, rule,
                           nullptr, 0.0f);
}

int obs_route_topk(obs_ctx* ctx, const float* logits, int32_t* ids, float* weights, uint32_t T,
                   uint32_t n_exp, uint32_t k, int norm_topk, int rule) {
  if (!ctx) return OBS_E_INVALID;
  if (!logits || !ids || !weights) return obs::set_error(ctx, OBS_E_INVALID, "obs_route_topk: null pointer");
  if (n_exp == 0 || n_exp > 256)
    return obs::set_error(ctx, OBS_E_SHAPE, "obs_route_topk: n_exp must be in [1, 256] (got %u)", n_exp);
  if (k == 0 || k > n_exp || k > 64)
    return obs::set_error(ctx, OBS_E_SHAPE, "obs_route_topk: k must be in [1, min(n_exp, 64)] (got %u)", k);
  if (rule != OBS_ROUTE_REF && rule != OBS_ROUTE_F32)
    return obs::set_error(ctx, OBS_E_INVALID, "obs_route_topk: unknown rule %d", rule);
  if (T == 0) return OBS_OK;
  return obs::launch_route_topk(ctx, logits, ids, weights, T, n_exp, k, norm_topk, rule);
}

}  // extern "C"
