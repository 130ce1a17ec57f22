// obs_decode.hip — decode MoE half of one layer for one token
// (src/forward.rs:421-441): router -> per selected expert
// h = silu(gate . x) * (up . x) -> y_r = down . h -> y = sum_r w_r * y_r.
//
// The reference pages the 8 selected experts off SSD into a pool
// (disk_io.rs:79-102, forward.rs:431-435) and issues 5 dispatches per expert;
// here the whole expert table is resident in HBM (stacked [E, ...] tensors)
// and the layer runs as 3 launches: router (with the post-attention norm),
// gate/up+SwiGLU, down+combine (one or two more where the router is not one
// launch: its top-k and the norm). Weights are read exactly once with 16-byte coalesced loads.
//
// Numerics: dots accumulate in fp32 using the per-group factored form
//   sum_c (q_c*s + b) * x_c = s * sum_c q_c*x_c + b * sum_c x_c
// (exact algebra; it removes one multiply-add per weight). h stays fp32,
// the combine accumulates sum_r w_r*y_r in fp32 (forward.rs:440) and rounds
// once to bf16.
#include "obs_q4_dequant.hpp"

namespace obs {
int check_router_shape(obs_ctx* ctx, const char* who, uint32_t in, uint32_t n_exp, uint32_t group);
}  // namespace obs

namespace {

using namespace obsd;

// A lane's share of a packed row: CH chunks of W words (8 columns each), chunk i
// at word W * (lane + 64 i), so a wave reads a row in whole, contiguous runs.
template <int W, int CH>
__device__ __forceinline__ void load_words(const uint32_t* row, uint32_t lane, uint32_t (&q)[W * CH]) {
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const uint32_t* p = row + W * (lane + 64u * i);
    if constexpr (W == 4) {
      const uint4 v = load_stream(p);
      q[4 * i] = v.x; q[4 * i + 1] = v.y; q[4 * i + 2] = v.z; q[4 * i + 3] = v.w;
    } else {
      const uint2 v = *reinterpret_cast<const uint2*>(p);
      q[2 * i] = v.x; q[2 * i + 1] = v.y;
    }
  }
}

// Sums of q_j * x_j over the 8 nibbles of w: even nibbles as the f16 subnormals
// q * 2^-24, odd ones as q * 2^-20 (masked in place), each converted exactly
// inside an fp32 fma. 13 instructions instead of the 19 of a shift, mask and
// conversion per nibble; the caller puts the powers of two back (dot_mix_sum).
// Exact while q_j * x_j * 2^-24 is not below fp32's normal range: a chunk whose
// values are all tiny is scaled first (mix_scale_up).
struct DotMix {
  float a24, a20;
};
__device__ __forceinline__ void dot8_q4_mix(uint32_t w, const float* x, DotMix& d) {
  const uint32_t w8 = w >> 8;
  const uint32_t p04 = w & 0x000F000Fu, p15 = w & 0x00F000F0u, p26 = w8 & 0x000F000Fu, p37 = w8 & 0x00F000F0u;
  d.a24 = fma_mix_f16<0>(p04, x[0], d.a24);
  d.a20 = fma_mix_f16<0>(p15, x[1], d.a20);
  d.a24 = fma_mix_f16<0>(p26, x[2], d.a24);
  d.a20 = fma_mix_f16<0>(p37, x[3], d.a20);
  d.a24 = fma_mix_f16<1>(p04, x[4], d.a24);
  d.a20 = fma_mix_f16<1>(p15, x[5], d.a20);
  d.a24 = fma_mix_f16<1>(p26, x[6], d.a24);
  d.a20 = fma_mix_f16<1>(p37, x[7], d.a20);
}
__device__ __forceinline__ float dot_mix_sum(const DotMix& d, float unscale) {
  return __builtin_fmaf(d.a20, 0x1p20f * unscale, d.a24 * (0x1p24f * unscale));
}

// The power of two that a lane's values of one chunk take before dot8_q4_mix,
// from their largest magnitude: 2^90 where all of them are below 2^-98 (2^-24 of
// that is 27 bits above fp32's smallest subnormal), else 1. Values that small
// beside larger ones of the chunk lose nothing that its sum would keep.
__device__ __forceinline__ float mix_scale_up(float largest) { return largest < 0x1p-98f ? 0x1p90f : 1.0f; }
__device__ __forceinline__ float mix_scale_down(float largest) { return largest < 0x1p-98f ? 0x1p-90f : 1.0f; }

constexpr uint32_t GU_WAVES = 4;
constexpr uint32_t GU_WAVES_MAX = 2048;  // waves a gate/up launch aims at: 8 per CU

// h[r, o] = silu(gate_e[o] . x) * (up_e[o] . x) for e = ids[r], one wave per PR
// consecutive (r, o) row pairs; lane l owns the 8*W columns of CH chunks (as
// load_words), each inside one quantization group. H = 512 * W * CH.
//
// Bound by HBM: k * I * H weights of both matrices at 4.5 bits. Every wave
// requests all of its rows at once (6 row pairs of H = 4096 are 24 KB a wave, 196
// KB in flight per CU), so the first rows' dots run while the last are on their
// way. Up to 12,288 row pairs (k 6, I 2048) all waves of an H = 4096 launch are
// resident at once, with 8 to a CU; at k 8, I 2048 a third of them run in a second
// round. E 16, H 4096, I 2048, k 6 (57 MB): 20.3 us with 2 rows a wave, 20.1 with 3,
// 22.2 with 6 and a shift-and-convert dot product over 64 contiguous columns a
// lane, 18.8 with the one below, 19.2 (3.0 TB/s) with its scaling of tiny chunks.
// NORM: x is normalised first, in obs_rmsnorm's sequence (its sum of squares over
// the columns a lane owns there), so no launch of its own is needed (4.6 us).
template <int W, int CH, int PR, bool NORM>
__global__ void __launch_bounds__(GU_WAVES * 64, 2) decode_gateup_kernel(
    const uint32_t* __restrict__ gw, const uint16_t* __restrict__ gs, const uint16_t* __restrict__ gb,
    const uint32_t* __restrict__ uw, const uint16_t* __restrict__ us, const uint16_t* __restrict__ ub,
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ norm_w, float eps, const int32_t* __restrict__ ids,
    float* __restrict__ h, uint32_t n_exp, uint32_t k, uint32_t I) {
  constexpr uint32_t C = 8 * W, H = 64 * C * CH, GROUP = 64, words = H / 8, groups = H / GROUP;
  constexpr uint32_t XQ = CH * C / 8;  // 16-byte pieces of a lane's share of x
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t row0 = __builtin_amdgcn_readfirstlane((blockIdx.x * GU_WAVES + threadIdx.x / 64u) * PR);
  const uint32_t rows = k * I;
  if (row0 >= rows) return;  // wave-uniform
  int32_t e[PR];
#pragma unroll
  for (int i = 0; i < PR; ++i) e[i] = ids[min(row0 + i, rows - 1u) / I];
  uint4 xq[XQ], nq[XQ], xn[XQ];
#pragma unroll
  for (uint32_t j = 0; j < XQ; ++j) {
    const uint32_t col = C * (lane + 64u * (8u * j / C)) + 8u * j % C;
    xq[j] = *reinterpret_cast<const uint4*>(x + col);
    if (NORM) {
      nq[j] = *reinterpret_cast<const uint4*>(norm_w + col);
      if (CH > 1) xn[j] = *reinterpret_cast<const uint4*>(x + CH * C * lane + 8u * j);  // the lane's columns in obs_rmsnorm
    }
  }
  uint32_t gq[PR][W * CH], uq[PR][W * CH];
  uint16_t sg[PR][CH], bg[PR][CH], su[PR][CH], bu[PR][CH];
#pragma unroll
  for (int i = 0; i < PR; ++i) {  // an id out of range: expert 0's rows, their sums unused
    const uint32_t ei = static_cast<uint32_t>(e[i]) < n_exp ? static_cast<uint32_t>(e[i]) : 0u;
    const uint64_t wrow = static_cast<uint64_t>(ei) * I + min(row0 + i, rows - 1u) % I;
    load_words<W, CH>(gw + wrow * words, lane, gq[i]);
    load_words<W, CH>(uw + wrow * words, lane, uq[i]);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const uint64_t srow = wrow * groups + (lane + 64u * c) * C / GROUP;
      sg[i][c] = gs[srow];
      bg[i][c] = gb[srow];
      su[i][c] = us[srow];
      bu[i][c] = ub[srow];
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // every load is on its way before the first wait
  float inv = 0.0f;
  if (NORM) {
    float ss = 0.0f;
#pragma unroll
    for (uint32_t j = 0; j < XQ; ++j) {
      const uint4 v = CH > 1 ? xn[j] : xq[j];
      const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        ss = __builtin_fmaf(bf16lo(d[p]), bf16lo(d[p]), ss);
        ss = __builtin_fmaf(bf16hi(d[p]), bf16hi(d[p]), ss);
      }
    }
    inv = 1.0f / __builtin_sqrtf(wave_sum_asc(ss) / static_cast<float>(H) + eps);
  }
  float xf[CH * C], xs[CH], unscale[CH];
#pragma unroll
  for (uint32_t j = 0; j < XQ; ++j) {
    const uint32_t d[4] = {xq[j].x, xq[j].y, xq[j].z, xq[j].w}, n[4] = {nq[j].x, nq[j].y, nq[j].z, nq[j].w};
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const uint32_t v = NORM ? pack_bf16x2((bf16lo(d[p]) * inv) * bf16lo(n[p]), (bf16hi(d[p]) * inv) * bf16hi(n[p])) : d[p];
      xf[8 * j + 2 * p] = bf16lo(v);
      xf[8 * j + 2 * p + 1] = bf16hi(v);
    }
  }
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    xs[c] = 0.0f;
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) xs[c] = xs[c] + xf[C * c + j];
    float m = 0.0f;
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) m = fmaxf(m, __builtin_fabsf(xf[C * c + j]));
    const float up = mix_scale_up(m);
    unscale[c] = mix_scale_down(m);
#pragma unroll
    for (uint32_t j = 0; j < C; ++j) xf[C * c + j] *= up;
  }
  float my_g = 0.0f, my_u = 0.0f;  // lane i < PR: the sums of row row0 + i
  bool mine = false;
#pragma unroll
  for (int i = 0; i < PR; ++i) {
    float pg = 0.0f, pu = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      DotMix ag{0.0f, 0.0f}, au{0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < W; ++j) {
        dot8_q4_mix(gq[i][W * c + j], xf + C * c + 8 * j, ag);
        dot8_q4_mix(uq[i][W * c + j], xf + C * c + 8 * j, au);
      }
      pg = __builtin_fmaf(bf16_to_f32(sg[i][c]), dot_mix_sum(ag, unscale[c]), __builtin_fmaf(bf16_to_f32(bg[i][c]), xs[c], pg));
      pu = __builtin_fmaf(bf16_to_f32(su[i][c]), dot_mix_sum(au, unscale[c]), __builtin_fmaf(bf16_to_f32(bu[i][c]), xs[c], pu));
    }
    pg = wave_sum_asc(pg);
    pu = wave_sum_asc(pu);
    my_g = lane == static_cast<uint32_t>(i) ? pg : my_g;
    my_u = lane == static_cast<uint32_t>(i) ? pu : my_u;
    mine = lane == static_cast<uint32_t>(i) ? static_cast<uint32_t>(e[i]) < n_exp : mine;
  }
  if (lane < PR && row0 + lane < rows) h[row0 + lane] = mine ? silu_mul(my_g, my_u) : 0.0f;
}

// y[o] = (residual[o]) + sum_r w_r * (down_{e_r}[o] . h_r), one wave per output
// row. The k * I columns of an output row are k * I / 32 chunks (16 bytes of one
// expert's row, half a quantization group); lane l takes chunks l, l + 64, ..., so
// a row's weights are at most 8 whole-wave loads (NC) whatever I is.
//
// Bound by HBM (k * I * H weights): a wave requests all of its weights before it
// uses the first. h is staged in LDS in the order the lanes read it
// ([chunk / 64][float4][lane], the lane xor-ed with the float4's index so that the
// stores of one chunk's 8 float4 spread over the banks), where the chunk's scaling
// of tiny values is also done once for the 8 waves. E 16, H 4096, I 2048, k 6 (28
// MB): 10.4 us (10.1 without that scaling; 11.1 with two output rows per wave, which
// reads h half as often). A lane that kept the I / 8 values of its part of a rank's
// h in registers spilled them from I = 1,024 on: 72.5 us.
constexpr uint32_t DN_WAVES = 8;

template <int NC>
__global__ void __launch_bounds__(DN_WAVES * 64, 2) decode_down_kernel(
    const uint32_t* __restrict__ dw, const uint16_t* __restrict__ ds, const uint16_t* __restrict__ db,
    const float* __restrict__ h, const int32_t* __restrict__ ids, const float* __restrict__ wts,
    const uint16_t* __restrict__ residual, uint16_t* __restrict__ y, uint32_t n_exp, uint32_t k,
    uint32_t H, uint32_t I, uint32_t group) {
  __shared__ float4 s_h[NC * 8 * 64];
  __shared__ float s_un[NC * 64];  // per chunk: what undoes its scaling (mix_scale_up)
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t o = __builtin_amdgcn_readfirstlane(blockIdx.x * DN_WAVES + tid / 64u);  // < H (H % 8 == 0)
  const uint32_t cpr = I / 32u, nch = k * cpr;  // chunks of an expert's row, of an output row
  float4 hv[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i)
    hv[i] = reinterpret_cast<const float4*>(h)[min(tid + 512u * i, nch * 8u - 1u)];
  uint32_t eo[NC];
  float wr[NC];
  bool ok[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const uint32_t c = lane + 64u * i, r = min(c, nch - 1u) / cpr;
    const int32_t e = ids[r];
    ok[i] = c < nch && static_cast<uint32_t>(e) < n_exp;
    eo[i] = ok[i] ? static_cast<uint32_t>(e) : 0u;  // an absent chunk reads expert 0's row, its sum unused
    wr[i] = wts[r];
  }
  uint4 q[NC];
  uint16_t sc[NC], bi[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const uint32_t col = min(lane + 64u * i, nch - 1u) % cpr;  // chunk within the expert's row
    const uint64_t wrow = static_cast<uint64_t>(eo[i]) * H + o;
    q[i] = load_stream(dw + wrow * (I / 8u) + 4u * col);
    const uint64_t srow = wrow * (I / group) + 32u * col / group;
    sc[i] = ds[srow];
    bi[i] = db[srow];
  }
  __builtin_amdgcn_sched_barrier(0);  // the weights are on their way before h is waited for
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const uint32_t f = tid + 512u * i, c = f / 8u, j = f % 8u;  // float4 j of chunk c
    float m = fmaxf(fmaxf(__builtin_fabsf(hv[i].x), __builtin_fabsf(hv[i].y)),
                    fmaxf(__builtin_fabsf(hv[i].z), __builtin_fabsf(hv[i].w)));
    m = fmaxf(m, dpp_f32<DPP_XOR1>(m));  // over the chunk's 8 lanes
    m = fmaxf(m, dpp_f32<DPP_XOR2>(m));
    m = fmaxf(m, dpp_f32<DPP_HALF_MIRROR>(m));
    const float up = mix_scale_up(m);
    const float4 v = make_float4(hv[i].x * up, hv[i].y * up, hv[i].z * up, hv[i].w * up);
    s_h[(c / 64u * 8u + j) * 64u + ((c % 64u) ^ j)] = v;  // (past nch: a copy of the last, never used)
    if (j == 0u) s_un[c] = mix_scale_down(m);
  }
  __syncthreads();
  float acc = 0.0f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const float unscale = s_un[64 * i + lane];
    float hf[32], hs = 0.0f;
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) {
      const float4 v = s_h[(i * 8u + j) * 64u + (lane ^ j)];
      hf[4 * j] = v.x; hf[4 * j + 1] = v.y; hf[4 * j + 2] = v.z; hf[4 * j + 3] = v.w;
      hs = hs + ((v.x + v.y) + (v.z + v.w));
    }
    DotMix a{0.0f, 0.0f};
    dot8_q4_mix(q[i].x, hf, a);
    dot8_q4_mix(q[i].y, hf + 8, a);
    dot8_q4_mix(q[i].z, hf + 16, a);
    dot8_q4_mix(q[i].w, hf + 24, a);
    const float part = __builtin_fmaf(bf16_to_f32(sc[i]), dot_mix_sum(a, unscale), bf16_to_f32(bi[i]) * (hs * unscale));
    acc = ok[i] ? __builtin_fmaf(wr[i], part, acc) : acc;
  }
  acc = wave_sum_asc(acc);
  if (lane == 0) y[o] = f32_to_bf16(residual ? bf16_to_f32(residual[o]) + acc : acc);
}

constexpr size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

}  // namespace

namespace obs {

int check_moe_config(obs_ctx* ctx, const char* who, const obs_moe_config* cfg) {
  if (!cfg) return set_error(ctx, OBS_E_INVALID, "%s: null config", who);
  if (cfg->group != 64) return set_error(ctx, OBS_E_SHAPE, "%s: group must be 64 (got %u)", who, cfg->group);
  if (cfg->hidden != 1024 && cfg->hidden != 2048 && cfg->hidden != 4096)
    return set_error(ctx, OBS_E_SHAPE, "%s: hidden must be 1024, 2048 or 4096 (got %u)", who, cfg->hidden);
  if (cfg->inter == 0 || cfg->inter % 256 != 0 || cfg->inter > 2048)
    return set_error(ctx, OBS_E_SHAPE, "%s: inter must be a multiple of 256 in [256, 2048] (got %u)", who, cfg->inter);
  if (cfg->n_exp == 0 || cfg->n_exp > 256)
    return set_error(ctx, OBS_E_SHAPE, "%s: n_exp must be in [1, 256] (got %u)", who, cfg->n_exp);
  if (cfg->top_k == 0 || cfg->top_k > cfg->n_exp || cfg->top_k > 8)
    return set_error(ctx, OBS_E_SHAPE, "%s: top_k must be in [1, min(n_exp, 8)] (got %u)", who, cfg->top_k);
  if (cfg->route_rule != OBS_ROUTE_REF && cfg->route_rule != OBS_ROUTE_F32)
    return set_error(ctx, OBS_E_INVALID, "%s: unknown route_rule %d", who, cfg->route_rule);
  return OBS_OK;
}

int check_moe_layer(obs_ctx* ctx, const char* who, const obs_moe_layer* L) {
  if (!L) return set_error(ctx, OBS_E_INVALID, "%s: null layer", who);
  if (!L->gate_w || !L->gate_s || !L->gate_b || !L->up_w || !L->up_s || !L->up_b || !L->down_w ||
      !L->down_s || !L->down_b || !L->router_w || !L->router_s || !L->router_b)
    return set_error(ctx, OBS_E_INVALID, "%s: null weight pointer in layer", who);
  if (!aligned(L->gate_w, 16) || !aligned(L->up_w, 16) || !aligned(L->down_w, 16) || !aligned(L->router_w, 16))
    return set_error(ctx, OBS_E_ALIGN, "%s: packed weights must be 16-byte aligned", who);
  if (L->norm_w && !aligned(L->norm_w, 16))
    return set_error(ctx, OBS_E_ALIGN, "%s: norm_w must be 16-byte aligned", who);
  return OBS_OK;
}

// norm_w (with eps): x is the layer's input and is normalised by the gate/up
// launch; nullptr: x as it is.
int launch_decode_experts(obs_ctx* ctx, const obs_moe_config* cfg, const obs_moe_layer* L, const uint16_t* x,
                          const uint16_t* norm_w, const uint16_t* residual, uint16_t* y, const int32_t* ids,
                          const float* w, float* h) {
  const uint32_t H = cfg->hidden, I = cfg->inter, k = cfg->top_k, E = cfg->n_exp, G = cfg->group;
  const uint32_t rows = k * I;
#define OBS_GATEUP(W, CH, PR, NORM)                                                                               \
  OBS_LAUNCH(ctx, "decode_gateup",                                                                                \
             (decode_gateup_kernel<W, CH, PR, NORM>                                                               \
              <<<(rows + GU_WAVES * PR - 1) / (GU_WAVES * PR), GU_WAVES * 64, 0, ctx->stream>>>(                  \
                  L->gate_w, L->gate_s, L->gate_b, L->up_w, L->up_s, L->up_b, x, norm_w, cfg->rms_eps, ids, h, E, \
                  k, I)))
  // Row pairs per wave: as many as keep the launch at 8 waves per CU, at most 6
  // (the registers of the rows in flight at H = 4096).
#define OBS_GATEUP_ROWS(W, CH, NORM)                                      \
  do {                                                                  \
    if (rows <= GU_WAVES_MAX) OBS_GATEUP(W, CH, 1, NORM);                 \
    else if (rows <= 2 * GU_WAVES_MAX) OBS_GATEUP(W, CH, 2, NORM);        \
    else if (rows <= 4 * GU_WAVES_MAX) OBS_GATEUP(W, CH, 4, NORM);        \
    else OBS_GATEUP(W, CH, 6, NORM);                                      \
  } while (0)
#define OBS_GATEUP_NORM(W, CH)                                            \
  do {                                                                  \
    if (norm_w) OBS_GATEUP_ROWS(W, CH, true);                             \
    else OBS_GATEUP_ROWS(W, CH, false);                                   \
  } while (0)
  switch (H) {
    case 1024: OBS_GATEUP_NORM(2, 1); break;
    case 2048: OBS_GATEUP_NORM(4, 1); break;
    default: OBS_GATEUP_NORM(4, 2); break;
  }
#undef OBS_GATEUP_NORM
#undef OBS_GATEUP_ROWS
#undef OBS_GATEUP
#define OBS_DOWN(NC)                                                                                              \
  OBS_LAUNCH(ctx, "decode_down", (decode_down_kernel<NC><<<H / DN_WAVES, DN_WAVES * 64, 0, ctx->stream>>>(        \
                                     L->down_w, L->down_s, L->down_b, h, ids, w, residual, y, E, k, H, I, G)))
  switch ((rows / 32 + 63) / 64) {  // whole-wave loads per output row, at most 8
    case 1: OBS_DOWN(1); break;
    case 2: OBS_DOWN(2); break;
    case 3: OBS_DOWN(3); break;
    case 4: OBS_DOWN(4); break;
    case 5: OBS_DOWN(5); break;
    case 6: OBS_DOWN(6); break;
    case 7: OBS_DOWN(7); break;
    default: OBS_DOWN(8); break;
  }
#undef OBS_DOWN
  return OBS_OK;
}

// Validates a decode call and picks its path (the one-launch fused kernel, or
// the several launches).
int decode_plan(obs_ctx* ctx, const char* who, const obs_moe_config* cfg, const obs_moe_layer* layer,
                const uint16_t* x, const uint16_t* y, bool* fused) {
  int rc = check_moe_config(ctx, who, cfg);
  if (rc) return rc;
  rc = check_moe_layer(ctx, who, layer);
  if (rc) return rc;
  if (!x || !y) return set_error(ctx, OBS_E_INVALID, "%s: null x or y", who);
  if (!aligned(x, 16)) return set_error(ctx, OBS_E_ALIGN, "%s: x must be 16-byte aligned", who);
  const bool shape_ok = fused_decode_supported(cfg);
  // the one-launch path spins on values other workgroups publish: all of its
  // workgroups must be resident at once, one per CU, and each group of 32 must
  // share an XCD (its L2) as the probe at obs_create found
  const bool cus_ok = (dispatch_gate(ctx->num_cus, ctx->xcd_map_ok, ctx->inorder_ok) & OBS_PATH_FUSED_DECODE) != 0u;
  if (ctx->decode_path == OBS_DECODE_FUSED && !shape_ok)
    return set_error(ctx, OBS_E_SHAPE, "%s: the fused path needs hidden 2048, inter 768, top_k 8, group 64, n_exp <= 256",
                     who);
  if (ctx->decode_path == OBS_DECODE_FUSED && !cus_ok)
    return set_error(ctx, OBS_E_UNSUPPORTED,
                     "%s: the fused path needs %u CUs with each group b %% 8 on one XCD (the device has %d CUs; XCD map %s)",
                     who, fused_decode_workgroups(), ctx->num_cus, ctx->xcd_map_ok ? "as expected" : "not as expected");
  *fused = shape_ok && cus_ok && ctx->decode_path != OBS_DECODE_MULTI;
  return OBS_OK;
}

// Workspace of the several-launch path: logits [E] | ids [k] | w [k] | h [k, I] | normed x [H].
size_t multi_ws_bytes(const obs_moe_config* cfg) {
  return align256(sizeof(float) * cfg->n_exp) + align256(sizeof(int32_t) * cfg->top_k) +
         align256(sizeof(float) * cfg->top_k) + align256(sizeof(float) * cfg->top_k * cfg->inter) +
         align256(sizeof(uint16_t) * cfg->hidden);
}

// The several-launch path over a workspace of multi_ws_bytes(cfg) at `base`.
int decode_multi(obs_ctx* ctx, const obs_moe_config* cfg, const obs_moe_layer* layer, const uint16_t* x,
                 const uint16_t* residual, uint16_t* y, int32_t* ids_out, float* w_out, char* base) {
  const uint32_t E = cfg->n_exp, k = cfg->top_k, H = cfg->hidden, I = cfg->inter;
  const size_t off_ids = align256(sizeof(float) * E);
  const size_t off_w = off_ids + align256(sizeof(int32_t) * k);
  const size_t off_h = off_w + align256(sizeof(float) * k);
  const size_t off_xn = off_h + align256(sizeof(float) * k * I);
  float* logits = reinterpret_cast<float*>(base);
  int32_t* ids = ids_out ? ids_out : reinterpret_cast<int32_t*>(base + off_ids);
  float* w = w_out ? w_out : reinterpret_cast<float*>(base + off_w);
  float* h = reinterpret_cast<float*>(base + off_h);
  int rc;
  // The router and experts see rmsnorm(x) (forward.rs:419-421): normalised inside
  // the router's and the gate/up launch, or by a launch of its own where the
  // router takes two.
  const uint16_t* norm_w = layer->norm_w;
  if (norm_w && !route_one_launch(ctx, 1)) {
    uint16_t* xn = reinterpret_cast<uint16_t*>(base + off_xn);
    rc = launch_rmsnorm(ctx, x, norm_w, xn, 1, H, cfg->rms_eps);
    if (rc) return rc;
    x = xn;
    norm_w = nullptr;
  }
  rc = launch_route(ctx, layer->router_w, layer->router_s, layer->router_b, x, logits, ids, w, 1, H, E, cfg->group, k,
                    cfg->norm_topk, cfg->route_rule, norm_w, cfg->rms_eps);
  if (rc) return rc;
  return launch_decode_experts(ctx, cfg, layer, x, norm_w, residual, y, ids, w, h);
}

}  // namespace obs

extern "C" {

int obs_moe_decode(obs_ctx* ctx, const obs_moe_config* cfg, const obs_moe_layer* layer, const uint16_t* x,
                   const uint16_t* residual, uint16_t* y, int32_t* ids_out, float* w_out) {
  if (!ctx) return OBS_E_INVALID;
  bool fused = false;
  int rc = obs::decode_plan(ctx, "obs_moe_decode", cfg, layer, x, y, &fused);
  if (rc) return rc;
  if (fused) return obs::launch_fused_decode(ctx, cfg, layer, x, residual, y, ids_out, w_out);
  void* ws = nullptr;
  rc = obs::ensure_decode_ws(ctx, obs::multi_ws_bytes(cfg), &ws);
  if (rc) return rc;
  return obs::decode_multi(ctx, cfg, layer, x, residual, y, ids_out, w_out, static_cast<char*>(ws));
}

int obs_moe_decode_static(obs_ctx* ctx, const obs_moe_config* cfg, const obs_moe_layer* layer, const uint16_t* x,
                          const uint16_t* residual, uint16_t* y, int32_t* ids_out, float* w_out) {
  if (!ctx) return OBS_E_INVALID;
  bool fused = false;
  int rc = obs::decode_plan(ctx, "obs_moe_decode_static", cfg, layer, x, y, &fused);
  if (rc) return rc;
  if (!ctx->scratch)
    return obs::set_error(ctx, OBS_E_UNSUPPORTED, "obs_moe_decode_static: no static scratch on device %d",
                          ctx->device);
  const size_t need = obs::multi_ws_bytes(cfg);
  if (need > obs::STATIC_MULTI_BYTES)
    return obs::set_error(ctx, OBS_E_NOMEM,
                          "obs_moe_decode_static: the shape needs %zu bytes of scratch, the static array holds %zu",
                          need, obs::STATIC_MULTI_BYTES);
  ctx->scratch_used = true;
  char* base = static_cast<char*>(ctx->scratch);
  if (fused) return obs::launch_fused_decode_ws(ctx, cfg, layer, x, residual, y, ids_out, w_out, base);
  return obs::decode_multi(ctx, cfg, layer, x, residual, y, ids_out, w_out, base + obs::STATIC_FUSED_BYTES);
}

int obs_set_decode_path(obs_ctx* ctx, int path) {
  if (!ctx) return OBS_E_INVALID;
  if (path != OBS_DECODE_AUTO && path != OBS_DECODE_MULTI && path != OBS_DECODE_FUSED)
    return obs::set_error(ctx, OBS_E_INVALID, "obs_set_decode_path: unknown path %d", path);
  ctx->decode_path = path;
  return OBS_OK;
}

int obs_device_status(obs_ctx* ctx) {
  if (!ctx) return OBS_E_INVALID;
  const int a = obs::fused_decode_status(ctx);
  const int b = obs::attn_fused_status(ctx);
  const int c = ctx->scratch_used ? obs::fused_decode_status_ws(ctx, ctx->scratch) : OBS_OK;
  const int f = obs::ffn_status(ctx);
  const int l = obs::layer_fused_status(ctx);
  return a != OBS_OK ? a : b != OBS_OK ? b : c != OBS_OK ? c : f != OBS_OK ? f : l;
}

}  // extern "C"
