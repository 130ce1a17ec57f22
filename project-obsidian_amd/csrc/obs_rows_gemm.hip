// obs_rows_gemm.hip — the dense 4-bit GEMM (obs_q4_matmul, Model::matmul_raw,
// forward.rs:313-321) below the size where the 128-row tiles of obs_prefill.hip
// fill the CUs twice over: the kernels here split a tile's K over the waves of a
// workgroup, so that a launch has more waves and each a shorter chain of
// dependent groups, and their tiles come in several sizes, so that one fills the
// CUs about once.
//
// Dequantization and accumulation are those of the grouped GEMM (bf16 =
// RNE(fp32(q s + b)), fp32 MFMA); the partial sums of the waves meet in LDS and
// are added in wave order in fp32, then rounded once. Every operand comes
// through a buffer resource: a 32-bit lane offset and a scalar one instead of a
// 64-bit address per load, which is what lets two workgroups share a CU
// (88-128 registers; with per-load addresses the 64-row form took 210), and
// activation rows at or past T read as zeros.
#include "obs_q4_dequant.hpp"

namespace {

using namespace obsd;

constexpr uint32_t GK = 64;          // quantization group
constexpr uint32_t LDS_STRIDE = 72;  // bf16 per staged activation row (64 + 8 padding)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
__device__ __forceinline__ u32x4_t load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ uint2 load8(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}

typedef float f32x4v __attribute__((ext_vector_type(4)));

// Four groups' scales and biases of one weight row as packed (s | b << 16) words.
__device__ __forceinline__ bool unpack_scales(uint2 sv, uint2 bv, uint32_t (&sb)[4]) {
  sb[0] = (sv.x & 0xffffu) | (bv.x << 16);
  sb[1] = (sv.x >> 16) | (bv.x & 0xffff0000u);
  sb[2] = (sv.y & 0xffffu) | (bv.y << 16);
  sb[3] = (sv.y >> 16) | (bv.y & 0xffff0000u);
  return scale_out_of_mix_range(sb[0]) || scale_out_of_mix_range(sb[1]) || scale_out_of_mix_range(sb[2]) ||
         scale_out_of_mix_range(sb[3]);
}

// Four rows (i0 .. i0 + 3 of the caller, one column) of the result as bf16: lanes
// c and c + 1 swap halves of their row pairs, so each store is a 4-byte column
// pair; the even lane writes rows i0 and i0 + 2, the odd lane i0 + 1 and i0 + 3.
__device__ __forceinline__ void store_quad(uint16_t* out, f32x4v c, uint32_t i0, uint32_t col, uint32_t T, uint32_t N) {
  const uint32_t odd = col & 1u, sel = odd ? 0x03020706u : 0x05040100u;
  const uint32_t p01 = pack_bf16_rne(c.x, c.y), p23 = pack_bf16_rne(c.z, c.w);
  const uint32_t s01 = static_cast<uint32_t>(dpp_i32<DPP_XOR1>(static_cast<int>(p01)));
  const uint32_t s23 = static_cast<uint32_t>(dpp_i32<DPP_XOR1>(static_cast<int>(p23)));
  const uint32_t i = i0 + odd;
  uint16_t* o = out + static_cast<size_t>(i) * N + (col & ~1u);
  if (i < T) *reinterpret_cast<uint32_t*>(o) = __builtin_amdgcn_perm(s01, p01, sel);
  if (i + 2u < T) *reinterpret_cast<uint32_t*>(o + 2u * static_cast<size_t>(N)) = __builtin_amdgcn_perm(s23, p23, sel);
}

// A workgroup's item: an XCD (b % 8) runs a contiguous run of column blocks with
// all their row tiles, so a weight row is read into one L2.
__device__ __forceinline__ bool item_of(uint32_t tiles, uint32_t ncb, uint32_t* tile, uint32_t* cb) {
  const uint32_t items = tiles * ncb, chunk = (items + 7u) / 8u;
  const uint32_t item = (blockIdx.x % 8u) * chunk + blockIdx.x / 8u;
  if (blockIdx.x / 8u >= chunk || item >= items) return false;
  *tile = item % tiles;
  *cb = item / tiles;
  return true;
}

// 32 MB rows x 32 columns, K over 8 waves. Wave w takes the 256-column units w,
// w + 8, ... A unit is 128 bytes of each weight row: its 4 groups' nibbles,
// scales and biases are loaded at once, straight to registers; the activations
// come a group at a time through a wave-private LDS slice (coalesced rows in,
// MFMA fragments out, the next group's loads in flight), so the loop has no
// barrier. 160 workgroups at N = 5,120 where 128-column tiles give 40.
constexpr uint32_t KW = 8;

template <uint32_t MB>
__global__ void __launch_bounds__(64 * KW, 4)
    q4_rows_gemm_kernel(const uint16_t* __restrict__ A, const uint32_t* __restrict__ w, const uint16_t* __restrict__ s,
                        const uint16_t* __restrict__ b, uint16_t* __restrict__ out, uint32_t T, uint32_t K, uint32_t N) {
  constexpr uint32_t ROWS = 32u * MB, SLICE = ROWS * LDS_STRIDE;  // bf16 of a wave's staging slice
  constexpr uint32_t TILE4 = MB * 4u * 64u;                      // f32x4 of one partial tile
  constexpr uint32_t LDS_A = KW * SLICE * 2u, LDS_R = KW * TILE4 * 16u;
  __shared__ __attribute__((aligned(16))) unsigned char s_mem[LDS_A > LDS_R ? LDS_A : LDS_R];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, nl = lane & 31u, h = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: a unit's offsets stay in SGPRs
  uint32_t tile, cb;
  if (!item_of((T + ROWS - 1u) / ROWS, N / 32u, &tile, &cb)) return;
  const uint32_t row0 = tile * ROWS, n = cb * 32u + nl;
  const uint32_t groups = K / GK, units = groups / 4u;
  const auto rA = buffer_of(A, 2u * T * K), rW = buffer_of(w, N * (K / 2u));
  const auto rS = buffer_of(s, 2u * N * groups), rB = buffer_of(b, 2u * N * groups);
  // staging: lane l moves 16 bytes (chunk l % 8) of rows l / 8 + 8 i of the slice
  const uint32_t ao = 2u * ((row0 + lane / 8u) * K + 8u * (lane & 7u));
  const uint32_t wo = n * (K / 2u) + 16u * h, so = 2u * n * groups;
  uint16_t* const sa = reinterpret_cast<uint16_t*>(s_mem) + wave * SLICE;
  f32x16_t acc[MB];
#pragma unroll
  for (uint32_t mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[mb][v] = 0.0f;

  for (uint32_t u = wave; u < units; u += KW) {  // uniform per wave
    u32x4_t q[4], ra[4u * MB];
#pragma unroll
    for (uint32_t g = 0; g < 4; ++g) q[g] = load16(rW, wo, 128u * u + 32u * g);
    const uint2 sv = load8(rS, so, 8u * u), bv = load8(rB, so, 8u * u);
    auto load_a = [&](uint32_t g) __attribute__((always_inline)) {
#pragma unroll
      for (uint32_t i = 0; i < 4u * MB; ++i) ra[i] = load16(rA, ao + 16u * i * K, 512u * u + 128u * g);
    };
    // a wave's LDS operations execute in order: the stores follow the reads of
    // the group before, and the reads of this group follow the stores
    auto stage = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (uint32_t i = 0; i < 4u * MB; ++i)
        *reinterpret_cast<u32x4_t*>(sa + (lane / 8u + 8u * i) * LDS_STRIDE + 8u * (lane & 7u)) = ra[i];
    };
    auto mma = [&](uint32_t st, bf16x8_t f) __attribute__((always_inline)) {
#pragma unroll
      for (uint32_t mb = 0; mb < MB; ++mb) {
        const bf16x8_t af = *reinterpret_cast<const bf16x8_t*>(sa + (32u * mb + nl) * LDS_STRIDE + 32u * h + 8u * st);
        acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, f, acc[mb], 0, 0, 0);
      }
    };
    load_a(0);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t sb[4];
    if (__any(unpack_scales(sv, bv, sb))) {  // scales beyond 2^100 (never in real checkpoints): reference-form dequant
#pragma unroll 1
      for (uint32_t g = 0; g < 4; ++g) {
        load_a(g);
        stage();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll 1
        for (uint32_t st = 0; st < 4; ++st)
          mma(st, dequant_word(w[static_cast<size_t>(n) * (K / 8u) + 8u * (4u * u + g) + 4u * h + st],
                               bf16_to_f32(s[static_cast<size_t>(n) * groups + 4u * u + g]),
                               bf16_to_f32(b[static_cast<size_t>(n) * groups + 4u * u + g])));
      }
      continue;
    }
#pragma unroll
    for (uint32_t g = 0; g < 4; ++g) {
      stage();
      if (g + 1u < 4u) load_a(g + 1u);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      const MixScale m = mix_scale(sb[g]);
#pragma unroll
      for (uint32_t st = 0; st < 4; ++st) {
        __builtin_amdgcn_sched_barrier(0);  // one K-step's fragments live at a time
        mma(st, dequant_word_mix(q[g][st], m));
      }
    }
  }

  // partial tiles: f32x4 (rows 8 v4 + 4 h + 0..3 of a 32-row block, column nl)
  // at [wave][mb][v4][lane]; wave w then adds entries w, w + 8, ...
  __syncthreads();
  f32x4v* const red = reinterpret_cast<f32x4v*>(s_mem);
#pragma unroll
  for (uint32_t mb = 0; mb < MB; ++mb)
#pragma unroll
    for (uint32_t v4 = 0; v4 < 4; ++v4)
      red[wave * TILE4 + (mb * 4u + v4) * 64u + lane] =
          f32x4v{acc[mb][4 * v4], acc[mb][4 * v4 + 1], acc[mb][4 * v4 + 2], acc[mb][4 * v4 + 3]};
  __syncthreads();
  for (uint32_t e = wave; e < TILE4 / 64u; e += KW) {  // uniform per wave: (mb, v4)
    f32x4v c = red[e * 64u + lane];
#pragma unroll
    for (uint32_t k = 1; k < KW; ++k) c += red[k * TILE4 + e * 64u + lane];
    store_quad(out, c, row0 + 8u * e + 4u * h, n, T, N);
  }
}

// 64 rows x 128 columns, K over two sets of 4 waves (wave wn of a set owns 32
// columns). A set stages its half of the activations' groups in LDS once for its
// 4 waves, double-buffered, activations and nibbles two groups ahead in
// registers; the two sets meet at each group's barrier. Where the 32-column
// tiles above re-read the activations too often (each row once per 32 columns).
constexpr uint32_t NB = 2, KS = 2;

__global__ void __launch_bounds__(256 * KS, 4)
    q4_ksplit_gemm_kernel(const uint16_t* __restrict__ A, const uint32_t* __restrict__ w, const uint16_t* __restrict__ s,
                          const uint16_t* __restrict__ b, uint16_t* __restrict__ out, uint32_t T, uint32_t K,
                          uint32_t N) {
  constexpr uint32_t ROWS = 32u * NB, COLS = 128u, BUF = ROWS * LDS_STRIDE;  // bf16 of a set's activation buffer
  constexpr uint32_t PV = NB * 4u / KS;  // row quads (f32x4 per lane) of the tile that a set adds up and stores
  constexpr uint32_t LDS_A = KS * 2u * BUF * 2u, LDS_R = KS * PV * 256u * 16u;
  __shared__ __attribute__((aligned(16))) unsigned char s_mem[LDS_A > LDS_R ? LDS_A : LDS_R];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, st_id = tid & 255u, wn = st_id >> 6;
  const uint32_t set = __builtin_amdgcn_readfirstlane(tid >> 8), nl = lane & 31u, h = lane >> 5;
  uint32_t tile, cb;
  if (!item_of((T + ROWS - 1u) / ROWS, N / COLS, &tile, &cb)) return;
  const uint32_t row0 = tile * ROWS, n = cb * COLS + 32u * wn + nl;
  const uint32_t groups = K / GK, ng = groups / KS, g0 = set * ng;  // the set's groups [g0, g0 + ng), ng % 4 == 0
  const auto rA = buffer_of(A, 2u * T * K), rW = buffer_of(w, N * (K / 2u));
  const auto rS = buffer_of(s, 2u * N * groups), rB = buffer_of(b, 2u * N * groups);
  const uint32_t ao = 2u * ((row0 + st_id / 8u) * K + 8u * (st_id & 7u));
  const uint32_t wo = n * (K / 2u) + 16u * h, so = 2u * n * groups;
  uint16_t* const sa = reinterpret_cast<uint16_t*>(s_mem) + set * 2u * BUF;
  // (past the set's last group its last one is loaded again, never used)
  auto load_w = [&](uint32_t g) __attribute__((always_inline)) { return load16(rW, wo, 32u * (g0 + min(g, ng - 1u))); };
  auto load_a = [&](uint32_t g, u32x4_t (&r)[NB]) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < NB; ++i) r[i] = load16(rA, ao + 64u * i * K, 128u * (g0 + min(g, ng - 1u)));
  };
  auto store_a = [&](uint32_t buf, const u32x4_t (&r)[NB]) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < NB; ++i)
      *reinterpret_cast<u32x4_t*>(sa + buf * BUF + (st_id / 8u + 32u * i) * LDS_STRIDE + 8u * (st_id & 7u)) = r[i];
  };
  f32x16_t acc[NB];
#pragma unroll
  for (uint32_t mb = 0; mb < NB; ++mb)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[mb][v] = 0.0f;

  u32x4_t ra[2][NB], q[4];
  uint2 sv = load8(rS, so, 2u * g0), bv = load8(rB, so, 2u * g0);
  q[0] = load_w(0);
  q[1] = load_w(1);
  load_a(0, ra[0]);
  load_a(1, ra[1]);
  __builtin_amdgcn_sched_barrier(0);
  store_a(0, ra[0]);
  for (uint32_t u = 0; u < ng; u += 4) {
    uint32_t sb[4];
    const bool wide = __any(unpack_scales(sv, bv, sb));  // uniform per wave
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t g = u + j, buf = j & 1u;
      __syncthreads();                       // group g staged in buffer `buf`; the other buffer is free
      store_a(buf ^ 1u, ra[(j + 1u) & 1u]);  // group g + 1, loaded a group ago
      load_a(g + 2u, ra[j & 1u]);
      q[(j + 2u) & 3u] = load_w(g + 2u);
      if (j == 1u) {
        const uint32_t gn = 2u * (g0 + min(u + 4u, ng - 4u));
        sv = load8(rS, so, gn);
        bv = load8(rB, so, gn);
      }
      __builtin_amdgcn_sched_barrier(0);
      auto mma = [&](uint32_t st, bf16x8_t f) __attribute__((always_inline)) {
        bf16x8_t af[NB];
#pragma unroll
        for (uint32_t mb = 0; mb < NB; ++mb)
          af[mb] = *reinterpret_cast<const bf16x8_t*>(sa + buf * BUF + (32u * mb + nl) * LDS_STRIDE + 32u * h + 8u * st);
#pragma unroll
        for (uint32_t mb = 0; mb < NB; ++mb) acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[mb], f, acc[mb], 0, 0, 0);
      };
      if (!wide) {
        const MixScale m = mix_scale(sb[j]);
#pragma unroll
        for (uint32_t st = 0; st < 4; ++st) mma(st, dequant_word_mix(q[j][st], m));
      } else {  // scales beyond 2^100 (never in real checkpoints): reference-form dequant
#pragma unroll 1
        for (uint32_t st = 0; st < 4; ++st)
          mma(st, dequant_word(st < 2u ? (st == 0u ? q[j].x : q[j].y) : (st == 2u ? q[j].z : q[j].w), bf16lo(sb[j]),
                               bf16hi(sb[j])));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // Part p of the tile's row quads (quad 4 mb + v4: rows 32 mb + 8 v4 + 4 h + 0..3,
  // one f32x4 per lane) belongs to set p: the other set hands its sums over
  // through LDS and the owner adds them, set 0's first.
  f32x4v* const red = reinterpret_cast<f32x4v*>(s_mem);
  auto quad = [&](uint32_t qi) __attribute__((always_inline)) {
    const uint32_t mb = qi / 4u, v = 4u * (qi % 4u);
    return f32x4v{acc[mb][v], acc[mb][v + 1u], acc[mb][v + 2u], acc[mb][v + 3u]};
  };
  __syncthreads();
#pragma unroll
  for (uint32_t p = 0; p < KS; ++p)
    if (p != set)  // uniform per wave
#pragma unroll
      for (uint32_t i = 0; i < PV; ++i) red[(p * PV + i) * 256u + st_id] = quad(p * PV + i);
  __syncthreads();
#pragma unroll
  for (uint32_t p = 0; p < KS; ++p)
    if (p == set)
#pragma unroll
      for (uint32_t i = 0; i < PV; ++i) {
        const f32x4v mine = quad(p * PV + i), other = red[(p * PV + i) * 256u + st_id];
        store_quad(out, p == 0u ? mine + other : other + mine, row0 + 8u * (p * PV + i) + 4u * h, n, T, N);
      }
}

// 32 NB rows x 128 (TWO: 256) columns, K over two sets of 4 waves, one workgroup
// per CU: for sizes whose tiles fill the CUs at most once. A wave owns 32 columns
// (TWO: of both halves) and all rows, so a dequantized weight fragment feeds NB
// products and an activation fragment feeds both halves; a set stages its
// activations in LDS as above. Against 128 x 128 and 128 x 256 tiles of one set
// of waves (obs_prefill.hip) a CU has two waves per SIMD where those had one, and
// 96 and 160 rows fit sizes that 128 rows leave with a nearly empty second
// round. What bounds it: the chain of a group (barrier, LDS reads, dequantization,
// products), 1.7 us for two groups of 128 x 256 at 52% of the matrix rate; with
// the staging left out it was 1.4, without the dequantization 1.5. Staged one
// group ahead instead of two: 3-5% slower; the next step's weights dequantized
// between a step's products, or a higher priority for one set: no faster.
// Measured, us, the 128-row tiles of obs_prefill.hip against the form taken:
//   N = 5,120 of K = 2,048: 500 rows 24.7 -> 18.3 (96 x 128), 700 27.8 -> 22.3
//   (128 x 128), 1,000 36.5 -> 29.6 (96 x 256), 1,300 38.0 -> 35.6 (128 x 256),
//   1,900 57.7 -> 45.3 (160 x 256);
//   N = 2,048 of K = 4,096: 1,300 47.4 -> 33, 1,900 47.2 -> 40.6, 2,500 63.2 -> 55.5.
template <uint32_t NB, bool TWO>
__global__ void __launch_bounds__(256 * KS, 2)
    q4_tile_gemm_kernel(const uint16_t* __restrict__ A, const uint32_t* __restrict__ w, const uint16_t* __restrict__ s,
                        const uint16_t* __restrict__ b, uint16_t* __restrict__ out, uint32_t T, uint32_t K, uint32_t N) {
  constexpr uint32_t ROWS = 32u * NB, CS = TWO ? 2u : 1u, COLS = 128u * CS, BUF = ROWS * LDS_STRIDE;
  static_assert(KS * 2u * BUF * 2u >= NB * 4u * 256u * 16u, "a column set's sums fit the activation buffers");
  extern __shared__ __attribute__((aligned(16))) unsigned char s_dyn[];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, st_id = tid & 255u, wn = st_id >> 6;
  const uint32_t set = __builtin_amdgcn_readfirstlane(tid >> 8), nl = lane & 31u, h = lane >> 5;
  uint32_t tile, cb;
  if (!item_of((T + ROWS - 1u) / ROWS, N / COLS, &tile, &cb)) return;
  const uint32_t row0 = tile * ROWS, n = cb * COLS + 32u * wn + nl;  // second column set: n + 128
  const uint32_t groups = K / GK, ng = groups / KS, g0 = set * ng;   // the set's groups [g0, g0 + ng), ng % 4 == 0
  const auto rA = buffer_of(A, 2u * T * K), rW = buffer_of(w, N * (K / 2u));
  const auto rS = buffer_of(s, 2u * N * groups), rB = buffer_of(b, 2u * N * groups);
  const uint32_t ao = 2u * ((row0 + st_id / 8u) * K + 8u * (st_id & 7u));
  const uint32_t wo = n * (K / 2u) + 16u * h, so = 2u * n * groups;
  const uint32_t w2 = 128u * (K / 2u), s2 = 256u * groups;  // from the first column set to the second
  uint16_t* const sa = reinterpret_cast<uint16_t*>(s_dyn) + set * 2u * BUF;
  // (past the set's last group its last one is loaded again, never used)
  auto load_w = [&](uint32_t g, u32x4_t (&r)[CS]) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t c = 0; c < CS; ++c) r[c] = load16(rW, wo, 32u * (g0 + min(g, ng - 1u)) + c * w2);
  };
  auto load_a = [&](uint32_t g, u32x4_t (&r)[NB]) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < NB; ++i) r[i] = load16(rA, ao + 64u * i * K, 128u * (g0 + min(g, ng - 1u)));
  };
  auto store_a = [&](uint32_t buf, const u32x4_t (&r)[NB]) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < NB; ++i)
      *reinterpret_cast<u32x4_t*>(sa + buf * BUF + (st_id / 8u + 32u * i) * LDS_STRIDE + 8u * (st_id & 7u)) = r[i];
  };
  f32x16_t acc[CS][NB];
#pragma unroll
  for (uint32_t c = 0; c < CS; ++c)
#pragma unroll
    for (uint32_t mb = 0; mb < NB; ++mb)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[c][mb][v] = 0.0f;

  u32x4_t ra[2][NB], q[2][CS];
  uint2 sv[CS], bv[CS];
  auto load_s = [&](uint32_t u) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t c = 0; c < CS; ++c) {
      const uint32_t at = 2u * (g0 + min(u, ng - 4u)) + c * s2;
      sv[c] = load8(rS, so, at);
      bv[c] = load8(rB, so, at);
    }
  };
  load_a(0, ra[0]);
  load_a(1, ra[1]);
  load_s(0);
  load_w(0, q[0]);
  load_w(1, q[1]);
  __builtin_amdgcn_sched_barrier(0);
  store_a(0, ra[0]);
  // one K-step: the activation fragments are requested first, the weights
  // dequantized while they arrive (left alone, each read sank to its product)
  auto k_step = [&](uint32_t buf, uint32_t st, auto dequant) __attribute__((always_inline)) {
    bf16x8_t af[NB], f[CS];
#pragma unroll
    for (uint32_t mb = 0; mb < NB; ++mb)
      af[mb] = *reinterpret_cast<const bf16x8_t*>(sa + buf * BUF + (32u * mb + nl) * LDS_STRIDE + 32u * h + 8u * st);
    __builtin_amdgcn_sched_barrier(0xE);  // VALU, SALU and MFMA may cross, memory may not
#pragma unroll
    for (uint32_t c = 0; c < CS; ++c) f[c] = dequant(c);
#pragma unroll
    for (uint32_t mb = 0; mb < NB; ++mb)
#pragma unroll
      for (uint32_t c = 0; c < CS; ++c)
        acc[c][mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[mb], f[c], acc[c][mb], 0, 0, 0);
  };
  bool big = false;  // some scale of the lane's is beyond dequant_word_mix's range
  for (uint32_t u = 0; u < ng; u += 4) {
    uint32_t sb[CS][4];
#pragma unroll
    for (uint32_t c = 0; c < CS; ++c) big = unpack_scales(sv[c], bv[c], sb[c]) || big;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t g = u + j, buf = j & 1u;
      __syncthreads();  // group g staged in buffer `buf`; the other buffer is free
      store_a(buf ^ 1u, ra[(j + 1u) & 1u]);
      load_a(g + 2u, ra[j & 1u]);
      __builtin_amdgcn_sched_barrier(0);  // first: they are waited for first
      u32x4_t qn[CS];
      load_w(g + 2u, qn);
      if (j == 1u) load_s(u + 4u);
      __builtin_amdgcn_sched_barrier(0);
      MixScale m[CS];
#pragma unroll
      for (uint32_t c = 0; c < CS; ++c) m[c] = mix_scale(sb[c][j]);
#pragma unroll
      for (uint32_t st = 0; st < 4; ++st)
        k_step(buf, st, [&](uint32_t c) __attribute__((always_inline)) { return dequant_word_mix(q[j & 1u][c][st], m[c]); });
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t c = 0; c < CS; ++c) q[j & 1u][c] = qn[c];
    }
  }

  // A scale beyond 2^100 (never in real checkpoints): the tile again from the
  // start with the reference-form dequant, a group at a time.
  if (__syncthreads_or(big)) {
#pragma unroll
    for (uint32_t c = 0; c < CS; ++c)
#pragma unroll
      for (uint32_t mb = 0; mb < NB; ++mb)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[c][mb][v] = 0.0f;
#pragma unroll 1
    for (uint32_t g = 0; g < ng; ++g) {
      load_a(g, ra[0]);
      __syncthreads();  // the group before is read
      store_a(0, ra[0]);
      __syncthreads();
#pragma unroll 1
      for (uint32_t st = 0; st < 4; ++st)
        k_step(0, st, [&](uint32_t c) __attribute__((always_inline)) {
          const size_t row = n + 128u * c, at = row * groups + g0 + g;
          return dequant_word(w[row * (K / 8u) + 8u * (g0 + g) + 4u * h + st], bf16_to_f32(s[at]), bf16_to_f32(b[at]));
        });
    }
  }

  // As in q4_ksplit_gemm_kernel, one column set at a time: half of its row quads
  // (quad 4 mb + v4: rows 32 mb + 8 v4 + 4 h + 0..3) belongs to each set of waves;
  // the other hands its sums over through LDS and the owner adds them, set 0's first.
  constexpr uint32_t PV = NB * 4u / KS;
  f32x4v* const red = reinterpret_cast<f32x4v*>(s_dyn);
#pragma unroll
  for (uint32_t c = 0; c < CS; ++c) {
    auto quad = [&](uint32_t qi) __attribute__((always_inline)) {
      const uint32_t mb = qi / 4u, v = 4u * (qi % 4u);
      return f32x4v{acc[c][mb][v], acc[c][mb][v + 1u], acc[c][mb][v + 2u], acc[c][mb][v + 3u]};
    };
    __syncthreads();
#pragma unroll
    for (uint32_t p = 0; p < KS; ++p)
      if (p != set)  // uniform per wave
#pragma unroll
        for (uint32_t i = 0; i < PV; ++i) red[(p * PV + i) * 256u + st_id] = quad(p * PV + i);
    __syncthreads();
#pragma unroll
    for (uint32_t p = 0; p < KS; ++p)
      if (p == set)
#pragma unroll
        for (uint32_t i = 0; i < PV; ++i) {
          const f32x4v mine = quad(p * PV + i), other = red[(p * PV + i) * 256u + st_id];
          store_quad(out, p == 0u ? mine + other : other + mine, row0 + 8u * (p * PV + i) + 4u * h, n + 128u * c, T, N);
        }
  }
}

struct TileForm {
  obs::RowsGemm which;
  uint32_t rows, cols, lds;
  double base, slope;  // its cost (q4_rows_gemm_pick)
  const void* fn;
};
template <uint32_t NB, bool TWO>
TileForm tile_form(obs::RowsGemm which, double base, double slope) {
  return TileForm{which, 32u * NB, TWO ? 256u : 128u, KS * 2u * 32u * NB * LDS_STRIDE * 2u, base, slope,
                  reinterpret_cast<const void*>(&q4_tile_gemm_kernel<NB, TWO>)};
}
const TileForm TILE_FORMS[] = {
    tile_form<3, false>(obs::RowsGemm::T96, 10.0, 3.5), tile_form<4, false>(obs::RowsGemm::T128, 11.5, 6.3),
    tile_form<3, true>(obs::RowsGemm::T96W, 18.0, 8.0), tile_form<4, true>(obs::RowsGemm::T128W, 23.0, 7.5),
    tile_form<5, true>(obs::RowsGemm::T160W, 29.0, 11.0)};

}  // namespace

namespace obs {

// Which kernel an obs_q4_matmul of T rows takes: the one with the least time by
// measured costs (us, MI355X, k = K / 2048 scaling what a workgroup does). One
// workgroup per CU runs at its own speed, more share the CU:
//   32 rows x 32 columns: 2.5 + 2.9 k, beyond a workgroup per CU 2.5 + (2.2 + 0.0093 n) k
//   64 x 32:              2.5 + 4.2 k, 2.5 + (4.2 + 0.012 n) k
//   (both: + 1.2 per MB of activations beyond one XCD's 4 MB L2, which every
//   XCD then reads past its L2: 2,048 rows x 512 columns 21.1, K in two 14.2)
//   64 x 128, K in two:   2.5 + max(10.6, 0.055 n) k
//   96 x 128, 128 x 128, 96 x 256, 128 x 256, 160 x 256, K in two, at most one
//   workgroup per CU (f = workgroups per CU): 5 + (10 + 3.5 f, 11.5 + 6.3 f,
//   18 + 8 f, 23 + 7.5 f, 29 + 11 f) k
//   128-row tiles (obs_prefill.hip): 2.5 + (9.8, 12.8, 17 or 20.9 by the row
//   blocks of its largest tile) k, beyond a workgroup per CU 2.5 + (24 + 0.026 n) k;
//   once 128 x 256 tiles fill the CUs, those: 2.5 + 35 k at one per CU, then
//   2.5 + (43 + 0.043 n) k; from two of them per CU on always these.
// Measured, 128 rows against the kernel taken, N = 5,120 of K = 2,048 and
// N = 2,048 of K = 4,096: 24 rows 12.5 -> 5.4 and 21.4 -> 7.5; 64: 15.3 -> 6.7
// and 27.1 -> 8.1; 200: 23.5 -> 13.2 and 42.3 -> 11.2; more rows above.
RowsGemm q4_rows_gemm_pick(uint32_t T, uint32_t K, uint32_t N, uint32_t cus) {
  const uint64_t tiles128 = (T + 127u) / 128u, n128 = tiles128 * (N / 128u);
  const uint64_t n256 = N % 256u == 0 ? tiles128 * (N / 256u) : 0u;  // 128 x 256 tiles, taken once they fill the CUs
  if (T == 0 || (n256 >= cus ? n256 : n128) >= 2u * cus || (static_cast<uint64_t>(T) + 192u) * K * 2u >= (1ull << 32) ||
      static_cast<uint64_t>(N) * (K / 2u) >= (1ull << 32))
    return RowsGemm::NONE;
  const double k = K / 2048.0, c = cus / 256.0;  // the slopes are per 256 CUs
  const uint32_t nb = T > 96u ? 4u : (T + 31u) / 32u;
  const double one[5] = {0.0, 9.8, 12.8, 17.0, 20.9};
  const double n32 = static_cast<double>((T + 31u) / 32u) * (N / 32u), n64 = static_cast<double>((T + 63u) / 64u) * (N / 32u);
  const double nks = static_cast<double>((T + 63u) / 64u) * (N / 128u);
  double best = (n256 > cus ? 43.0 + 0.043 * static_cast<double>(n256) / c : n256 == cus ? 35.0
                 : n128 <= cus ? one[nb] : 24.0 + 0.026 * static_cast<double>(n128) / c) * k;
  RowsGemm pick = RowsGemm::NONE;
  auto offer = [&](double cost, RowsGemm which) {
    if (cost < best) {
      best = cost;
      pick = which;
    }
  };
  const double past = static_cast<double>(T) * K * 2.0 / 1048576.0 - 4.0, spill = past > 0.0 ? 1.2 * past : 0.0;
  offer(spill + (n32 <= cus ? 2.9 : 2.2 + 0.0093 * n32 / c) * k, RowsGemm::R32);
  offer(spill + (n64 <= cus ? 4.2 : 4.2 + 0.012 * n64 / c) * k, RowsGemm::R64);
  if (K % (KS * 4u * GK) == 0) {
    offer((0.055 * nks / c > 10.6 ? 0.055 * nks / c : 10.6) * k, RowsGemm::KSPLIT);
    for (const TileForm& f : TILE_FORMS) {
      const uint64_t n = static_cast<uint64_t>((T + f.rows - 1u) / f.rows) * (N / f.cols);
      if (N % f.cols == 0 && n <= cus) offer(2.5 + (f.base + f.slope * static_cast<double>(n) / cus) * k, f.which);
    }
  }
  return pick;
}

// The tile forms stage more than 64 KB of activations: their limit is raised
// once per context, at creation.
int rows_gemm_init(obs_ctx* ctx) {
  for (const TileForm& f : TILE_FORMS)
    OBS_HIP_TRY(ctx, hipFuncSetAttribute(f.fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(f.lds)));
  return OBS_OK;
}

int launch_q4_rows_gemm(obs_ctx* ctx, RowsGemm which, const uint32_t* w, const uint16_t* s, const uint16_t* b,
                        const uint16_t* X, uint16_t* Y, uint32_t T, uint32_t K, uint32_t N) {
  for (const TileForm& f : TILE_FORMS) {
    if (f.which != which) continue;
    const uint32_t grid = ((T + f.rows - 1u) / f.rows * (N / f.cols) + 7u) / 8u * 8u;
    void* args[] = {&X, &w, &s, &b, &Y, &T, &K, &N};
    OBS_LAUNCH(ctx, "q4_matmul",
               OBS_HIP_TRY(ctx, hipLaunchKernel(f.fn, dim3(grid), dim3(256 * KS), args, f.lds, ctx->stream)));
    return OBS_OK;
  }
  const uint32_t rows = which == RowsGemm::R32 ? 32u : 64u, cols = which == RowsGemm::KSPLIT ? 128u : 32u;
  const uint32_t grid = ((T + rows - 1u) / rows * (N / cols) + 7u) / 8u * 8u;  // every XCD the same number
  if (which == RowsGemm::R32)
    OBS_LAUNCH(ctx, "q4_matmul", (q4_rows_gemm_kernel<1><<<grid, 64 * KW, 0, ctx->stream>>>(X, w, s, b, Y, T, K, N)));
  else if (which == RowsGemm::R64)
    OBS_LAUNCH(ctx, "q4_matmul", (q4_rows_gemm_kernel<2><<<grid, 64 * KW, 0, ctx->stream>>>(X, w, s, b, Y, T, K, N)));
  else
    OBS_LAUNCH(ctx, "q4_matmul", (q4_ksplit_gemm_kernel<<<grid, 256 * KS, 0, ctx->stream>>>(X, w, s, b, Y, T, K, N)));
  return OBS_OK;
}

}  // namespace obs
