// tile_gemm.hip -- grouped expert GEMM on bf16 MFMA with MXFP4 weights dequantised in registers: the
// expert projections of every f32 batch, and of the bf16 batches too small for gemm.hip, but single
// tokens (the expert GEMV, kernels.hip).
//
// replaces w1_swiglu_dense_kernel / w2_scatter_dense_kernel (src/quant/gpu.rs:89-192) for those
// batches (the reference runs them per 256-token tile and per used expert, src/moe/mod.rs:262-404).
//
// Same operands and roundings as the expert GEMV: A = exact bf16 of code x scale,
// B = the activation row as NT bf16 terms (bf16 rows: themselves; f32 rows: hi + bf16 of the
// residual, or rounded once), f32 accumulation, v_mfma_f32_16x16x32_bf16.  K order: lane group q of
// a step s supplies K [32 q + 8 s, +8) of the 128-wide K-group for both operands, which is the
// tiled weight layout as stored (one dword of a lane's 16 bytes per step).
//
// Why tiles: GEMV passes hold 8 .. 14 token rows, so a batch re-streamed every expert's weights and
// re-staged whole rows per pass; a tile reads its weights once for 32 or 64 tokens while the rows
// pass through LDS K-group by K-group.  Up to ~100 tokens (20B shapes) the launch is bound by the
// weight stream: 17 tokens gate_up 54 -> 47 us (283 MB, 6.0 TB/s), down 30 -> 26 us.  Large f32 batches are
// bound by the matrix cores: 523 tokens 793 + 423 -> 182 + 117 us, 4096 tokens 918 + 483 us (1.16
// PFLOP/s of the two terms' products; plain bf16 MFMAs reach 1.8).  Weights are read nontemporally
// in the 16- and 32-token shapes only (gate_up 58 -> 50 us at 45 tokens: the router rows and token rows stay in
// the caches); the 64-token shape re-reads them from L2 for the next tiles.  At decode sizes the
// short items refill the CUs as they end, where the GEMV's fixed shares waited for the slowest: 8 tokens
// 38 + 22 -> 35 + 19 us with one layer's weights (over four layers in turn, which no cache holds, the step
// 75.5 -> 73.9 us), 16 tokens in f32 64 + 33 -> 52 + 27 us, D = F = 256 with 16 tokens 14 + 13 -> 7 + 7 us
// (every prefix and segment entry an item needs comes in one round trip, and waves whose token
// columns are all empty skip the split).
#include <type_traits>

#include "kernels.hpp"
#include "mx_device.hpp"

namespace burnext {

namespace {
typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));

constexpr uint32_t kWaves = 4;
// one term of one K-group in LDS: TOK token rows of 128 bf16
constexpr uint32_t term_bytes(uint32_t tok) { return tok * 256u; }
// padded row stride (floats) of the gate_up epilogue's staging: 32 RT features per token
constexpr uint32_t ep_stride(uint32_t rt) { return 32u * rt + 4u; }
constexpr uint32_t ring_bytes(int nt, uint32_t rt, uint32_t tok) {
  const uint32_t ring = 2u * (uint32_t)nt * term_bytes(tok), ep = tok * ep_stride(rt) * 4u;
  return ring > ep ? ring : ep;
}
constexpr int kLgkmcnt0 = 0xF | (7 << 4) | (3 << 14);

// Barrier of the double-buffered stage: a wave's LDS writes and reads are complete (lgkmcnt(0))
// before it arrives; its register loads stay in flight (__syncthreads() would drain them).
__device__ __forceinline__ void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(kLgkmcnt0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// One 8-value chunk of a B row on its way from global memory to LDS.
template <typename XT> struct BChunk;
template <> struct BChunk<float> {
  float4 a, b;
};
template <> struct BChunk<uint16_t> {
  uint4 a;
};
__device__ __forceinline__ void bchunk_load(BChunk<float> &c, const float *p) {
  c.a = *(const float4 *)p;
  c.b = *(const float4 *)(p + 4);
}
__device__ __forceinline__ void bchunk_load(BChunk<uint16_t> &c, const uint16_t *p) { c.a = *(const uint4 *)p; }
// values at K >= kt are zero (rows are padded with whatever the writer left there)
__device__ __forceinline__ void bchunk_mask(BChunk<float> &c, uint32_t nv) {
  float *v = (float *)&c;
#pragma unroll
  for (uint32_t j = 0; j < 8u; ++j) v[j] = j < nv ? v[j] : 0.0f;
}
__device__ __forceinline__ void bchunk_mask(BChunk<uint16_t> &c, uint32_t nv) {
  uint32_t *v = (uint32_t *)&c;
#pragma unroll
  for (uint32_t j = 0; j < 4u; ++j) v[j] = 2u * j + 1u < nv ? v[j] : 2u * j < nv ? v[j] & 0xFFFFu : 0u;
}
template <int NT>
__device__ __forceinline__ void bchunk_terms(const BChunk<float> &c, uint4 (&t)[NT]) {
  const float v[8] = {c.a.x, c.a.y, c.a.z, c.a.w, c.b.x, c.b.y, c.b.z, c.b.w};
  uint32_t w[4][NT];
#pragma unroll
  for (int j = 0; j < 4; ++j) split_bf16x2<NT>(v[2 * j], v[2 * j + 1], w[j]);
#pragma unroll
  for (int n = 0; n < NT; ++n) t[n] = make_uint4(w[0][n], w[1][n], w[2][n], w[3][n]);
}
template <int NT>
__device__ __forceinline__ void bchunk_terms(const BChunk<uint16_t> &c, uint4 (&t)[NT]) {
  t[0] = c.a;
}

// What a workgroup's item is.
struct Item {
  int e, seg0;
  uint32_t rb, m0, ntok;
  int32_t *rows_l;  // LDS [TOK]: B row of each token (columns beyond the tile: its first token's)
  int32_t *slot_l;  // LDS [TOK]: down's output slot
  const int32_t *perm_l;  // LDS (TOK 16): the batch's segment entries
  uint8_t *ring;    // LDS: [2 buffers][NT terms][TOK][256 bytes], and the epilogue's staging
};

template <uint32_t RT> struct ScaleRegs { typedef uint32_t type __attribute__((ext_vector_type(RT))); };

// The item's K-loop and epilogue for NTT = ceil(ntok / 16) token columns.
// Per K-group: the next K-group's B chunks go from registers to the other LDS buffer (split into
// terms on the way), the one after that is requested, then the MFMAs of this one, then its weight
// registers are refilled two K-groups ahead; one barrier.  LDS row of token t: 16 chunks of 16 bytes,
// chunk c in slot c ^ (t & 15): the operand reads (16 consecutive tokens, one chunk) and the writes
// (whole rows) are free of bank conflicts.
template <bool GATE_UP, typename XT, int NT, uint32_t RT, uint32_t TOK, int NTT>
__device__ __forceinline__ void tile_body(const TileArgs &a, const Item &it) {
  constexpr uint32_t kTermBytes = term_bytes(TOK), kRows = 16u * RT * kWaves;
  using SReg = typename ScaleRegs<RT>::type;
  // the segment entries (decode sizes: already in LDS) first: their round trip runs beside the first
  // weights'
  int32_t slot = 0;
  const uint32_t m_own = it.m0 + (threadIdx.x < it.ntok ? threadIdx.x : 0u);
  if (threadIdx.x < TOK) slot = TOK == 16u ? it.perm_l[it.seg0 + (int32_t)m_own] : a.perm[it.seg0 + (int32_t)m_own];
  const uint32_t lane = threadIdx.x & 63u, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t i16 = lane & 15u, q = lane >> 4;
  const uint32_t nkg = (a.nb + 3u) >> 2, tail = a.nb - 4u * (nkg - 1u), nkq = (nkg + 3u) >> 2, ngr = (a.nrt + 3u) >> 2;
  const uint8_t *wexp = a.wb + (size_t)it.e * a.wb_estride;
  const uint32_t rt0 = (it.rb * kWaves + wv) * RT;  // this wave's first row tile
  const uint8_t *arow[RT];
#pragma unroll
  for (uint32_t rt = 0; rt < RT; ++rt)  // rows beyond the expert are never stored
    arow[rt] = wexp + (size_t)min(rt0 + rt, a.nrt - 1u) * a.nb * 256u;
  // its row tiles' scale dwords in the GEMM's copy
  const uint8_t *srow = a.ws + (size_t)it.e * a.ws_estride + (size_t)min(rt0 >> 2, ngr - 1u) * nkq * 1024u + (rt0 & 3u) * 4u;
  // (the load counts of an iteration are the same on every path, so that the compiler's waits stay
  // partial: no branch around a load in the K-loop)
  auto load_a = [&](uint32_t kg, u32x4_t (&A)[RT]) {
    // lanes outside the last K-group's blocks read the row tile's first block: their B values are zero
    const uint32_t off = lane * 16u + ((kg + 1u == nkg && q >= tail) ? 0u : kg * 1024u);
#pragma unroll
    for (uint32_t rt = 0; rt < RT; ++rt)
      A[rt] = RT <= 2u ? __builtin_nontemporal_load((const u32x4_t *)(arow[rt] + off)) : *(const u32x4_t *)(arow[rt] + off);
  };
  // weights PA and B chunks PB K-groups ahead: few token columns leave registers for more
  constexpr uint32_t PA = NTT <= 2 ? 4u : 2u, PB = NTT == 1 ? 4u : NTT == 2 ? 2u : 1u;
  const uint32_t last = nkg - 1u;
  u32x4_t A[PA][RT];
  SReg sc = *(const SReg *)(srow + lane * 16u), sn = sc;
#pragma unroll
  for (uint32_t j = 0; j < PA; ++j) load_a(min(j, last), A[j]);
  if (threadIdx.x < TOK) {
    it.rows_l[threadIdx.x] = GATE_UP ? slot / (int32_t)a.topk : it.seg0 + (int32_t)m_own;
    it.slot_l[threadIdx.x] = slot;
  }
  stage_barrier();
  // B staging: thread -> chunk tid & 15 of tokens (tid >> 4) + 16 p
  const uint32_t ch = threadIdx.x & 15u, tk = threadIdx.x >> 4;
  const XT *brow[NTT];
#pragma unroll
  for (int p = 0; p < NTT; ++p)
    brow[p] = (const XT *)a.brows + (size_t)it.rows_l[tk + 16u * (uint32_t)p] * a.bstride;
  auto stage_load = [&](uint32_t kg, BChunk<XT> (&R)[NTT]) {
    const uint32_t k = kg * 128u + 8u * ch;
    const uint32_t off = k < a.bstride ? k : 0u;  // bstride is a multiple of 32
#pragma unroll
    for (int p = 0; p < NTT; ++p) bchunk_load(R[p], brow[p] + off);
  };
  // MASK: K-group kg may be the last (zeros from kt on)
  auto stage_store = [&](uint32_t kg, uint32_t buf, BChunk<XT> (&R)[NTT], auto MASK) {
    uint8_t *st = it.ring + buf * (NT * kTermBytes);
    const uint32_t k = kg * 128u + 8u * ch, nv = k < a.kt ? min(8u, a.kt - k) : 0u;
#pragma unroll
    for (int p = 0; p < NTT; ++p) {
      // (wave-uniform) columns beyond the tile keep what LDS holds: their results are never stored
      if (16u * (uint32_t)p + 4u * wv >= it.ntok) continue;
      if constexpr (decltype(MASK)::value) bchunk_mask(R[p], nv);
      const uint32_t t = tk + 16u * (uint32_t)p;
      uint4 terms[NT];
      bchunk_terms<NT>(R[p], terms);
#pragma unroll
      for (int n = 0; n < NT; ++n) *(uint4 *)(st + n * kTermBytes + t * 256u + ((ch ^ (t & 15u)) << 4)) = terms[n];
    }
  };

  f32x4_t acc[RT][NTT];  // starts at the expert's bias rows
#pragma unroll
  for (uint32_t rt = 0; rt < RT; ++rt) {
    const uint32_t r0 = it.rb * kRows + wv * 16u * RT + rt * 16u + 4u * q;
    const f32x4_t b4 = *(const f32x4_t *)(a.bias + (size_t)it.e * a.bias_estride + min(r0, a.bias_estride - 4u));
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt) acc[rt][tt] = b4;
  }

  BChunk<XT> R[PB][NTT];
  stage_load(0, R[0]);
  stage_store(0, 0, R[0], std::true_type{});
#pragma unroll
  for (uint32_t j = 1; j <= PB; ++j) stage_load(min(j, last), R[j % PB]);
  stage_barrier();
  const uint32_t boff = i16 * 256u + (((4u * q) ^ i16) << 4);
  // K-group kg at position P = kg mod 4 (of its scale block, and of the register sets)
  auto iter = [&](uint32_t kg, auto P, auto MASK) {
    constexpr uint32_t kp = decltype(P)::value;
    // (beyond the last K-group: a store that nothing reads)
    stage_store(min(kg + 1u, last), (kg + 1u) & 1u, R[(kp + 1u) % PB], MASK);
    stage_load(min(kg + 1u + PB, last), R[(kp + 1u) % PB]);
    if constexpr (kp == 1u) sn = *(const SReg *)(srow + (min((kg >> 2) + 1u, nkq - 1u) * 1024u + lane * 16u));
    const uint8_t *st = it.ring + (kg & 1u) * (NT * kTermBytes);
    float s[RT];
#pragma unroll
    for (uint32_t rt = 0; rt < RT; ++rt) s[rt] = e8m0_to_f32((sc[rt] >> (8u * kp)) & 255u);
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
      bf16x8_t Af[RT];
#pragma unroll
      for (uint32_t rt = 0; rt < RT; ++rt) Af[rt] = fp4x8_to_bf16x8(A[kp % PA][rt][k], s[rt]);
#pragma unroll
      for (int tt = 0; tt < NTT; ++tt)
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const bf16x8_t B = *(const bf16x8_t *)(st + n * kTermBytes + (uint32_t)tt * 4096u + (boff ^ (k << 4)));
#pragma unroll
          for (uint32_t rt = 0; rt < RT; ++rt)
            acc[rt][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Af[rt], B, acc[rt][tt], 0, 0, 0);
        }
    }
    // schedule: operand reads three ahead of the four MFMAs that use them
    __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);  // 0x100: LDS reads, 0x008: MFMAs
#pragma unroll
    for (int f = 0; f < 4 * NTT * NT - 3; ++f) {
      __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 12, 0);
    load_a(min(kg + PA, last), A[kp % PA]);
    if constexpr (kp == 3u) sc = sn;
    stage_barrier();
  };
  using P0 = std::integral_constant<uint32_t, 0>;
  using P1 = std::integral_constant<uint32_t, 1>;
  using P2 = std::integral_constant<uint32_t, 2>;
  using P3 = std::integral_constant<uint32_t, 3>;
  constexpr std::false_type full{};
  constexpr std::true_type mask{};
  uint32_t kg = 0;
  for (; kg + 5u < nkg; kg += 4u) {
    iter(kg, P0{}, full);
    iter(kg + 1u, P1{}, full);
    iter(kg + 2u, P2{}, full);
    iter(kg + 3u, P3{}, full);
  }
  // the last 1 .. 5 K-groups, nested so that no path joins another before the end
  iter(kg, P0{}, mask);
  if (kg + 1u < nkg) {
    iter(kg + 1u, P1{}, mask);
    if (kg + 2u < nkg) {
      iter(kg + 2u, P2{}, mask);
      if (kg + 3u < nkg) {
        iter(kg + 3u, P3{}, mask);
        if (kg + 4u < nkg) iter(kg + 4u, P0{}, mask);
      }
    }
  }

  if constexpr (GATE_UP) {
    // lane (q, j): rows 4 q .. 4 q + 3 of a tile are the (gate, linear) pairs of features 2 q and
    // 2 q + 1; the item's [token][32 RT features] leave through LDS as whole row segments
    constexpr uint32_t kS = ep_stride(RT), kC = 8u * RT;  // staging stride (floats), 16-byte chunks per token
    float *o_l = (float *)it.ring;
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt)
#pragma unroll
      for (uint32_t rt = 0; rt < RT; ++rt) {
        const f32x4_t v = acc[rt][tt];
        *(float2 *)(o_l + ((uint32_t)tt * 16u + i16) * kS + wv * 8u * RT + rt * 8u + 2u * q) =
            make_float2(swiglu_clamp_f(v[0], v[1], a.alpha, a.limit), swiglu_clamp_f(v[2], v[3], a.alpha, a.limit));
      }
    __syncthreads();
    for (uint32_t c = threadIdx.x; c < it.ntok * kC; c += blockDim.x) {
      const uint32_t tok = c / kC, cc = c % kC, f = it.rb * (kRows / 2u) + 4u * cc;
      if (f >= a.out_rows) continue;
      const float4 v = *(const float4 *)(o_l + tok * kS + 4u * cc);
      float *o = a.out + (size_t)(it.seg0 + (int32_t)(it.m0 + tok)) * a.out_stride + f;
      if (f + 4u <= a.out_rows) {
        *(float4 *)o = v;
      } else {
        const float vv[4] = {v.x, v.y, v.z, v.w};
        for (uint32_t j = 0; j < 4u; ++j)
          if (f + j < a.out_rows) o[j] = vv[j];
      }
    }
  } else {
    // token-major slot rows, b2 added once: 64 contiguous bytes per token and row tile
#pragma unroll
    for (int tt = 0; tt < NTT; ++tt) {
      const uint32_t tok = (uint32_t)tt * 16u + i16;
      if (tok >= it.ntok) continue;
      float *orow = a.out + (size_t)it.slot_l[tok] * a.out_stride;
#pragma unroll
      for (uint32_t rt = 0; rt < RT; ++rt) {
        const uint32_t r0 = it.rb * kRows + wv * 16u * RT + rt * 16u + 4u * q;
        const f32x4_t v = acc[rt][tt];
        if (r0 + 4u <= a.out_rows) {
          *(f32x4_t *)(orow + r0) = v;
        } else {
#pragma unroll
          for (uint32_t j = 0; j < 4u; ++j)
            if (r0 + j < a.out_rows) orow[r0 + j] = v[j];
        }
      }
    }
  }
}
}  // namespace

size_t tile_lds_bytes(int nt, const TileShape &t) {
  return ring_bytes(nt, t.row_tiles, t.tok) + 2 * t.tok * 4 + 64 + 2 * (kMaxExperts + 1) * 4 +
         (t.tok == 16u ? kSmallRouteMaxTokens * kMaxTopK * 4 : 0u);
}

// Work items (token tile of TOK routed tokens of one expert, block of 64 RT weight rows) in the
// grouped GEMM's order (gemm.hip): each XCD takes a contiguous run of the realised items, which go
// in groups of 8 token tiles, row block by row block, so that an XCD's L2 serves the weights of a
// group and its B rows repeatedly.
template <bool GATE_UP, typename XT, int NT, uint32_t RT, uint32_t TOK>
__global__ __launch_bounds__(256, RT <= 2 ? 4 : 2) void expert_tile_kernel(TileArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  int32_t *rows_l = (int32_t *)(smem + ring_bytes(NT, RT, TOK));
  int32_t *slot_l = rows_l + TOK, *info_l = slot_l + TOK, *toff_l = info_l + 16, *soff_l = toff_l + kMaxExperts + 1;
  // every prefix an item needs in one round trip; decode-sized batches (TOK 16) have one tile per
  // active expert, listed in `active`
  constexpr bool kOneTile = TOK == 16u;
  for (uint32_t t = threadIdx.x; t <= a.E; t += blockDim.x) {
    toff_l[t] = !kOneTile ? a.tile_off[t] : t < a.E ? a.active[t] : *a.num_active;
    soff_l[t] = a.seg_off[t];
  }
  int32_t *perm_l = soff_l + kMaxExperts + 1;
  if constexpr (kOneTile)
    for (uint32_t t = threadIdx.x; t < a.nperm; t += blockDim.x) perm_l[t] = a.perm[t];
  if (threadIdx.x == 0) info_l[0] = -1;
  __syncthreads();
  const uint32_t b = blockIdx.x, ntile = (uint32_t)toff_l[a.E], N = a.nrb * ntile, Q = (N + 7u) / 8u;
  const uint32_t item = (b & 7u) * Q + (b >> 3);
  if ((b >> 3) >= Q || item >= N) return;  // workgroup-uniform: no item
  uint32_t rb, gt;
  if constexpr (kOneTile) {
    gt = item / a.nrb;
    rb = item - gt * a.nrb;
  } else {
    const uint32_t grp = item / (8u * a.nrb), r = item - grp * 8u * a.nrb, gsz = min(8u, ntile - grp * 8u);
    rb = r / gsz;
    gt = grp * 8u + (r - rb * gsz);
    for (uint32_t e = threadIdx.x; e < a.E; e += blockDim.x)
      if (gt >= (uint32_t)toff_l[e] && gt < (uint32_t)toff_l[e + 1]) {
        info_l[0] = (int32_t)e;
        info_l[1] = (int32_t)(gt - (uint32_t)toff_l[e]);
      }
    __syncthreads();
  }
  Item it;
  it.e = __builtin_amdgcn_readfirstlane(kOneTile ? toff_l[gt] : info_l[0]);
  if (it.e < 0) return;  // workgroup-uniform
  it.seg0 = __builtin_amdgcn_readfirstlane(soff_l[it.e]);
  const uint32_t M = (uint32_t)(__builtin_amdgcn_readfirstlane(soff_l[it.e + 1]) - it.seg0);
  it.rb = rb;
  it.m0 = kOneTile ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane(info_l[1]) * TOK;
  it.ntok = min(TOK, M - it.m0);
  it.rows_l = rows_l;
  it.slot_l = slot_l;
  it.perm_l = perm_l;
  it.ring = smem;
  const uint32_t c16 = (it.ntok + 15u) / 16u;
  if (TOK == 16u || c16 == 1u) return tile_body<GATE_UP, XT, NT, RT, TOK, 1>(a, it);
  if constexpr (TOK == 32u) {
    return tile_body<GATE_UP, XT, NT, RT, TOK, 2>(a, it);
  } else if constexpr (TOK == 64u) {
    if (c16 == 2u) return tile_body<GATE_UP, XT, NT, RT, TOK, 2>(a, it);
    if (c16 == 3u) return tile_body<GATE_UP, XT, NT, RT, TOK, 3>(a, it);
    return tile_body<GATE_UP, XT, NT, RT, TOK, 4>(a, it);
  }
}

namespace {
using TileKernel = void (*)(TileArgs);
template <uint32_t RT, uint32_t TOK>
TileKernel tile_kernel_of(int nt, bool gate_up, bool x_bf16) {
  if (gate_up && nt == 1 && x_bf16) return expert_tile_kernel<true, uint16_t, 1, RT, TOK>;
  if (gate_up && nt == 2 && !x_bf16) return expert_tile_kernel<true, float, 2, RT, TOK>;
  if (!gate_up && nt == 1) return expert_tile_kernel<false, float, 1, RT, TOK>;
  if (!gate_up && nt == 2) return expert_tile_kernel<false, float, 2, RT, TOK>;
  return nullptr;
}
// The instantiation of a launch, null if there is none.
TileKernel tile_kernel(int nt, bool gate_up, bool x_bf16, const TileShape &t) {
  if (t.row_tiles == kTileLarge.row_tiles && t.tok == kTileLarge.tok) return tile_kernel_of<kTileLarge.row_tiles, kTileLarge.tok>(nt, gate_up, x_bf16);
  if (t.row_tiles == kTileSmall.row_tiles && t.tok == kTileSmall.tok) return tile_kernel_of<kTileSmall.row_tiles, kTileSmall.tok>(nt, gate_up, x_bf16);
  if (t.row_tiles == kTileDecode.row_tiles && t.tok == kTileDecode.tok) return tile_kernel_of<kTileDecode.row_tiles, kTileDecode.tok>(nt, gate_up, x_bf16);
  return nullptr;
}
}  // namespace

hipError_t configure_tile_kernels() {
  hipError_t err = hipSuccess;
  for (const TileShape &t : {kTileDecode, kTileSmall, kTileLarge})
    for (int nt = 1; nt <= 2; ++nt)
      for (int up = 0; up <= 1; ++up) {
        const hipError_t e = hipFuncSetAttribute((const void *)tile_kernel(nt, up != 0, nt == 1, t),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)tile_lds_bytes(nt, t));
        if (err == hipSuccess) err = e;
      }
  return err;
}

hipError_t launch_tile(const TileArgs &a, const TileShape &t, int nt, bool gate_up, bool x_bf16, uint32_t grid,
                       hipStream_t s) {
  const TileKernel k = tile_kernel(nt, gate_up, x_bf16, t);
  if (!k || grid == 0 || (grid & 7u) != 0 || a.nrb == 0 || a.nrt == 0 || a.nb == 0 || a.bstride % 32u != 0 ||
      a.bstride < a.kt || a.out_stride % 4u != 0 || a.E > kMaxExperts || a.bias_estride % 16u != 0 ||
      (t.tok == 16u && a.nperm > kSmallRouteMaxTokens * kMaxTopK))
    return hipErrorInvalidValue;
  return launch_kernel(k, dim3(grid), dim3(64 * kWaves), tile_lds_bytes(nt, t), s, a);
}

}  // namespace burnext
