// LDS-tiled grouped GEMM for the MFMA-bound regime: many tokens per expert
// (a prefill-shaped batch), the same frag-packed bf16 weights as the decode
// GEMMs.
//
//   Y[t, n] = sum_k X[row(t), k] * W_e[n, k]   for the tokens t of expert e
//
// Block tile 256 weight rows x up to 160 tokens, 4 waves, two blocks per CU.  Wave
// w owns rows 64 w .. +64 (four 16-row blocks) of every token of the tile: it
// loads its weight fragments straight into registers (the packed layout is MFMA
// operand order, 1 KiB contiguous per fragment, each read by one wave of the
// block only), four 32-wide k steps ahead, and reads the token operand, which
// the four waves share, from LDS.  The tokens' rows are copied global -> LDS in
// stages of 64 k (whole 128-byte lines per routed token, buffer_load_dwordx4 ...
// lds) in a ring of four stages with one barrier per stage.
//
// Why this split: per 32-wide k step of a CU (two blocks, 256 rows x 256 tokens)
// the matrix cores need 1024 clocks and the LDS serves 64 KiB of operand reads
// + 16 KiB of copies in ~640.  With both operands in LDS (one 8-wave block of
// 256 x 256 per CU, waves of 128 x 64) the same step moved 96 + 32 KiB through
// the LDS, ~1024 clocks, and took ~1800.  Two independent blocks also overlap
// one's group scan, first stage and epilogue (13 of the former block's 60 us)
// with the other's k loop.
//
// The inner loop is compiled for 32 .. 160 tokens and picked by the tile's live
// tokens.  A group of c tokens is cut into ceil(c / 160) equal tiles: with 128-token
// tiles a batch of ~128 tokens per expert left half the experts a second tile of a
// few tokens that streamed the expert's weights again (2048 tokens routed at random:
// gate/up 187 us against 143 at exactly 128 per expert).
//
// Epilogues: EPI_SWIGLU_BF16 (gate / up row blocks interleaved in the packing,
// so both halves of a pair sit in the same wave) and EPI_SCALE_F32 (affinity
// scaled fp32 rows), with the same element math as the decode GEMMs.
#include "common.h"
#include "gemm_epi.h"
#include "mkd_internal.h"
#include "launch_rules.h"

namespace mkd {

namespace {

constexpr int kTileRows = 256;           // packed weight rows per block
constexpr int kTileTok = 160;            // tokens per block (at most)
constexpr int kRB = kTileRows / 16;      // row blocks per block (16)
constexpr int kNW = 4;                   // waves; each owns kRB / kNW = 4 row blocks
constexpr int kStages = 4;               // LDS ring of 64-k token stages
constexpr int kStageTokBytes = 128;      // one token's 64 k of a stage
constexpr int kRingBytes = kStages * kTileTok * kStageTokBytes;
// the SwiGLU epilogue stages the whole h tile, [160 tokens][128 + 8 columns]
// bf16 (the padding shifts each token row by 4 banks), then the row indices
constexpr int kHsLd = 136;
constexpr int kLdsBytes = kRingBytes;
static_assert(kTileTok * kHsLd * 2 + kTileTok * 4 <= kRingBytes, "h staging fits the ring");
static_assert(2 * kLdsBytes <= 160 * 1024, "two blocks per CU");

// s_waitcnt with only vmcnt = n (expcnt / lgkmcnt left at their maxima); gfx9
// encoding: vmcnt[3:0] in bits 3:0, vmcnt[5:4] in bits 15:14.
template <int N>
MKD_DEV void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "6-bit vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}
// Keeps memory operations and their issue order on either side (the waits below
// count them).
MKD_DEV void issue_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
MKD_DEV void block_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
// (NT: the non-temporal cache policy, bit 1 of the auxiliary operand.)
template <bool NT>
MKD_DEV u32x4_t load_frag(__amdgpu_buffer_rsrc_t src, int voff, int soff) {
  return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(src, voff, soff, NT ? 2 : 0));
}
MKD_DEV void copy_rows_lds(__amdgpu_buffer_rsrc_t src, void* dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (__attribute__((address_space(3))) void*)dst, 16, voff,
                                           soff, 0, 0);
}

template <int V>
struct IntC {
  static constexpr int value = V;
};

// What a block works on.
struct TileJob {
  const uint16_t* wp;      // the expert's packed weights
  int nb0;                 // first row block
  int count, base, t0;     // the tile's end and first token in the group, the group's first pair
  int expert, kq;          // expert (bias), K slice
  int s0, S;               // first 32-wide k step, k steps
};

// The k loop and epilogue for tiles of at most 16 * WT tokens; PAIRS: the k steps
// are a multiple of 4.  ONCE: the group is this one tile, so no other block reads its
// weights: they are loaded non-temporal, which leaves the caches to the token rows
// (moe_prefill at 300 tokens 237 -> 219 us, at 1003 294 -> 270, at 2048 351 -> 344; with
// several tiles per group it would cost them their shared reads, 2048 tokens in
// 128-token tiles 347 -> 385).  Weight fragments are loaded four k steps ahead, two where
// the accumulators leave no registers for more (WT > 8).
template <int EPI, int WT, bool PAIRS, bool ONCE = false>
MKD_DEV void tile_body(const GemmArgs& a, const TileJob& jb, char* lds) {
  constexpr int C = (WT + 1) / 2;        // 8-token copies per wave per stage
  constexpr int H0 = (WT + 1) / 2, H1 = WT / 2;   // token tiles of a step's halves
  constexpr int AD = WT > 8 ? 2 : 4;     // weight k steps in flight
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int KB = a.K / 32, NB = (a.N + 15) / 16;
  const int S = jb.S, NS = (S + 1) / 2;  // k steps, 64-wide stages (the last may hold one step)
  const __amdgpu_buffer_rsrc_t wsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(jb.wp), 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t xsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.x), 0, 0x7fffffff, 0x00020000);

  // ---- token copies: copy f = w + 4 j moves tokens 8 f .. +8 of a stage, lane l
  // the 16-byte chunk (l % 8) ^ swz(token) of token 8 f + l / 8 (whole lines per
  // token), landing at byte 16 l of the copy's 1 KiB: token t's chunk c sits at
  // slot c ^ swz(t), swz(t) = (t / 2) % 8.  A lane group's 16 operand reads (16
  // tokens, one chunk) then cover all 64 banks once.
  int voff[C];
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int t = (w + kNW * j) * 8 + (lane >> 3);      // (past 16 WT: into unused slots)
    const int tc = min(jb.t0 + t, jb.count - 1);        // absent: any valid row
    const int row = a.pair_row ? a.pair_row[jb.base + tc] : jb.base + tc;
    voff[j] = (row * a.ldx + jb.s0 * 32) * 2 + (((lane & 7) ^ ((t >> 1) & 7)) << 4);
  }
  // half a stage (odd S): chunks 4-7 lie past the row's k range, chunk & 3 is read
  // instead (swz(t) / 4 is w % 2 for every copy of wave w)
  const bool odd = !PAIRS && (S & 1);
  const int past = (((lane >> 2) ^ w) & 1) * 64;
  auto issue = [&](int s) {
    char* dst = lds + (s & (kStages - 1)) * (kTileTok * kStageTokBytes);
    const int none = s < NS ? 0 : -1, sub = odd && s == NS - 1 ? past : 0;
    issue_fence();
#pragma unroll
    for (int j = 0; j < C; ++j)
      copy_rows_lds(xsrc, dst + (w + kNW * j) * 1024, (voff[j] - sub) | none, s * 128);
    issue_fence();
  };
  // ---- weight fragments: this wave's row blocks, 1 KiB per k step each ----
  int aoff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)            // rows past N: any valid block
    aoff[i] = __builtin_amdgcn_readfirstlane((min(jb.nb0 + 4 * w + i, NB - 1) * KB + jb.s0) * 1024);
  u32x4_t af[AD][4];                     // [k step % AD][row block]
  auto load_a = [&](u32x4_t (&f)[4], int step) {
    const int vo = lane * 16 | (step < S ? 0 : -1);
    issue_fence();
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = load_frag<ONCE>(wsrc, vo, aoff[i] + step * 1024);
    issue_fence();
  };
  // ---- operand reads: token tile j, step h of the stage in ring slot s % 4 ----
  const int rd = (lane & 15) * kStageTokBytes + (((lane >> 4) ^ ((lane >> 1) & 7)) << 4);
  auto read_b = [&](auto& b, int s, int h, int j0) {
    constexpr int n = sizeof(b) / sizeof(b[0]);
    const char* st = lds + (s & (kStages - 1)) * (kTileTok * kStageTokBytes) + (rd ^ (h * 64));
#pragma unroll
    for (int j = 0; j < n; ++j)
      b[j] = *reinterpret_cast<const u32x4_t*>(st + (j0 + j) * 16 * kStageTokBytes);
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4_t acc[4][WT];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < WT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto mul = [&](const u32x4_t (&f)[4], const auto& b, int j0) {
    constexpr int n = sizeof(b) / sizeof(b[0]);
#pragma unroll
    for (int j = 0; j < n; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i][j0 + j] = mfma16x16x32(f[i], b[j], acc[i][j0 + j]);
    __builtin_amdgcn_sched_barrier(0);
  };

  // Issue order of a wave's vector-memory operations (the waits count them); A0 / A1
  // are the 4 loads of a stage's first / second k step, d = AD / 2 stages ahead:
  //   prologue: copies(0) copies(1) A(0) copies(2) [A(1) if d = 2]
  //   stage s:  A0(s+d) [barrier] copies(s+3) A1(s+d)
  // Past the last stage they are issued with an offset past the buffer (no memory
  // access, zeros), so the counts and the compiler's own waits on the weight
  // registers stay exact without branches.  In the middle of stage s every wave
  // waits for its copies of stage s + 1 and takes the stage's one barrier:
  //  * after it stage s + 1 is readable (its first operands are read before the
  //    next barrier);
  //  * every wave's reads of stage s - 1 are complete (consumed by its MFMAs),
  //    so that ring slot takes stage s + 3.
  // Operations issued after copies(s + 1): A1 A0 copies(s+2) A1 A0 = 16 + C from
  // stage 2 on, and at least 12 + C in stages 0 and 1.
  issue(0);
  issue(1);
  load_a(af[0], 0);
  load_a(af[1], 1);
  issue(2);
  if (AD == 4) {
    load_a(af[AD - 2], 2);
    load_a(af[AD - 1], 3);
  }
  wait_vmcnt<4 * AD + 2 * C>();          // copies(0) landed: that many issued after them
  block_barrier();
  u32x4_t b0[H0], b1[H1];
  read_b(b0, 0, 0, 0);
  auto first = [&](int s, u32x4_t (&f0)[4]) {
    read_b(b1, s, 0, H0);
    mul(f0, b0, 0);
    read_b(b0, s, 1, 0);
    mul(f0, b1, H0);
  };
  auto second = [&](int s, u32x4_t (&f0)[4], u32x4_t (&f1)[4]) {
    load_a(f0, 2 * s + AD);
    wait_vmcnt<12 + C>();
    block_barrier();
    issue(s + 3);
    read_b(b1, s, 1, H0);
    mul(f1, b0, 0);
    read_b(b0, s + 1, 0, 0);             // (past the last stage: unused)
    mul(f1, b1, H0);
    load_a(f1, 2 * s + 1 + AD);
  };
  // PAIRS (S a multiple of 4: 2048, 768 and the padded 3072 of the two models): one exit,
  // so that the compiler's counts at the loop head are those of a full turn.  Otherwise
  // (2880 is 90 steps) the loop leaves after any step; the early exits cost it deeper
  // waits, and there is one form, for 160 tokens, whatever the tile holds.
  if (PAIRS) {
    for (int s = 0; s < NS; s += 2) {
      first(s, af[0]);
      second(s, af[0], af[1]);
      first(s + 1, af[AD - 2]);
      second(s + 1, af[AD - 2], af[AD - 1]);
    }
  } else {
    for (int s = 0;; s += 2) {
      first(s, af[0]);
      if (2 * s + 1 == S) break;
      second(s, af[0], af[1]);
      if (2 * s + 2 == S) break;
      first(s + 1, af[AD - 2]);
      if (2 * s + 3 == S) break;
      second(s + 1, af[AD - 2], af[AD - 1]);
      if (2 * s + 4 == S) break;
    }
  }

  // ---- epilogue: lane holds rows 4*(lane/16)+e of each row block, token lane%16 ----
  wait_vmcnt<0>();                       // every copy has landed
  const int q4 = (lane >> 4) * 4;
  constexpr int NT = 16 * WT;            // tokens of the tile
  if (EPI == EPI_SWIGLU_BF16) {
    // The h tile goes out through LDS: the waves store their SwiGLU values as
    // [token][128 h columns + 8] bf16, then 16 threads write each token's
    // 256-byte row segment in 16-byte stores -- directly, a store instruction
    // wrote 8 bytes into each of 16 scattered rows per lane group.
    const int I = a.N / 2;
    const uint16_t* bp = a.bias ? a.bias + (long long)jb.expert * a.bias_group_stride : nullptr;
    uint16_t* hs = reinterpret_cast<uint16_t*>(lds);
    int* orow_s = reinterpret_cast<int*>(hs + kTileTok * kHsLd);
    int orow = 0;
    if (tid < NT) {
      const int tc = min(jb.t0 + tid, jb.count - 1);
      orow = a.pair_out_row ? a.pair_out_row[jb.base + tc] : jb.base + tc;
    }
    __syncthreads();                     // every wave is past its last operand reads
    if (tid < NT) orow_s[tid] = orow;
    // (the activation is picked once per block, outside the element loops)
    auto h_tile = [&](auto kind) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int nbg = jb.nb0 + w * 4 + 2 * p;       // gate row block (even), up = nbg + 1
        if (nbg + 1 >= NB) continue;                  // h columns past I (never stored)
        const int n = (nbg >> 1) * 16 + q4;           // logical intermediate index
        const int nl = (w * 2 + p) * 16 + q4;         // its column in the tile's 128
        float gb[4] = {0.f, 0.f, 0.f, 0.f}, ub[4] = {0.f, 0.f, 0.f, 0.f};
        if (bp) {
#pragma unroll
          for (int e = 0; e < 4; ++e) { gb[e] = bf2f(bp[n + e]); ub[e] = bf2f(bp[I + n + e]); }
        }
#pragma unroll
        for (int j = 0; j < WT; ++j) {
          const int tl = j * 16 + (lane & 15);
          float o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = gated_value<decltype(kind)::value>(a, acc[2 * p][j][e] + gb[e], acc[2 * p + 1][j][e] + ub[e]);
          *reinterpret_cast<uint2*>(hs + tl * kHsLd + nl) = uint2{pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
        }
      }
    };
    const int kind = gated_kind(a);
    if (kind == kGatedQwen) h_tile(IntC<kGatedQwen>{});
    else if (kind == kGatedSigmoid) h_tile(IntC<kGatedSigmoid>{});
    else h_tile(IntC<kGatedGelu>{});
    __syncthreads();
    // N % 32 == 0, so I % 16 == 0: an 8-column piece is all below I or all past it
    const int c8 = (tid & 15) * 8;
    const int n = (jb.nb0 >> 1) * 16 + c8;
    if (n < I) {
      for (int tl = tid >> 4; tl < NT; tl += 16) {
        if (jb.t0 + tl >= jb.count) break;
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(hs + tl * kHsLd + c8);
        *reinterpret_cast<u32x4_t*>(static_cast<uint16_t*>(a.y) + (long long)orow_s[tl] * a.ldy + n) = v;
      }
    }
  } else {   // EPI_SCALE_F32
    // (K slices: the bias joins the first slice's partial)
    const uint16_t* bp = a.bias && jb.kq == 0 ? a.bias + (long long)jb.expert * a.bias_group_stride : nullptr;
    // Each wave turns its 64 rows x 16 tokens through its own 4 KiB of LDS and stores
    // 256 contiguous bytes per token (16 lanes x 16 bytes), with no barrier among
    // the waves.  Straight from the registers a store covers 64 bytes of each of 16
    // rows: 2048 tokens 119 instead of 112 us.  (Non-temporal stores of the grouped rows
    // make no difference: moe_prefill at 1003 tokens 274.6 us plain and 274.9, at 8192
    // 794.2 and 794.3.)
    constexpr int kLd = 68;                           // 64 rows + 4 floats of padding
    float* stg = reinterpret_cast<float*>(lds) + w * 16 * kLd;
    __syncthreads();                                  // every wave is past its last operand reads
    float* ybase = static_cast<float*>(a.y) + jb.kq * a.part_stride;
    const int n0 = (jb.nb0 + w * 4) * 16, n = n0 + (lane & 15) * 4;
    // the output rows and scales of tokens lane, lane + 64, lane + 128 of the tile
    int orow[(WT + 3) / 4];
    float osc[(WT + 3) / 4];
#pragma unroll
    for (int k = 0; k < (WT + 3) / 4; ++k) {
      const int t = min(jb.t0 + 64 * k + lane, jb.count - 1);
      orow[k] = a.pair_out_row ? a.pair_out_row[jb.base + t] : jb.base + t;
      osc[k] = a.pair_scale ? a.pair_scale[orow[k]] : 1.0f;
    }
    float bb[4] = {0.f, 0.f, 0.f, 0.f};               // this lane's four rows as stored
    if (bp) {
#pragma unroll
      for (int e = 0; e < 4; ++e) bb[e] = n + e < a.N ? bf2f(bp[n + e]) : 0.f;
    }
#pragma unroll
    for (int j = 0; j < WT; ++j) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4_t*>(stg + (lane & 15) * kLd + i * 16 + q4) = acc[i][j];
      wave_lds_sync();
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int tl = 4 * u + (lane >> 4), tt = j * 16 + tl;   // token of the 16, of the tile
        f32x4_t v = *reinterpret_cast<const f32x4_t*>(stg + tl * kLd + (lane & 15) * 4);
        const int row = __shfl(orow[j / 4], tt & 63, 64);
        const float sc = __shfl(osc[j / 4], tt & 63, 64);
        if (jb.t0 + tt >= jb.count) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (v[e] + bb[e]) * sc;
        float* y = ybase + (long long)row * a.ldy + n;
        if (n + 3 < a.N) {
          *reinterpret_cast<f32x4_t*>(y) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < a.N) y[e] = v[e];
        }
      }
      wave_lds_sync();
    }
  }
}

}  // namespace

template <int EPI>
__global__ void __launch_bounds__(64 * kNW, 2) gemm_tile_kernel(GemmArgs a, int gx, int dense_tok) {
  extern __shared__ __attribute__((aligned(16))) char tile_lds[];
  char* lds = tile_lds;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform in an SGPR
  // Grid: gx n tiles x work items, linear.  Work items are the token tiles of all
  // groups in group order (group g owns ceil(count_g / 160) consecutive items); the grid
  // holds an upper bound (ceil(T*K / 160) + groups) and the block finds its
  // group by a scan of the device-side group counts.  XCD-aware order: blocks
  // are dealt round-robin to the 8 XCDs by linear id, so each XCD is given a
  // contiguous run of the LIVE logical tiles (n tile fastest, then item): the
  // blocks that share an expert's weight tiles and token rows run together on
  // one XCD's L2, and every XCD gets an eighth of the work.  (Dealing out the
  // grid's upper bound instead put its dead items -- those past the last live
  // token tile -- on the last XCDs: at 2048 tokens over 128 experts 128 of 192
  // 256-token items were live, and two XCDs sat idle.)
  int* scan_s = reinterpret_cast<int*>(lds);   // before any copy into the ring
  int* item_s = scan_s + 8;
  const int L = blockIdx.x;
  // (tile_deal_rule: XCD L % 8 owns a contiguous run of the live tiles, its
  // k-th block takes tile k of it, blocks past the run have no work; the grid
  // holds at least `live` blocks, so every tile is taken)
  auto deal = [&](int live, int& lt) { return tile_deal_rule(live, L, &lt); };
  int lt = 0;
  bool once = false;                     // a group of one tile

  TileJob jb;
  jb.wp = a.w;
  jb.expert = jb.kq = 0;
  if (a.grp_expert) {
    // thread i holds the token-tile counts of groups 2 i and 2 i + 1 (<= 512
    // groups); block-wide inclusive scan in group order; the owner of the
    // block's item publishes it
    const int ng = *a.n_groups;
    const int g0 = 2 * tid;
    const int tiles0 = ((g0 < ng ? a.grp_count[g0] : 0) + kTileTok - 1) / kTileTok;
    const int tiles1 = ((g0 + 1 < ng ? a.grp_count[g0 + 1] : 0) + kTileTok - 1) / kTileTok;
    int x = tiles0 + tiles1;             // wave inclusive scan (64 lanes)
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) scan_s[w] = x;
    if (tid == 0) item_s[0] = -1;
    __syncthreads();
    int before = 0, items = 0;
    for (int q = 0; q < kNW; ++q) {
      const int v = scan_s[q];
      if (q < w) before += v;
      items += v;
    }
    const bool mine = deal(gx * items, lt);
    const int item = lt / gx;
    const int end = before + x, mid = end - tiles1, beg = mid - tiles0;
    if (mine && item >= beg && item < end) {
      item_s[0] = item < mid ? g0 : g0 + 1;
      item_s[1] = item - (item < mid ? beg : mid);
    }
    __syncthreads();
    const int g = __builtin_amdgcn_readfirstlane(item_s[0]);
    if (g < 0) return;                   // past the last live token tile (uniform)
    const int k = __builtin_amdgcn_readfirstlane(item_s[1]);
    const int cnt = a.grp_count[g];
    const int per = tile_even_rule(cnt, kTileTok);   // the group's equal tiles
    jb.t0 = k * per;
    jb.count = min(cnt, jb.t0 + per);
    once = cnt <= kTileTok;
    jb.base = a.grp_offset[g];
    jb.expert = a.grp_expert[g];
    jb.wp += (long long)jb.expert * a.w_group_stride;
    __syncthreads();                     // item_s read by every wave before the copies
  } else {
    // dense: the items are token tiles x K slices (kgrid > 1: fp32 partials, one
    // per slice, at y + slice * part_stride; the slice is the slowest index, so
    // an XCD's run shares one K slice of the weights)
    if (!deal((int)gridDim.x, lt)) return;   // (the grid is exact here)
    const int items = (int)gridDim.x / gx / (a.kgrid > 1 ? a.kgrid : 1);
    const int r = lt / gx;
    jb.kq = r / items;
    jb.base = 0;
    jb.t0 = (r - jb.kq * items) * dense_tok;
    jb.count = min(a.T, jb.t0 + dense_tok);
    if (jb.t0 >= a.T) return;
  }
  jb.nb0 = (lt % gx) * kRB;
  jb.S = a.grp_expert || a.kgrid <= 1 ? a.K / 32 : a.K / 32 / a.kgrid;
  jb.s0 = jb.kq * jb.S;
  const int live = jb.count - jb.t0;
  if (jb.S & 3) {
    tile_body<EPI, 10, false>(a, jb, lds);
  } else if (once) {
    if (live <= 32) tile_body<EPI, 2, true, true>(a, jb, lds);
    else if (live <= 64) tile_body<EPI, 4, true, true>(a, jb, lds);
    else if (live <= 96) tile_body<EPI, 6, true, true>(a, jb, lds);
    else if (live <= 128) tile_body<EPI, 8, true, true>(a, jb, lds);
    else tile_body<EPI, 10, true, true>(a, jb, lds);
  } else {                               // (grouped: 81 .. 160 tokens but for a last tile)
    if (live <= 32) tile_body<EPI, 2, true>(a, jb, lds);
    else if (live <= 64) tile_body<EPI, 4, true>(a, jb, lds);
    else if (live <= 96) tile_body<EPI, 6, true>(a, jb, lds);
    else if (live <= 112) tile_body<EPI, 7, true>(a, jb, lds);
    else if (live <= 128) tile_body<EPI, 8, true>(a, jb, lds);
    else if (live <= 144) tile_body<EPI, 9, true>(a, jb, lds);
    else tile_body<EPI, 10, true>(a, jb, lds);
  }
}

int gemm_tile_lds_bytes() { return kLdsBytes; }

bool gemm_tile_supported(int N, int K, int epi) {
  if (K % 32 != 0 || K <= 0 || N <= 0) return false;
  if (epi == EPI_SWIGLU_BF16) return N % 32 == 0;
  return epi == EPI_SCALE_F32;
}

bool gemm_tile_kgrid_ok(int K, int kgrid) {
  const int KB = K / 32;
  return kgrid >= 1 && kgrid <= 8 && K % 32 == 0 && KB % kgrid == 0;
}

// K slices for a dense tiled GEMM whose output tiles leave CUs idle (a short
// prefill pass: the attention output projection at 2048 tokens has 64 tiles):
// the largest of 2, 4, 8 that keeps tiles x slices within two blocks per CU (the
// rule counts pairs of 128-token tiles, one pair per CU) and at least 16 k steps
// per slice.  The partials cost T * N * 4 bytes per slice
// written and read again by the consumer.
int gemm_tile_kgrid(int N, int K, int T) {
  static_assert(kTileRows == 256, "tile_kgrid_rule counts 256 x 2 x 128 tile pairs");
  return tile_kgrid_rule(N, K, T, device_cus());
}

hipError_t gemm_tile_launch(const GemmArgs& a, int epi, int groups_max, long long total_rows,
                            hipStream_t s) {
  if (!gemm_tile_supported(a.N, a.K, epi) || groups_max <= 0 || total_rows <= 0)
    return hipErrorInvalidValue;
  // the SwiGLU epilogue writes h in 16-byte pieces
  if (epi == EPI_SWIGLU_BF16 && ((a.ldy & 7) || (reinterpret_cast<uintptr_t>(a.y) & 15)))
    return hipErrorInvalidValue;
  // K slices: dense fp32 partials only, each slice's rows clear of the next's
  const int kg = a.kgrid > 1 ? a.kgrid : 1;
  if (kg > 1 && (a.grp_expert || epi != EPI_SCALE_F32 || a.pair_scale || !gemm_tile_kgrid_ok(a.K, kg) ||
                 a.part_stride < total_rows * a.ldy))
    return hipErrorInvalidValue;
  // work items: every group's token tiles; with total_rows = sum of the group
  // sizes, sum_g ceil(c_g / 160) <= ceil(total_rows / 160) + groups.  Dense:
  // token tiles sized to give every CU one (tile_dense_rule).
  const int gx = (a.N + kTileRows - 1) / kTileRows;
  const int tok = a.grp_expert ? kTileTok : tile_dense_rule(gx * kg, a.T, device_cus());
  const long long items = (total_rows + tok - 1) / tok + (a.grp_expert ? groups_max : 0);
  if (items * kg * gx > 0x7fffffff / (64 * kNW)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(items * kg * gx));
  // 80 KiB of dynamic LDS is above the default launch limit (set per kernel)
  if (epi == EPI_SWIGLU_BF16) {
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tile_kernel<EPI_SWIGLU_BF16>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes))
      return e;
    return timed_launch(gemm_tile_kernel<EPI_SWIGLU_BF16>, grid, dim3(64 * kNW), kLdsBytes, s, a, gx, tok);
  }
  if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tile_kernel<EPI_SCALE_F32>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes))
    return e;
  return timed_launch(gemm_tile_kernel<EPI_SCALE_F32>, grid, dim3(64 * kNW), kLdsBytes, s, a, gx, tok);
}

}  // namespace mkd
