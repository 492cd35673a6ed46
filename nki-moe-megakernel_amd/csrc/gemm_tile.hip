// LDS-tiled grouped GEMM for the MFMA-bound regime: many tokens per expert
// (a prefill-shaped batch), the same frag-packed bf16 weights as the decode
// GEMMs.
//
//   Y[t, n] = sum_k X[row(t), k] * W_e[n, k]   for the tokens t of expert e
//
// Block tile 256 weight rows x up to 128 tokens, 4 waves, two blocks per CU.  Wave
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
// The inner loop is compiled for 32, 64, 96 and 128 tokens and picked by the
// tile's live tokens, so a group's last tile (or a small expert's only one)
// multiplies at most 31 absent tokens.
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
constexpr int kTileTok = 128;            // tokens per block (at most)
constexpr int kRB = kTileRows / 16;      // row blocks per block (16)
constexpr int kNW = 4;                   // waves; each owns kRB / kNW = 4 row blocks
constexpr int kStages = 4;               // LDS ring of 64-k token stages
constexpr int kStageTokBytes = 128;      // one token's 64 k of a stage
constexpr int kRingBytes = kStages * kTileTok * kStageTokBytes;
// the fp32 epilogue stages half of the output tile in LDS, [128 tokens][128 + 4
// rows] (the 4 floats of padding spread a lane group's 16 rows over the banks),
// then the block's output row indices
constexpr int kStgLd = 132;
constexpr int kStgBytes = kTileTok * kStgLd * 4 + kTileTok * 4;
// the SwiGLU epilogue stages the whole h tile, [128 tokens][128 + 8 columns]
// bf16 (the padding shifts each token row by 4 banks), then the row indices
constexpr int kHsLd = 136;
static_assert(kTileTok * kHsLd * 2 + kTileTok * 4 <= kStgBytes, "h staging fits the fp32 staging area");
constexpr int kLdsBytes = kRingBytes > kStgBytes ? kRingBytes : kStgBytes;
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
// A non-template wrapper (the builtin stays out of template instantiation).
MKD_DEV u32x4_t load_frag(__amdgpu_buffer_rsrc_t src, int voff, int soff) {
  return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(src, voff, soff, 0));
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
  int count, base, t0;     // the group's tokens, its first pair, the tile's first token
  int expert, kq;          // expert (bias), K slice
  int s0, S;               // first 32-wide k step, k steps
};

// The k loop and epilogue for tiles of at most 16 * WT tokens (WT even); PAIRS:
// the k steps are a multiple of 4.
template <int EPI, int WT, bool PAIRS>
MKD_DEV void tile_body(const GemmArgs& a, const TileJob& jb, char* lds) {
  constexpr int C = WT / 2;              // 8-token copies per wave per stage
  constexpr int HT = WT / 2;             // token tiles per half step
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
    const int t = (w + kNW * j) * 8 + (lane >> 3);
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
  u32x4_t af[4][4];                      // [k step % 4][row block]
  auto load_a = [&](u32x4_t (&f)[4], int step) {
    const int vo = lane * 16 | (step < S ? 0 : -1);
    issue_fence();
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = load_frag(wsrc, vo, aoff[i] + step * 1024);
    issue_fence();
  };
  // ---- operand reads: token tile j, step h of the stage in ring slot s % 4 ----
  const int rd = (lane & 15) * kStageTokBytes + (((lane >> 4) ^ ((lane >> 1) & 7)) << 4);
  auto read_b = [&](u32x4_t (&b)[HT], int s, int h, int half) {
    const char* st = lds + (s & (kStages - 1)) * (kTileTok * kStageTokBytes) + (rd ^ (h * 64));
#pragma unroll
    for (int j = 0; j < HT; ++j)
      b[j] = *reinterpret_cast<const u32x4_t*>(st + (half * HT + j) * 16 * kStageTokBytes);
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4_t acc[4][WT];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < WT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto mul = [&](const u32x4_t (&f)[4], const u32x4_t (&b)[HT], int half) {
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i][half * HT + j] = mfma16x16x32(f[i], b[j], acc[i][half * HT + j]);
    __builtin_amdgcn_sched_barrier(0);
  };

  // Issue order of a wave's vector-memory operations (the waits count them):
  //   prologue: copies(0) copies(1) A(0) copies(2) A(1)
  //   stage s:  A0(s+2) [barrier] copies(s+3) A1(s+2)      (A0 / A1: 4 loads each)
  // Past the last stage they are issued with an offset past the buffer (no memory
  // access, zeros), so the counts and the compiler's own waits on the weight
  // registers stay exact without branches.  In the middle of stage s every wave
  // waits for its copies of stage s + 1 and takes the stage's one barrier:
  //  * after it stage s + 1 is readable (its first operands are read before the
  //    next barrier);
  //  * every wave's reads of stage s - 1 are complete (consumed by its MFMAs),
  //    so that ring slot takes stage s + 3.
  // Operations issued after copies(s + 1): A1(s) A0(s+1) copies(s+2) A1(s+1)
  // A0(s+2) = 16 + C (the prologue's order adds to that, so the wait holds there
  // too).
  issue(0);
  issue(1);
  load_a(af[0], 0);
  load_a(af[1], 1);
  issue(2);
  load_a(af[2], 2);
  load_a(af[3], 3);
  wait_vmcnt<16 + 2 * C>();              // copies(0) landed: 2 C + 16 issued after them
  block_barrier();
  u32x4_t b0[HT], b1[HT];
  read_b(b0, 0, 0, 0);
  auto first = [&](int s, u32x4_t (&f0)[4]) {
    read_b(b1, s, 0, 1);
    mul(f0, b0, 0);
    read_b(b0, s, 1, 0);
    mul(f0, b1, 1);
  };
  auto second = [&](int s, u32x4_t (&f0)[4], u32x4_t (&f1)[4]) {
    load_a(f0, 2 * s + 4);
    wait_vmcnt<16 + C>();
    block_barrier();
    issue(s + 3);
    read_b(b1, s, 1, 1);
    mul(f1, b0, 0);
    read_b(b0, s + 1, 0, 0);             // (past the last stage: unused)
    mul(f1, b1, 1);
    load_a(f1, 2 * s + 5);
  };
  // PAIRS (S a multiple of 4, every shape of the two models): one exit, so that the
  // compiler's counts at the loop head are those of a full turn.  Otherwise the
  // loop leaves after any step; the early exits cost it deeper waits.
  if (PAIRS) {
    for (int s = 0; s < NS; s += 2) {
      first(s, af[0]);
      second(s, af[0], af[1]);
      first(s + 1, af[2]);
      second(s + 1, af[2], af[3]);
    }
  } else {
    for (int s = 0;; s += 2) {
      first(s, af[0]);
      if (2 * s + 1 == S) break;
      second(s, af[0], af[1]);
      if (2 * s + 2 == S) break;
      first(s + 1, af[2]);
      if (2 * s + 3 == S) break;
      second(s + 1, af[2], af[3]);
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
    // The tile goes out through LDS, half (128 rows) at a time: the waves of
    // that half store their scaled accumulators as [token][row], then every
    // thread writes 16 contiguous bytes of a token's 512-byte row segment --
    // directly, a store instruction wrote 64 bytes into each of 16 scattered
    // output rows, and the stores took ~40 % of the down projection's time.
    float* stg = reinterpret_cast<float*>(lds);
    int* orow_s = reinterpret_cast<int*>(stg + kTileTok * kStgLd);
    // all affinities up front (y is float too, so loads among the stores could
    // not be moved past them)
    float sc[WT];
#pragma unroll
    for (int j = 0; j < WT; ++j) {
      const int tc = min(jb.t0 + j * 16 + (lane & 15), jb.count - 1);
      sc[j] = a.pair_scale ? a.pair_scale[a.pair_out_row ? a.pair_out_row[jb.base + tc] : jb.base + tc] : 1.0f;
    }
    int orow = 0;
    if (tid < NT) {
      const int tc = min(jb.t0 + tid, jb.count - 1);
      orow = a.pair_out_row ? a.pair_out_row[jb.base + tc] : jb.base + tc;
    }
    __syncthreads();                     // every wave is past its last operand reads
    if (tid < NT) orow_s[tid] = orow;
    float* ybase = static_cast<float*>(a.y) + jb.kq * a.part_stride;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (w >> 1 == half) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int n = (jb.nb0 + w * 4 + i) * 16 + q4;
          float bb[4] = {0.f, 0.f, 0.f, 0.f};
          if (bp) {
#pragma unroll
            for (int e = 0; e < 4; ++e) bb[e] = (n + e < a.N) ? bf2f(bp[n + e]) : 0.f;
          }
#pragma unroll
          for (int j = 0; j < WT; ++j) {
            const int tl = j * 16 + (lane & 15);
            *reinterpret_cast<f32x4_t*>(stg + tl * kStgLd + ((w & 1) * 4 + i) * 16 + q4) =
                f32x4_t{(acc[i][j][0] + bb[0]) * sc[j], (acc[i][j][1] + bb[1]) * sc[j],
                        (acc[i][j][2] + bb[2]) * sc[j], (acc[i][j][3] + bb[3]) * sc[j]};
          }
        }
      }
      __syncthreads();
      const int c4 = (tid & 31) * 4;                  // row offset within the half
      const int n = (jb.nb0 + half * 8) * 16 + c4;
      for (int tl = tid >> 5; tl < NT; tl += 8) {
        if (jb.t0 + tl >= jb.count) break;
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(stg + tl * kStgLd + c4);
        float* y = ybase + (long long)orow_s[tl] * a.ldy + n;
        if (n + 3 < a.N) {
          *reinterpret_cast<f32x4_t*>(y) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < a.N) y[e] = v[e];
        }
      }
      __syncthreads();                   // the half is read before the next one is written
    }
  }
}

}  // namespace

template <int EPI>
__global__ void __launch_bounds__(64 * kNW, 2) gemm_tile_kernel(GemmArgs a, int gx) {
  extern __shared__ __attribute__((aligned(16))) char tile_lds[];
  char* lds = tile_lds;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform in an SGPR
  // Grid: gx n tiles x work items, linear.  Work items are the token tiles of all
  // groups in group order (group g owns ceil(count_g / 128) consecutive items); the grid
  // holds an upper bound (ceil(T*K / 128) + groups) and the block finds its
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
      item_s[1] = (item - (item < mid ? beg : mid)) * kTileTok;
    }
    __syncthreads();
    const int g = __builtin_amdgcn_readfirstlane(item_s[0]);
    if (g < 0) return;                   // past the last live token tile (uniform)
    jb.t0 = __builtin_amdgcn_readfirstlane(item_s[1]);
    jb.count = a.grp_count[g];
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
    jb.count = a.T;
    jb.base = 0;
    jb.t0 = (r - jb.kq * items) * kTileTok;
    if (jb.t0 >= jb.count) return;
  }
  jb.nb0 = (lt % gx) * kRB;
  jb.S = a.grp_expert || a.kgrid <= 1 ? a.K / 32 : a.K / 32 / a.kgrid;
  jb.s0 = jb.kq * jb.S;
  const int live = min(jb.count - jb.t0, kTileTok);
  if (jb.S & 3) tile_body<EPI, 8, false>(a, jb, lds);
  else if (live <= 32) tile_body<EPI, 2, true>(a, jb, lds);
  else if (live <= 64) tile_body<EPI, 4, true>(a, jb, lds);
  else if (live <= 96) tile_body<EPI, 6, true>(a, jb, lds);
  else tile_body<EPI, 8, true>(a, jb, lds);
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
  static_assert(kTileRows == 256 && kTileTok == 128, "tile_kgrid_rule counts 256 x 2 x 128 tile pairs");
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
  // sizes, sum_g ceil(c_g / 128) <= ceil(total_rows / 128) + groups
  const long long items = (total_rows + kTileTok - 1) / kTileTok + (a.grp_expert ? groups_max : 0);
  const int gx = (a.N + kTileRows - 1) / kTileRows;
  if (items * kg * gx > 0x7fffffff / (64 * kNW)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(items * kg * gx));
  // 66.5 KiB of dynamic LDS is above the default launch limit (set per kernel)
  if (epi == EPI_SWIGLU_BF16) {
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tile_kernel<EPI_SWIGLU_BF16>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes))
      return e;
    return timed_launch(gemm_tile_kernel<EPI_SWIGLU_BF16>, grid, dim3(64 * kNW), kLdsBytes, s, a, gx);
  }
  if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tile_kernel<EPI_SCALE_F32>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes))
    return e;
  return timed_launch(gemm_tile_kernel<EPI_SCALE_F32>, grid, dim3(64 * kNW), kLdsBytes, s, a, gx);
}

}  // namespace mkd
