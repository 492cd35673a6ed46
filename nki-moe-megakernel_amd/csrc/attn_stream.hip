// Split-K decode attention for grids that fill the chip (and for FP8 caches of any
// size): one pass over a chunk of 64 .. 512 positions per block, bound by HBM.
//
// Block (kv head g, chunk c, query row b), 4 waves.  Wave w takes the chunk's
// 32-position steps w, w + 4, ... with an online softmax; per step (two 16-row
// tiles)
//   S = K_tile . q^T  v_mfma_f32_16x16x32_bf16, A = 16 K rows, B = the GQA query
//                     heads (16 columns); D lane l holds S[pos 4 (l/16) + i][head l % 16]
//   O += P . V        the two tiles' positions on the 32-deep MFMA, P straight from
//                     the S layout, V rows as they come (lane column l % 16 owns D / 16
//                     contiguous elements of its rows; d-tile dt is element dt)
// A step's K registers are refilled with the next step's rows as soon as its scores
// are formed and its V registers after its P . V, so every wave has 8 (FP8) or
// 16 KiB (bf16) in flight through the softmax, and one prior-length and one
// block-table round trip per chunk instead of one per tile pair.  At 64 sequences
// of 512 .. 8192 positions on a paged cache the former form (256-position chunks,
// each wave loading K, then V, of two tiles at a time, every lane dividing for its
// own table entry) took 161 us per layer, this one 108-111 (554 MB fetched, 5.1 TB/s);
// FP8 at 16 x 4096 positions 300 us in plain VALU math (attn_kvfmt_kernel), 29 here
// (72 MB fetched, 50 of them rows: the mask's lines are read by every XCD).  The masked
// bf16 forms of 128-wide heads spill 11 to 13 registers (the eight mask bytes a lane
// holds a step ahead); no other form does.
//
// FP8 caches (e4m3 codes, attention_block_tkg.py:133-134, :749-754): a code is
// exactly a bf16 value, so the scores are those of the stored values with fp32
// accumulation; the probabilities, which this path keeps in fp32, go to the MFMA
// as three bf16 terms that add up to the fp32 value (8 significand bits each).
// Each lane reads 32 contiguous bytes of a K row (head elements (l/16) D/4 .. , in
// the q operand alike).
//
// A 16-position tile lies in one cache block (block lengths are multiples of 16
// here; others keep attn_fused_kernel / attn_kvfmt_kernel), so its base address is
// one scalar table lookup, made a step ahead.  Rows come through a per-tile buffer
// resource: a tile with no valid block, a step past the chunk and a step whose
// every position is masked for the group have zero records -- the loads return
// zeros without touching memory.
#include "common.h"
#include "fp8.h"
#include "mkd_internal.h"
#include "attn_common.h"

namespace mkd {

namespace {

constexpr int kStWaves = 4;
constexpr int kStStep = 32;                   // positions per wave step
constexpr int kStMaxNew = 8;                  // new tokens per sequence

// Wrappers outside the template (dword-count variants of one buffer load; NT: the
// non-temporal cache policy, bit 1 of the auxiliary operand).
template <bool NT>
MKD_DEV u32x4_t buf_ld16(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, NT ? 2 : 0));
}
template <bool NT>
MKD_DEV uint2 buf_ld8(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, NT ? 2 : 0));
}
MKD_DEV uint32_t buf_ld4(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
}
MKD_DEV __amdgpu_buffer_rsrc_t buf_of(const char* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p), 0, bytes, 0x00020000);
}
MKD_DEV f32x2_t cvt2_fp8_lo(uint32_t v) { return __builtin_amdgcn_cvt_pk_f32_fp8((int)v, false); }
MKD_DEV f32x2_t cvt2_fp8_hi(uint32_t v) { return __builtin_amdgcn_cvt_pk_f32_fp8((int)v, true); }

// eight e4m3 codes -> eight bf16 (exact)
MKD_DEV u32x4_t fp8x8_to_bf16(uint32_t a, uint32_t b) {
  const f32x2_t x = cvt2_fp8_lo(a), y = cvt2_fp8_hi(a), z = cvt2_fp8_lo(b), w = cvt2_fp8_hi(b);
  return u32x4_t{pack2bf(x[0], x[1]), pack2bf(y[0], y[1]), pack2bf(z[0], z[1]), pack2bf(w[0], w[1])};
}

}  // namespace

// NTL: non-temporal cache loads, chunks dealt before kv heads (attn_stream_launch).
template <int D, int GQA, bool FP8, bool MASK, bool NTL>
__global__ void __launch_bounds__(64 * kStWaves, FP8 && D == 64 ? 4 : 3) attn_stream_kernel(AttnArgs a) {
  constexpr int EB = FP8 ? 1 : 2;             // bytes per cached element
  constexpr int NK = D / 32, NDT = D / 16;
  constexpr int KL = D * EB / 64;             // 16-byte loads of a lane's K row share
  constexpr int VD = D * EB / 64;             // dwords of a lane's V row share
  __shared__ float m_s[kStWaves][16], l_s[kStWaves][16];
  __shared__ __attribute__((aligned(16))) float o_s[kStWaves][GQA][D];
  __shared__ __attribute__((aligned(16))) uint16_t q_s[GQA][D];
  __shared__ __attribute__((aligned(16))) uint16_t kn_s[kStMaxNew][D], vn_s[kStMaxNew][D];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q4 = lane >> 4, col = lane & 15;
  const int L = blockIdx.x + gridDim.x * blockIdx.y, b = blockIdx.z;
  const int g = NTL ? L / gridDim.y : blockIdx.x, c = NTL ? L % gridDim.y : blockIdx.y;
  const int CP = a.chunk, chunk0 = c * CP;
  const int NT = new_tokens(a), seq = seq_of(a, b), tk = tok_of(a, b);
  const int n = __builtin_amdgcn_readfirstlane(prior_len(a, b)), total = n + NT;
  if (chunk0 >= total) return;                // whole block: uniform exit
  const int nst = (min(CP, total - chunk0) + kStStep - 1) / kStStep;

  // ---- this wave's steps: tile addresses ----
  const long long head0 = (long long)seq * a.cache_b_stride + g * a.cache_h_stride;   // flat
  const int row_b = (a.block_table ? a.nkv * D : D) * EB;                             // bytes per position
  const int last_tile = max(n - 1, 0) & ~15;  // the last tile holding a prior position
  auto tile_of = [&](int st, int u) { return min(chunk0 + st * kStStep + 16 * u, last_tile); };
  auto tile_blk = [&](int st, int u) -> int {
    return a.block_table ? a.block_table[(long long)seq * a.tbl_stride + tile_of(st, u) / a.blk_len] : 0;
  };
  // byte offset of the tile's first row; records = 0 where there is nothing to read
  auto tile_off = [&](int st, int u, int blk, bool live, int& records) -> long long {
    const int t0 = tile_of(st, u);
    bool ok = live && n > 0;
    long long e;
    if (a.block_table) {
      ok = ok && (unsigned)blk < (unsigned)a.num_blocks;
      e = ok ? (((long long)blk * a.blk_len + t0 % a.blk_len) * a.nkv + g) * D : 0;
    } else {
      e = head0 + (long long)t0 * D;
    }
    records = ok ? 16 * row_b : 0;
    return e * EB;
  };
  // last row of the tile that holds a prior position (rows past it re-read it)
  auto tile_rmax = [&](int st, int u) { return max(min(15, n - 1 - tile_of(st, u)), 0); };
  const char* kc = reinterpret_cast<const char*>(a.k_cache);
  const char* vc = reinterpret_cast<const char*>(a.v_cache);

  u32x4_t kr[2][KL];
  uint32_t vr[2][4][VD];
  auto load_k = [&](int st, const int (&blk)[2], bool live) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      int rec;
      const long long off = tile_off(st, u, blk[u], live, rec);
      const __amdgpu_buffer_rsrc_t r = buf_of(kc + off, rec);
      const int vo = min(col, tile_rmax(st, u)) * row_b;
#pragma unroll
      for (int j = 0; j < KL; ++j)
        kr[u][j] = buf_ld16<NTL>(r, vo + (FP8 ? q4 * (D / 4) + 16 * j : q4 * 16 + 64 * j));
    }
  };
  auto load_v = [&](int st, const int (&blk)[2], bool live) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      int rec;
      const long long off = tile_off(st, u, blk[u], live, rec);
      const __amdgpu_buffer_rsrc_t r = buf_of(vc + off, rec);
      const int rm = tile_rmax(st, u);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int vo = min(4 * q4 + j, rm) * row_b + col * (4 * VD);
        if constexpr (VD == 4) {
          const u32x4_t v = buf_ld16<NTL>(r, vo);
#pragma unroll
          for (int e = 0; e < 4; ++e) vr[u][j][e] = v[e];
        } else if constexpr (VD == 2) {
          const uint2 v = buf_ld8<NTL>(r, vo);
          vr[u][j][0] = v.x;
          vr[u][j][1] = v.y;
        } else {
          vr[u][j][0] = buf_ld4(r, vo);
        }
      }
    }
  };
  // the mask bytes of a lane's 8 scores of a step (position 16 u + 4 q4 + i, head col)
  uint8_t mb[2][4];
  auto load_mask = [&](int st) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tp = min(chunk0 + st * kStStep + 16 * u + 4 * q4 + i, total - 1);
        const int mt = tp < n ? tp : (a.mask_s_ctx - NT + (tp - n));
        mb[u][i] = a.mask[(((long long)mt * (a.B / NT) + seq) * a.nq + g * GQA + min(col, GQA - 1)) * NT + tk];
      }
  };
  auto mask_bits = [&]() {
    uint32_t v = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) v |= (mb[k >> 2][k & 3] != 0 ? 1u : 0u) << k;
    return v;
  };

  // the block's query heads and the sequence's new k | v rows, 16 bytes per thread
  // (GQA D <= 2048, 2 NT D <= 2048), ahead of the cache rows: a wave's loads
  // complete in order
  static_assert(GQA * D <= 64 * kStWaves * 8 && 2 * kStMaxNew * D <= 64 * kStWaves * 8, "one piece per thread");
  const long long hs = (long long)(GQA + 2) * D;
  const int e0 = threadIdx.x * 8;
  const u32x4_t qv = ld16(a.prep + ((long long)b * a.nkv + g) * hs + min(e0, GQA * D - 8));
  const int ns = min(e0 / (2 * D), NT - 1), ne = e0 % (2 * D);
  const u32x4_t nv = ld16(a.prep + (((long long)seq * NT + ns) * a.nkv + g) * hs + GQA * D + ne);

  int st = w;
  int blk[2] = {tile_blk(st, 0), tile_blk(st, 1)}, blkn[2];
  uint32_t bits = 0xffu, bits_n = 0xffu;
  bool live = st < nst;
  if constexpr (MASK) {
    load_mask(min(st, nst - 1));
    bits = mask_bits();
    load_mask(min(st + kStWaves, nst - 1));
    live = live && __any(bits != 0);
  }
  load_k(st, blk, live);
  load_v(st, blk, live);

  if (e0 < GQA * D) st16(&q_s[0][0] + e0, qv);
  if (e0 < 2 * NT * D) {                      // the new rows as stored
    uint16_t* dst = ne < D ? &kn_s[ns][ne] : &vn_s[ns][ne - D];
    if (NT == 1 && a.kv_new && n >= chunk0 && n < chunk0 + CP)   // staged for the combine's scatter
      st16(a.kv_new + (((long long)b * 2 + (ne < D ? 0 : 1)) * a.nkv + g) * D + (ne & (D - 1)), nv);
    if constexpr (FP8) {
      const float scale = ne < D ? a.k_scale[0] : a.v_scale[0];
      u32x4_t v;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[k] = e4m3_to_bf16(fp8_quant(bf_lo(nv[k]), scale)) | (e4m3_to_bf16(fp8_quant(bf_hi(nv[k]), scale)) << 16);
      st16(dst, v);
    } else {
      st16(dst, nv);
    }
  }
  __syncthreads();
  // head element of slot 0 of k step kk of this lane (A and B operands alike)
  auto d_of = [&](int kk) { return FP8 ? q4 * (D / 4) + 8 * kk : 32 * kk + 8 * q4; };
  u32x4_t qf[NK];
#pragma unroll
  for (int kk = 0; kk < NK; ++kk)
    qf[kk] = col < GQA ? ld16(&q_s[col][d_of(kk)]) : u32x4_t{0u, 0u, 0u, 0u};

  f32x4_t o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;               // head col: running max, this lane's share of the sum

  for (; st < nst; st += kStWaves) {
    const int p0 = chunk0 + st * kStStep;
    const bool edge = p0 + kStStep > n;       // holds new tokens or positions past them (uniform)
    // ---- scores ----
    float sc[2][4];
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      u32x4_t kf[NK];
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) {
        if constexpr (FP8) kf[kk] = fp8x8_to_bf16(kr[u][kk / 2][(kk & 1) * 2], kr[u][kk / 2][(kk & 1) * 2 + 1]);
        else kf[kk] = kr[u][kk];
      }
      if (edge) {
        const int t = p0 + 16 * u + col;
        if (t >= n && t < total) {
#pragma unroll
          for (int kk = 0; kk < NK; ++kk) kf[kk] = ld16(&kn_s[t - n][d_of(kk)]);
        }
      }
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) acc = mfma16x16x32(kf[kk], qf[kk], acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = a.round_qwen ? rbf(rbf(acc[i]) * a.scale) : acc[i] * a.scale;
        bool ok = p0 + 16 * u + 4 * q4 + i < total;
        if constexpr (MASK) ok = ok && ((bits >> (4 * u + i)) & 1u);
        sc[u][i] = ok ? v : -INFINITY;
        mx = fmaxf(mx, sc[u][i]);
      }
    }
    // ---- the next step's K rows (and the mask after it) ----
    const int sn = st + kStWaves;
    bool live_n = sn < nst;
    if constexpr (MASK) {
      bits_n = mask_bits();
      live_n = live_n && __any(bits_n != 0);
      load_mask(min(sn + kStWaves, nst - 1));
    }
    blkn[0] = tile_blk(sn, 0);
    blkn[1] = tile_blk(sn, 1);
    load_k(sn, blkn, live_n);
    // ---- online softmax, per head (lanes sharing col) ----
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);
    if (__any(mn > m)) {                      // uniform: a maximum moved
      const float alpha = m == -INFINITY ? 0.f : expf(m - mn);
      l *= alpha;
      m = mn;
      // o rows are heads 4 q4 + i: their factors from the lanes holding them
      float al[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) al[i] = __shfl(alpha, 4 * q4 + i, 64);
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[dt][i] *= al[i];
    }
    u32x4_t ph, pm, pl;                       // p = ph (+ pm + pl for FP8: exact)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float p[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[i] = m == -INFINITY ? 0.f : expf(sc[u][i] - m);
        l += p[i];
      }
      ph[2 * u] = pack2bf(p[0], p[1]);
      ph[2 * u + 1] = pack2bf(p[2], p[3]);
      if constexpr (FP8) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int j = 2 * u + k;
          const float r0 = p[2 * k] - bf_lo(ph[j]), r1 = p[2 * k + 1] - bf_hi(ph[j]);
          pm[j] = pack2bf(r0, r1);
          pl[j] = pack2bf(r0 - bf_lo(pm[j]), r1 - bf_hi(pm[j]));
        }
      }
    }
    // ---- P . V ----
    if (edge) {   // new tokens' rows from LDS, rows past them zero
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int t = p0 + 16 * u + 4 * q4 + j;
          if (t >= n) {
#pragma unroll
            for (int e = 0; e < VD; ++e) {
              if constexpr (FP8) vr[u][j][e] = 0u;   // (e4m3 new rows: added below as bf16)
              else vr[u][j][e] = t < total ? *reinterpret_cast<const uint32_t*>(&vn_s[t - n][col * NDT + 2 * e]) : 0u;
            }
          }
        }
    }
    if constexpr (FP8) {
      // two head elements (half a dword of each row) at a time
#pragma unroll
      for (int e = 0; e < 2 * VD; ++e) {
        float x[2][4][2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const f32x2_t v = (e & 1) ? cvt2_fp8_hi(vr[u][j][e >> 1]) : cvt2_fp8_lo(vr[u][j][e >> 1]);
            x[u][j][0] = v[0];
            x[u][j][1] = v[1];
            if (edge) {
              const int t = p0 + 16 * u + 4 * q4 + j;
              if (t >= n && t < total) {
#pragma unroll
                for (int k = 0; k < 2; ++k) x[u][j][k] = bf2f(vn_s[t - n][col * NDT + 2 * e + k]);
              }
            }
          }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const u32x4_t bop = {pack2bf(x[0][0][k], x[0][1][k]), pack2bf(x[0][2][k], x[0][3][k]),
                               pack2bf(x[1][0][k], x[1][1][k]), pack2bf(x[1][2][k], x[1][3][k])};
          o[2 * e + k] = mfma16x16x32(ph, bop, o[2 * e + k]);
          o[2 * e + k] = mfma16x16x32(pm, bop, o[2 * e + k]);
          o[2 * e + k] = mfma16x16x32(pl, bop, o[2 * e + k]);
        }
      }
    } else {
      // the operand's 16-bit halves from two V rows by one byte permute per dword
      // (selector 0x05040100: bytes 0-1 of each row; 0x07060302: bytes 2-3)
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        const int e = dt >> 1;
        const uint32_t sel = (dt & 1) ? 0x07060302u : 0x05040100u;
        u32x4_t bop;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          bop[2 * u] = __builtin_amdgcn_perm(vr[u][1][e], vr[u][0][e], sel);
          bop[2 * u + 1] = __builtin_amdgcn_perm(vr[u][3][e], vr[u][2][e], sel);
        }
        o[dt] = mfma16x16x32(ph, bop, o[dt]);
      }
    }
    load_v(sn, blkn, live_n);
    if constexpr (MASK) bits = bits_n;
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);

  // ---- merge the waves into this chunk's partial ----
  if (lane < 16) { m_s[w][lane] = m; l_s[w][lane] = l; }
#pragma unroll
  for (int i = 0; i < 4; ++i) {               // o[dt][i] = O[head 4 q4 + i][d = col NDT + dt]
    const int h = 4 * q4 + i;
    if (h < GQA)
#pragma unroll
      for (int q = 0; q < NDT / 4; ++q)
        *reinterpret_cast<f32x4_t*>(&o_s[w][h][col * NDT + 4 * q]) =
            f32x4_t{o[4 * q][i], o[4 * q + 1][i], o[4 * q + 2][i], o[4 * q + 3][i]};
  }
  __syncthreads();
  for (int idx = threadIdx.x * 4; idx < GQA * D; idx += 64 * kStWaves * 4) {
    const int h = idx / D, d = idx % D;
    float M = -INFINITY;
#pragma unroll
    for (int q = 0; q < kStWaves; ++q) M = fmaxf(M, m_s[q][h]);
    float L = 0.f;
    f32x4_t O = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < kStWaves; ++q) {
      const float f = (m_s[q][h] == -INFINITY) ? 0.f : expf(m_s[q][h] - M);
      L += l_s[q][h] * f;
      O += *reinterpret_cast<const f32x4_t*>(&o_s[q][h][d]) * f;
    }
    const long long slot = ((long long)b * a.nq + g * GQA + h) * a.n_chunks + c;
    *reinterpret_cast<f32x4_t*>(a.part_o + slot * D + d) = O;
    if (d == 0) *reinterpret_cast<float2*>(a.part_ml + slot * 2) = float2{M, L};
  }
}

namespace {

// Non-temporal loads where one layer's cache is at least twice the 256 MB memory-side
// cache.  Whole steps of 6 layers, always / this rule / never: 64 sequences x 8128
// 2.29-2.40 / 2.29-2.38 / 2.45 ms, 32 x 8128 1.79-1.81 / 1.80-1.81 / 1.86 ms.  Smaller
// caches gain too within a model, where the other layers' caches lie between two uses
// (64 x 2048 1.81-1.84 / 1.82-1.86 / 1.84-1.85 ms; 64-wide heads, 32 x 4096, 4 layers,
// 1001 / 1009 us); the line is where it is for a layer called again and again on one
// cache (16 x 8128: 231 / 223 / 224 us).
template <int D, int GQA>
hipError_t stream_launch(const AttnArgs& a, hipStream_t s) {
  const dim3 grid(a.nkv, a.n_chunks, a.B), block(64 * kStWaves);
  if (a.kv_fp8)
    return a.mask ? timed_launch(attn_stream_kernel<D, GQA, true, true, false>, grid, block, 0, s, a)
                  : timed_launch(attn_stream_kernel<D, GQA, true, false, false>, grid, block, 0, s, a);
  if (a.mask) return timed_launch(attn_stream_kernel<D, GQA, false, true, false>, grid, block, 0, s, a);
  const long long seqs = a.prefill ? 1 : a.B / (a.s_tkg > 1 ? a.s_tkg : 1);
  const bool nt = 4LL * seqs * a.nkv * a.S_max * D >= 512LL << 20;   // K and V, 2 bytes each
  return nt ? timed_launch(attn_stream_kernel<D, GQA, false, false, true>, grid, block, 0, s, a)
            : timed_launch(attn_stream_kernel<D, GQA, false, false, false>, grid, block, 0, s, a);
}

}  // namespace

// Whole 16-position tiles per cache block, 16-byte aligned cache rows, prepared
// heads; chunks of whole steps.  A sliding-window ring (one chunk of at most W
// rows) keeps attn_fused_kernel: at 32 sequences x 128 rows it takes 14 us there
// and 6 here, 1 % of such a model's step, and its rounding (probabilities against
// the maximum of 64 positions per wave) stays as the routing checks know it.
bool attn_stream_ok(const AttnArgs& a) {
  const int nt = a.s_tkg > 1 ? a.s_tkg : 1;
  const int gqa = a.nkv > 0 ? a.nq / a.nkv : 0;
  return a.prep && !a.k_transposed && a.window == 0 && (a.d == 64 || a.d == 128) && gqa * a.nkv == a.nq &&
         (gqa == 1 || gqa == 2 || gqa == 4 || gqa == 8 || gqa == 16) && nt <= kStMaxNew && a.B % nt == 0 &&
         a.chunk > 0 && a.chunk % kStStep == 0 && (!a.block_table || a.blk_len % 16 == 0) &&
         (!a.kv_fp8 || (a.k_scale && a.v_scale)) && a.n_chunks <= 65535 && a.B <= 65535 &&
         ((reinterpret_cast<uintptr_t>(a.k_cache) | reinterpret_cast<uintptr_t>(a.v_cache)) & 15) == 0;
}

// Positions per block where the launch's chunk is 256 (attn_chunk_for: the grid
// covers the chip): 512 while that still leaves 2048 blocks -- half the partials
// for the combine, twice the steps to pipeline.  (The workspace is sized for the
// smaller chunk.)
int attn_stream_chunk(const AttnArgs& a) {
  const int nt = a.s_tkg > 1 ? a.s_tkg : 1;
  const long long blocks = (long long)((a.S_max + nt + 511) / 512) * a.nkv * a.B;
  return a.chunk == 256 && blocks >= 2048 ? 512 : a.chunk;
}

hipError_t attn_stream_launch(const AttnArgs& a, hipStream_t s) {
  if (!attn_stream_ok(a)) return hipErrorInvalidValue;
  const int gqa = a.nq / a.nkv;
#define MKD_ST(D_)                                    \
  switch (gqa) {                                      \
    case 1: return stream_launch<D_, 1>(a, s);        \
    case 2: return stream_launch<D_, 2>(a, s);        \
    case 4: return stream_launch<D_, 4>(a, s);        \
    case 8: return stream_launch<D_, 8>(a, s);        \
    case 16: return stream_launch<D_, 16>(a, s);      \
  }
  if (a.d == 128) { MKD_ST(128) }
  else { MKD_ST(64) }
#undef MKD_ST
  return hipErrorInvalidValue;
}

}  // namespace mkd
