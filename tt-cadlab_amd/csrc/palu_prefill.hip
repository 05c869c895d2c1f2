// Prefill attention of one layer over whole prompts: causal attention of every prompt position over the
// prompt's own latents, as near to exact as an fp32 attention (fp32 K, V, probabilities and sums, score operands
// of 22 bits; below), which PaluAttention's prefill computed before (reference palu_tt/attention.py:380-480). Replaces the
// chain of torch ops (casts, einsum rebuilds, RoPE, head repeats, fp32 SDPA) with three launches over the QKV
// projection's bf16 output rows:
//   1. palu_latent_fill: the new latents (or, on the stock K path, the rotated keys) into the caches;
//   2. palu_prefill_rebuild_kernel: K = RoPE(lat u_k) in fp32 (bf16 MFMA, whose products are exact, fp32
//      accumulation), and V: the latent rows themselves where V stays latent, or lat u_v in fp32;
//   3. palu_prefill_attn_kernel: flash attention.
//
// Precision on 16-bit matrix cores. Scores: q and K are each the sum of two fp16 planes of their value over a power-of-two
// scale (plane_scale: one per query row and one per key, applied again to the scores), 22 bits, and a product is
// three MFMAs, hm + mh + hh. Probabilities (and a rebuilt V) are the sum of three bf16 planes h + m + l (24
// bits, and bf16 has fp32's range); with a V latent, which is exactly bf16, a product is three MFMAs, between two such
// sums six (terms below 2^-24 dropped). All sums are fp32. Measured against 64 bits over 17 to 4096 positions, ranks 32 to
// 512 and scores of spread 1 and 4, the result before its bf16 rounding is off by 2.3e-7 to 1.06e-6 (relative 2-norm);
// with three bf16 planes and six MFMAs for the scores as well it is 2.5e-7 to 1.29e-6 (twice as many fp32 additions),
// and the fp32 SDPA chain that the kernels replace 3.3e-7 to 1.76e-6.
//
// With per-head latents V is never rebuilt: softmax(q K^T) (v_lat u_v) = (softmax(q K^T) v_lat) u_v, so the
// probabilities multiply the bf16 latent rows (three MFMAs over r_v columns instead of six over 128) and u_v
// is applied once per query at the end.
//
// Per query head and (query, key) pair 3 x 128 + 3 x r_v multiply-adds, 3 x 128 + 6 x 128 where V is rebuilt.
#include "palu_kernel.h"

#include <algorithm>

namespace {

constexpr int PF_ROWS = 256;              // query rows (position, head of the KV group) per workgroup
constexpr int PF_KTILES = 16;             // K tiles of a 32-key record: 2 planes x 2 half-blocks x 4 dim blocks

struct PrefillArgs {
  const __bf16* x;                        // QKV projection rows [U * S][ldx]
  long long ldx;
  int U, S, nkv, rep, hpg;
  int k_off, k_gs, r_k, full_k;           // K latent columns (full_k: the whole rotated-later heads)
  int v_off, v_gs, r_v;
  const __bf16* u_k;                      // [nkv][r_k][128]
  const __bf16* u_v;                      // [nkv][r_v][128] (v_split, or the up-projection), or null
  const float* cos_t;
  const float* sin_t;
  int table_rows;
  float qscale;                           // softmax scale * log2 e
  __bf16* rec;                            // records [U * nkv][nblk][tiles][64][8] (K tiles fp16, V tiles bf16)
  float* ksc;                             // power-of-two scales of the keys' planes [U * nkv][nblk][32]
  __bf16* uvt;                            // u_v^T tiles [nkv][KBV][8][64][8] (up-projection)
  __bf16* out;                            // [U * S][ldo]
  long long ldo;
  int nblk, tiles;
};

// rope_meta of four values, the table read in 16 bytes (its columns come in equal pairs).
__device__ __forceinline__ void rope4(float (&v)[4], const float* cos_t, const float* sin_t, int pr, int c) {
  const f32x4 cs = *reinterpret_cast<const f32x4*>(cos_t + (long long)pr * HD + c);
  const f32x4 sn = *reinterpret_cast<const f32x4*>(sin_t + (long long)pr * HD + c);
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    const float x0 = v[i], x1 = v[i + 1];
    v[i] = fmaf(x0, cs[i], -(x1 * sn[i]));
    v[i + 1] = fmaf(x1, cs[i], x0 * sn[i]);
  }
}

// x = h + m + l in bf16 planes.
__device__ __forceinline__ void split3(float x, __bf16& h, __bf16& m, __bf16& l) {
  h = (__bf16)x;
  const float r = x - (float)h;
  m = (__bf16)r;
  l = (__bf16)(r - (float)m);
}

__device__ __forceinline__ void split3x8(const float (&v)[8], bf16x8& h, bf16x8& m, bf16x8& l) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    __bf16 a, b, c;
    split3(v[j], a, b, c);
    h[j] = a;
    m[j] = b;
    l[j] = c;
  }
}

// x = s (h + m) with fp16 planes h, m of x / s: s a power of two that puts the largest magnitude of the key or query that
// x belongs to (amax) in [2^14, 2^15), so that the planes hold 22 bits of every value above amax 2^-17 (and an
// absolute 2^-39 amax of the rest). Each key has its own scale: with one for the 32 keys of a record (until then 16
// multiplications a record and lane fewer: 4096 positions at r 64 / 64 323.8 us against 325.3, two prompts of 777 with
// grouped latents 110.1, 111.3) a key 2^24 times the others left these 1e-3 of error in their scores, and an infinite
// one made them NaN. amax is that of the finite values; 0 gives s = 2^-15.
__device__ __forceinline__ float plane_scale(float amax, float& inv) {
  const int e = max(-100, __builtin_amdgcn_frexp_expf(amax)) - 15;   // at most 128 - 15: inv is a normal number
  inv = __builtin_amdgcn_ldexpf(1.f, -e);
  return __builtin_amdgcn_ldexpf(1.f, e);
}

// A score is (sum of plane products) x key scale x row scale; between the two products it carries this power of two, which
// keeps it and both factors in range: keys up to 2^122 in all 128 dims at once (2^127 in a few) and any bf16 query.
constexpr float KEY_SCALE = 0x1p-18f;
constexpr float INF = __builtin_inff();

__device__ __forceinline__ void split2x8(const float (&v)[8], float inv, f16x8& h, f16x8& m) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float y = v[j] * inv;
    h[j] = (_Float16)y;
    m[j] = (_Float16)(y - (float)h[j]);
  }
}

// Position of operand column nn of half-block c of a 32-position block (the K-tile order of the caches): the
// scores of tile c then leave lane (n, g) with keys 8 g + 4 c .. + 3, so the two tiles together are the eight
// consecutive keys of the PV product's operand.
__device__ __forceinline__ int blk_pos(int nn, int c) { return 8 * (nn >> 2) + 4 * c + (nn & 3); }

// Records of one (user, KV head, 32-position block): fp16 K planes as MFMA operand tiles [plane][c][kb] (lane (n, g) of
// tile (c, kb) holds dims 32 kb + {4 g .. + 3, 16 + 4 g .. + 3} of position blk_pos(n, c)) and V tiles behind them
// (tile mt, lane (m, g): positions 8 g .. + 7 of column 16 mt + m; three planes of 8 tiles when V is rebuilt).
// Positions past the prompt are zero. blockIdx.y 0 writes K, 1 writes V; a wave takes one block. u_k / u_v go
// through LDS 64 ranks at a time, transposed. Bound by memory and latency (the rebuild is S x r x 128 products a
// head, against S / 2 of them per query for the attention).
constexpr int PF_RC = 64;                 // ranks per staged chunk
constexpr int PF_US = PF_RC + 8;          // its padded row

template <bool VSPLIT>
__global__ __launch_bounds__(256) void palu_prefill_rebuild_kernel(const PrefillArgs a) {
  __shared__ __attribute__((aligned(16))) __bf16 ut[HD * PF_US];
  const bool isv = blockIdx.y == 1;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nq = (a.nblk + 3) >> 2;
  const int uk = blockIdx.x / nq, kvh = uk % a.nkv, u = uk / a.nkv;
  const int jb = (blockIdx.x - uk * nq) * 4 + w;
  const bool live = jb < a.nblk;          // uniform per wave; every wave stays for the barriers
  const __bf16* xu = a.x + (long long)u * a.S * a.ldx;
  __bf16* rec = a.rec + ((long long)uk * a.nblk + (live ? jb : 0)) * a.tiles * 512;
  const int grp = kvh / a.hpg;

  if (isv && !VSPLIT) {                   // V stays latent: a transposing copy, and u_v^T for the up-projection
    if (live && !a.u_v) {                 // whole V heads: element by element, so that a non-finite value stays in its column
      for (int mt = 0; mt < 8; ++mt) {
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int p = 32 * jb + 8 * g + j;
          const __bf16 v = xu[(long long)min(p, a.S - 1) * a.ldx + a.v_off + (long long)grp * a.v_gs + 16 * mt + n];
          o[j] = p < a.S ? v : (__bf16)0.f;
        }
        *reinterpret_cast<bf16x8*>(rec + ((PF_KTILES + mt) * 64 + lane) * 8) = o;
      }
    } else if (live) {
      // 32 columns at a time: rows in 16-byte pieces (operand order, position blk_pos(n, c)), regrouped into the two
      // 16-column tiles by products with an identity tile, which are exact (a non-finite value spreads over them, as it does
      // over the head in the product with u_v). Element loads and the table in 4-byte loads took 5 us longer (three prompts of
      // 200 42 -> 37 us in all, four of 512 71 -> 67).
      bf16x8 id[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j) id[h][j] = (8 * g + j == 16 * h + n) ? (__bf16)1.0f : (__bf16)0.0f;
      const __bf16* xr[2];
      bool in[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int p = 32 * jb + blk_pos(n, c);
        in[c] = p < a.S;
        xr[c] = xu + (long long)min(p, a.S - 1) * a.ldx + a.v_off + (long long)grp * a.v_gs;
      }
      bf16x8 x[4][2];                     // r_v <= 128 here
#pragma unroll
      for (int vb = 0; vb < 4; ++vb)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int col = 32 * vb + 8 * g;
          x[vb][c] = *reinterpret_cast<const bf16x8*>(xr[c] + (col < a.r_v ? col : 0));
          if (!in[c]) x[vb][c] = bf16x8{};
        }
#pragma unroll
      for (int mt = 0; mt < 8; ++mt) {
        if (16 * mt >= a.r_v) continue;
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
        const bf16x8 o = pack8(mfma16(x[mt >> 1][0], id[mt & 1], z), mfma16(x[mt >> 1][1], id[mt & 1], z));
        *reinterpret_cast<bf16x8*>(rec + ((PF_KTILES + mt) * 64 + lane) * 8) = o;
      }
    }
    if (a.uvt && u == 0 && blockIdx.x == uk * nq) {
      // lane (m, g) of tile (kb, dt), element j: u_v[32 kb + 16 (j / 4) + 4 g + j % 4][16 dt + m], the rank order in
      // which the accumulated O_lat sits in registers; zero past r_v
      const int kbv = (a.r_v + 31) / 32;
      for (int t = w; t < kbv * 8; t += 4) {
        const int kb = t >> 3, dt = t & 7;
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int r = 32 * kb + 16 * (j >> 2) + 4 * g + (j & 3);
          o[j] = r < a.r_v ? a.u_v[((long long)kvh * a.r_v + min(r, a.r_v - 1)) * HD + 16 * dt + n] : (__bf16)0.f;
        }
        *reinterpret_cast<bf16x8*>(a.uvt + (((long long)kvh * kbv * 8 + t) * 64 + lane) * 8) = o;
      }
    }
    return;
  }

  const int r_all = isv ? a.r_v : a.r_k;
  const int off = isv ? a.v_off + grp * a.v_gs : a.k_off + grp * a.k_gs;
  const __bf16* um = (isv ? a.u_v : a.u_k) + (long long)kvh * r_all * HD;
  int p[2];                               // this lane's positions
  const __bf16* xr[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    p[c] = 32 * jb + blk_pos(n, c);
    xr[c] = xu + (long long)min(p[c], a.S - 1) * a.ldx + off;
  }
  f32x4 acc[2][8];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  if (!isv && a.full_k) {                 // the projection's own K heads
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const bf16x4 v = *reinterpret_cast<const bf16x4*>(xr[c] + 16 * t + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[c][t][i] = p[c] < a.S ? (float)v[i] : 0.f;
      }
  } else {
    for (int r0 = 0; r0 < r_all; r0 += PF_RC) {
      __syncthreads();
      for (int e = tid; e < PF_RC * (HD / 8); e += 256) {
        const int rr = e & (PF_RC - 1), d0 = (e / PF_RC) * 8;
        const bf16x8 v = r0 + rr < r_all ? *reinterpret_cast<const bf16x8*>(um + (long long)(r0 + rr) * HD + d0) : bf16x8{};
#pragma unroll
        for (int j = 0; j < 8; ++j) ut[(d0 + j) * PF_US + rr] = v[j];
      }
      __syncthreads();
#pragma unroll
      for (int kb = 0; kb < PF_RC / 32; ++kb) {
        const int rr = r0 + 32 * kb + 8 * g;
        bf16x8 lat[2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
          lat[c] = (rr < r_all && p[c] < a.S) ? *reinterpret_cast<const bf16x8*>(xr[c] + rr) : bf16x8{};
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const bf16x8 uu = *reinterpret_cast<const bf16x8*>(ut + (16 * t + n) * PF_US + 32 * kb + 8 * g);
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[c][t] = isv ? mfma16(lat[c], uu, acc[c][t]) : mfma16(uu, lat[c], acc[c][t]);
        }
      }
    }
  }
  if (!live) return;
  if (!isv) {
    // lane (n, g), tile c: dims 16 t + 4 g + i of position blk_pos(n, c); two tiles make one operand slot
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int pr = min(p[c], a.table_rows - 1);
      float amax = 0.f;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        float q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = acc[c][t][i];
        rope4(q, a.cos_t, a.sin_t, pr, 16 * t + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[c][t][i] = q[i];
          amax = fmaxf(amax, fabsf(q[i]));
        }
      }
      amax = wave_max_xor48(amax);                              // over the key's four lanes
      const bool inf = amax == INF;
      if (__any(inf)) {
        float fin = 0.f;
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) fin = fmaxf(fin, fabsf(acc[c][t][i]) < INF ? fabsf(acc[c][t][i]) : 0.f);
        fin = wave_max_xor48(fin);
        amax = inf ? fin : amax;
      }
      float inv;
      const float sc = plane_scale(amax, inv);
      if (g == 0) a.ksc[((long long)uk * a.nblk + jb) * BLK + blk_pos(n, c)] = sc * KEY_SCALE;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = acc[c][2 * kb + (i >> 2)][i & 3];
        f16x8 h, m;
        split2x8(v, inv, h, m);
        if (inf) {
          // An infinite value goes to the m plane alone, which meets only the query's h plane: its score is then
          // infinite, or NaN where infinities of both signs meet, as the product in fp32 is.
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (fabsf(v[j]) == INF) {
              h[j] = (_Float16)0.f;
              m[j] = (_Float16)v[j];
            }
        }
        __bf16* o = rec + ((c * 4 + kb) * 64 + lane) * 8;
        *reinterpret_cast<f16x8*>(o) = h;
        *reinterpret_cast<f16x8*>(o + 8 * 512) = m;
      }
    }
  } else {
    // lane (n, g), tile t: column 16 t + n at positions 8 g + 4 c + i
    bf16x8 h, m, l;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      float v[8];
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[4 * c + i] = acc[c][t][i];
      split3x8(v, h, m, l);
      __bf16* o = rec + ((PF_KTILES + t) * 64 + lane) * 8;
      *reinterpret_cast<bf16x8*>(o) = h;
      *reinterpret_cast<bf16x8*>(o + 8 * 512) = m;
      *reinterpret_cast<bf16x8*>(o + 16 * 512) = l;
    }
  }
}

// Flash attention over the records. A workgroup owns PF_ROWS rows of one (user, KV head), a row being one
// (position, query head of the group) in position-major order, so the group's heads share every K and V tile. A
// wave owns NG column groups of 16 rows; its rotated, scaled query sits in registers as two planes. Each 32-key
// record is copied to LDS once per workgroup (three buffers, one barrier a record: record j + 2 is loaded during record j
// and written at its end, so that the first K tiles of j + 1 can be read before the barrier) and every K tile read from LDS
// feeds up to 2 NG MFMAs. K tiles are read one dim block ahead of their products and V tiles ahead of the softmax (two
// buffers and reads where the compiler put them: 4096 positions at r 64 / 64 312 -> 309 us with the rebuild, 2048 at 64 /
// 128 183 -> 172, one box; 320 to 325 and 170 on others, with a scale to every key). Running half of the waves half a record behind the others, so that one half's softmax meets the other's
// products, was slower (323 us). At 4096 positions the matrix cores are busy 46 % and the vector ALU 38 % of the time: a
// softmax of eight keys costs a lane about 110 instructions beside 36 MFMAs. Scores are computed transposed
// (keys x rows), so a lane holds eight keys of one row per column group: softmax in the exp2 domain with a lazily
// refreshed maximum (cross-lane work only when a score passes it by 2^8), probabilities split into planes in
// place, and they are the PV product's operand as they stand.
// The workgroups of one head have ids a multiple of U * nkv apart, longest rows first: with 8 KV heads a head's
// records stay in one XCD's L2, and the short rows fill in behind the long ones.
template <int VT, bool VSPLIT, bool UP, int NW, int NG>
__global__ __launch_bounds__(NW * 64, NW == 8 ? 2 : 1) void palu_prefill_attn_kernel(const PrefillArgs a) {
  static_assert(NW * NG * 16 == PF_ROWS, "rows per workgroup");
  constexpr int NT = PF_KTILES + (VSPLIT ? 3 * VT : VT);
  constexpr int LPW = (NT + NW - 1) / NW;                  // tiles a wave copies per record
  extern __shared__ __attribute__((aligned(16))) char smem[];
  bf16x8* lds = reinterpret_cast<bf16x8*>(smem);

  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int heads = a.U * a.nkv;
  const int nqb = (int)(((long long)a.S * a.rep + PF_ROWS - 1) / PF_ROWS);
  const int uk = blockIdx.x % heads, kvh = uk % a.nkv, u = uk / a.nkv;
  const int qb = nqb - 1 - blockIdx.x / heads;
  const int rows = a.S * a.rep;
  const int row0 = qb * PF_ROWS + w * 16 * NG;

  int pos[NG];
  f16x8 q[2][NG][4];
  float qsc[NG];
#pragma unroll
  for (int gr = 0; gr < NG; ++gr) {
    const int row = min(row0 + 16 * gr + n, rows - 1);     // rows past the prompt repeat its last one, unstored
    pos[gr] = row / a.rep;
    const int head = kvh * a.rep + (row - pos[gr] * a.rep);
    const __bf16* xq = a.x + ((long long)u * a.S + pos[gr]) * a.ldx + (long long)head * HD;
    const int pr = min(pos[gr], a.table_rows - 1);
    float v[4][8], amax = 0.f;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int d = 16 * (2 * kb + hh) + 4 * g;
        const bf16x4 xv = *reinterpret_cast<const bf16x4*>(xq + d);
        float t[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) t[i] = (float)xv[i];
        rope4(t, a.cos_t, a.sin_t, pr, d);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[kb][4 * hh + i] = t[i] * a.qscale;
          amax = fmaxf(amax, fabsf(v[kb][4 * hh + i]));
        }
      }
    float inv;
    qsc[gr] = plane_scale(wave_max_xor48(amax), inv) / KEY_SCALE;   // over the row's four lanes
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) split2x8(v[kb], inv, q[0][gr][kb], q[1][gr][kb]);
  }
  // Keys this wave and this workgroup need; rows are position-major, so the first and last rows bound the wave.
  const int w_lo = min(row0, rows - 1) / a.rep, w_hi = min(row0 + 16 * NG - 1, rows - 1) / a.rep;
  const int nst = min(qb * PF_ROWS + PF_ROWS - 1, rows - 1) / a.rep / BLK + 1;

  const bf16x8* rec = reinterpret_cast<const bf16x8*>(a.rec) + (long long)uk * a.nblk * NT * 64 + lane;
  bf16x8 st[LPW];
  auto load = [&](int j) {
#pragma unroll
    for (int i = 0; i < LPW; ++i) st[i] = rec[((long long)j * NT + min(w + i * NW, NT - 1)) * 64];
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int i = 0; i < LPW; ++i)
      lds[(buf * NT + min(w + i * NW, NT - 1)) * 64 + lane] = st[i];   // past the last tile: that one again, the same bytes
  };

  f32x4 O[NG][VT];
  float m_run[NG], l_run[NG];
#pragma unroll
  for (int gr = 0; gr < NG; ++gr) {
    m_run[gr] = NEG_INF;
    l_run[gr] = 0.f;
#pragma unroll
    for (int t = 0; t < VT; ++t) O[gr][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // Workgroup barrier over LDS: this wave's LDS writes and reads are done, its global loads stay in flight.
  auto barrier = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  load(0);
  put(0);
  load(min(1, nst - 1));
  put(1);
  barrier();
  // One dim block's K tiles (both planes and half-blocks), read a block ahead of their products; the scheduling fences
  // keep the compiler from sinking each read to its use.
  f16x8 kt2[2][2][2];
  auto fence = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
  auto read_k = [&](f16x8 (&x)[2][2], const bf16x8* kt, int kb) {
#pragma unroll
    for (int pl = 0; pl < 2; ++pl)
#pragma unroll
      for (int c = 0; c < 2; ++c) x[pl][c] = __builtin_bit_cast(f16x8, kt[(8 * pl + c * 4 + kb) * 64]);
  };
  // The scales of this lane's keys, loaded before the record's barrier.
  const f32x4* kscale = reinterpret_cast<const f32x4*>(a.ksc + (long long)uk * a.nblk * BLK + 8 * g);
  f32x4 ksc[2] = {kscale[0], kscale[1]};
  int buf = 0;
  read_k(kt2[0], lds + lane, 0);
  for (int j = 0; j < nst; ++j) {
    const int base = j * BLK;
    const bool live = base <= w_hi;       // uniform per wave
    const bf16x8* kt = lds + buf * NT * 64 + lane;
    load(min(j + 2, nst - 1));
    fence();
    f32x4 s[NG][2];
#pragma unroll
    for (int gr = 0; gr < NG; ++gr)
#pragma unroll
      for (int c = 0; c < 2; ++c) s[gr][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (live) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        if (kb < 3) read_k(kt2[(kb + 1) & 1], kt, kb + 1);
        fence();
        // km qh + kh qm + kh qh
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int gr = 0; gr < NG; ++gr) s[gr][c] = mfma16(kt2[kb & 1][t == 0][c], q[t == 1][gr][kb], s[gr][c]);
        fence();
      }
    }
    const bf16x8* vt = kt + PF_KTILES * 64;
    bf16x8 vh[VSPLIT ? 1 : VT];
    if constexpr (!VSPLIT) {              // the V tiles, in flight during the softmax
#pragma unroll
      for (int t = 0; t < VT; ++t) vh[t] = vt[t * 64];
      fence();
    }
    if (live) {
      if (base + BLK - 1 > w_lo) {                          // the diagonal: keys past a row's own position
#pragma unroll
        for (int gr = 0; gr < NG; ++gr)
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (base + 8 * g + 4 * c + i > pos[gr]) s[gr][c][i] = NEG_INF;
      }
      float bm[NG];                                         // the keys' scales here, the row's in the exponent
      bool up = false;
#pragma unroll
      for (int gr = 0; gr < NG; ++gr) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[gr][c][i] *= ksc[c][i];
        bm[gr] = max8(s[gr][0], s[gr][1]) * qsc[gr];
        up = up || bm[gr] > m_run[gr] + LAZY_RESCALE_LOG2;
      }
      if (__any(up)) {
#pragma unroll
        for (int gr = 0; gr < NG; ++gr) {
          const float mn = fmaxf(m_run[gr], wave_max_xor48(bm[gr]));
          const float alpha = m_run[gr] == NEG_INF ? 0.f : __builtin_amdgcn_exp2f(m_run[gr] - mn);
#pragma unroll
          for (int t = 0; t < VT; ++t) O[gr][t] *= alpha;
          l_run[gr] *= alpha;
          m_run[gr] = mn;
        }
      }
      bf16x8 ph[NG], pm[NG], pl[NG];
#pragma unroll
      for (int gr = 0; gr < NG; ++gr) {
        const float mref = m_run[gr] == NEG_INF ? 0.f : m_run[gr];
        float p[8];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) p[4 * c + i] = __builtin_amdgcn_exp2f(fmaf(s[gr][c][i], qsc[gr], -mref));
        l_run[gr] += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        split3x8(p, ph[gr], pm[gr], pl[gr]);
      }
      fence();
      if constexpr (VSPLIT) {
        // two V tiles (three planes each) at a time, read a pair ahead
        static_assert(VT % 2 == 0, "V tiles are taken in pairs");
        bf16x8 vv[2][3][2];
        auto read_v = [&](bf16x8 (&x)[3][2], int t0) {
#pragma unroll
          for (int pl = 0; pl < 3; ++pl)
#pragma unroll
            for (int t = 0; t < 2; ++t) x[pl][t] = vt[(pl * VT + t0 + t) * 64];
        };
        read_v(vv[0], 0);
#pragma unroll
        for (int t0 = 0; t0 < VT; t0 += 2) {
          const int cur = (t0 >> 1) & 1;
          if (t0 + 2 < VT) read_v(vv[cur ^ 1], t0 + 2);
          fence();
          auto pv = [&](int pl, const bf16x8 (&pp)[NG]) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
              for (int gr = 0; gr < NG; ++gr) O[gr][t0 + t] = mfma16(vv[cur][pl][t], pp[gr], O[gr][t0 + t]);
          };
          pv(2, ph);
          pv(0, pl);
          pv(1, pm);
          pv(1, ph);
          pv(0, pm);
          pv(0, ph);
          fence();
        }
      } else {
        // one plane of P over all V tiles before the next: consecutive products have different accumulators
        auto pv = [&](const bf16x8 (&pp)[NG]) {
#pragma unroll
          for (int t = 0; t < VT; ++t)
#pragma unroll
            for (int gr = 0; gr < NG; ++gr) O[gr][t] = mfma16(vh[t], pp[gr], O[gr][t]);
        };
        pv(pl);
        pv(pm);
        pv(ph);
      }
    }
    fence();
    buf = buf == 2 ? 0 : buf + 1;
    put(buf == 2 ? 0 : buf + 1);
#pragma unroll
    for (int c = 0; c < 2; ++c) ksc[c] = kscale[min(j + 1, nst - 1) * (BLK / 4) + c];
    read_k(kt2[0], lds + buf * NT * 64 + lane, 0);   // the next record's first tiles: written a record ago
    barrier();
  }

#pragma unroll
  for (int gr = 0; gr < NG; ++gr) {
    const float inv = 1.f / wave_sum_xor48(l_run[gr]);
    const int row = row0 + 16 * gr + n;
    const int head = kvh * a.rep + (row - pos[gr] * a.rep);
    __bf16* o = a.out + ((long long)u * a.S + pos[gr]) * a.ldo + (long long)head * HD + 4 * g;
    const bool ok = row < rows;
    if constexpr (UP) {
      // O_lat (normalised, fp32 as three planes) times u_v: the accumulators are the operand as they stand
      constexpr int KBV = (VT + 1) / 2;
      f32x4 y[8];
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) y[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < KBV; ++kb) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = O[gr][2 * kb][i] * inv;
          v[4 + i] = 2 * kb + 1 < VT ? O[gr][2 * kb + 1 < VT ? 2 * kb + 1 : 0][i] * inv : 0.f;
        }
        bf16x8 h, m, l;
        split3x8(v, h, m, l);
        const bf16x8* uv = reinterpret_cast<const bf16x8*>(a.uvt) + ((long long)kvh * KBV + kb) * 8 * 64 + lane;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
          const bf16x8 t = uv[dt * 64];
          y[dt] = mfma16(t, l, y[dt]);
          y[dt] = mfma16(t, m, y[dt]);
          y[dt] = mfma16(t, h, y[dt]);
        }
      }
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        bf16x4 b;
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = (__bf16)y[dt][i];
        if (ok) *reinterpret_cast<bf16x4*>(o + 16 * dt) = b;
      }
    } else {
#pragma unroll
      for (int t = 0; t < VT; ++t) {
        bf16x4 b;
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = (__bf16)(O[gr][t][i] * inv);
        if (ok) *reinterpret_cast<bf16x4*>(o + 16 * t) = b;
      }
    }
  }
}

template <int VT, bool VSPLIT, bool UP>
int launch_attn(const PrefillArgs& a, hipStream_t s) {
  constexpr int NW = 8, NG = 2;
  auto kern = palu_prefill_attn_kernel<VT, VSPLIT, UP, NW, NG>;
  constexpr int lds = 3 * (PF_KTILES + (VSPLIT ? 3 * VT : VT)) * 1024;
  static bool attr_set = false;
  if (!attr_set) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return fail(PALU_EHIP, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    attr_set = true;
  }
  const long long nqb = ((long long)a.S * a.rep + PF_ROWS - 1) / PF_ROWS;
  hipLaunchKernelGGL(kern, dim3((unsigned)(nqb * a.U * a.nkv)), dim3(NW * 64), lds, s, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? PALU_OK : fail(PALU_EHIP, "prefill attention launch: %s", hipGetErrorString(e));
}

// Cache fill: positions 0 .. n_pos - 1 of cache rows 0 .. users - 1 from the projection's rows. Row-major and K-tile
// caches take 8 columns per thread (rotated first when cos_t is given: whole 128-wide heads); V-tile caches take one
// column of 8 positions per thread, which is one 16-byte slot (element stores where the prompt ends inside it, so
// positions past it keep what they hold).
struct FillArgs {
  __bf16* cache;
  long long c_sb, c_sg;
  const __bf16* src;
  long long ld, s_sg;
  int U, G, n_pos, width;
  const float* cos_t;
  const float* sin_t;
  int table_rows;
};

template <int LAYOUT>
__global__ __launch_bounds__(256) void palu_latent_fill_kernel(const FillArgs a) {
  const int per = LAYOUT == PALU_LAYOUT_TILED_V ? a.width : a.width / 8;
  const int np = LAYOUT == PALU_LAYOUT_TILED_V ? (a.n_pos + 7) / 8 : a.n_pos;
  const long long total = (long long)a.U * a.G * np * per;
  for (long long e = blockIdx.x * 256LL + threadIdx.x; e < total; e += (long long)gridDim.x * 256) {
    const int v = (int)(e % per);
    const long long r = e / per;
    const int g = (int)(r % a.G);
    const long long up = r / a.G;
    const int p = (int)(up % np), u = (int)(up / np);
    __bf16* stream = a.cache + u * a.c_sb + g * a.c_sg;
    if constexpr (LAYOUT == PALU_LAYOUT_TILED_V) {
      const int p0 = 8 * p, cnt = min(8, a.n_pos - p0);
      const __bf16* s = a.src + ((long long)u * a.n_pos + p0) * a.ld + g * a.s_sg + v;
      bf16x8 o = {};
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < cnt) o[j] = s[j * a.ld];
      __bf16* d = stream + tiled_v_offset(p0, v, a.width);
      if (cnt == 8) {
        *reinterpret_cast<bf16x8*>(d) = o;
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (j < cnt) d[j] = o[j];
      }
    } else {
      bf16x8 x = *reinterpret_cast<const bf16x8*>(a.src + ((long long)u * a.n_pos + p) * a.ld + g * a.s_sg + 8 * v);
      if (a.cos_t) {
        float f[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] = (float)x[j];
        rope_meta<8>(f, a.cos_t, a.sin_t, min(p, a.table_rows - 1), 8 * v);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = (__bf16)f[j];
      }
      if constexpr (LAYOUT == PALU_LAYOUT_ROWS) *reinterpret_cast<bf16x8*>(stream + (long long)p * a.width + 8 * v) = x;
      else store_k8(stream, p, 8 * v, a.width, x);
    }
  }
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// V tiles per record: the latent's (V kept latent, up to 128 wide) or three planes of 8.
int v_tiles(int n_kv, int n_groups, int r_v) { return n_kv == n_groups && r_v <= HD ? r_v / 16 : 24; }

bool prefill_shape_ok(int users, int seq, int n_heads, int n_kv, int n_groups, int r_k, int r_v) {
  return users > 0 && seq > 0 && n_kv > 0 && n_heads > 0 && n_heads % n_kv == 0 && n_groups > 0 && n_kv % n_groups == 0 &&
         r_k > 0 && r_k % 16 == 0 && r_v > 0 && r_v % 16 == 0 && (long long)seq * (n_heads / n_kv) < (1LL << 30) &&
         ((long long)seq * (n_heads / n_kv) + PF_ROWS - 1) / PF_ROWS * users * n_kv < (1LL << 30) &&
         (long long)users * n_kv * ((seq + 127) / 128) < (1LL << 30);
}

}  // namespace

extern "C" size_t palu_prefill_workspace_bytes(int users, int seq, int n_heads, int n_kv, int n_groups, int r_k, int r_v) {
  if (!prefill_shape_ok(users, seq, n_heads, n_kv, n_groups, r_k, r_v)) return 0;
  const size_t blocks = (size_t)users * n_kv * ((seq + 31) / 32);
  return blocks * (PF_KTILES + v_tiles(n_kv, n_groups, r_v)) * 1024 + (size_t)n_kv * 4 * 8 * 1024 + blocks * BLK * sizeof(float);
}

extern "C" int palu_prefill_attention(const void* qkv, long long ld, int users, int seq, int n_heads, int n_kv, int n_groups,
                                      int k_col_offset, int r_k, const void* u_k, int v_col_offset, int r_v,
                                      const void* u_v, const float* cos_table, const float* sin_table, int table_rows,
                                      float scale, void* out, long long ld_out, void* workspace, size_t workspace_bytes,
                                      hipStream_t stream) {
  palu::g_err[0] = 0;
  const char* who = "palu_prefill_attention";
  if (!qkv || !cos_table || !sin_table || !out || !workspace) return fail(PALU_EINVAL, "%s: a required pointer is null", who);
  if (!prefill_shape_ok(users, seq, n_heads, n_kv, n_groups, r_k, r_v))
    return fail(PALU_EINVAL, "%s: users %d, seq %d, %d / %d heads, %d groups, r_k %d, r_v %d (ranks multiples of 16)", who,
                users, seq, n_heads, n_kv, n_groups, r_k, r_v);
  const bool per_head = n_kv == n_groups;
  if (!u_k && !(per_head && r_k == HD)) return fail(PALU_EINVAL, "%s: u_k is needed unless K is whole (r_k %d)", who, r_k);
  if (!u_v && !(per_head && r_v == HD)) return fail(PALU_EINVAL, "%s: u_v is needed unless V is whole (r_v %d)", who, r_v);
  if (table_rows < seq) return fail(PALU_EINVAL, "%s: %d table rows for %d positions", who, table_rows, seq);
  const long long cols = std::max({(long long)n_heads * HD, (long long)k_col_offset + (long long)n_groups * r_k,
                                   (long long)v_col_offset + (long long)n_groups * r_v});
  if (k_col_offset < 0 || v_col_offset < 0 || k_col_offset % 8 || v_col_offset % 8 || ld < cols || ld % 8)
    return fail(PALU_EINVAL, "%s: column offsets %d, %d and the row stride %lld must be multiples of 8 inside the row", who,
                k_col_offset, v_col_offset, ld);
  if (ld_out < (long long)n_heads * HD || ld_out % 4)
    return fail(PALU_EINVAL, "%s: output row stride %lld must hold the heads and be a multiple of 4", who, ld_out);
  if (!al16(qkv) || !al16(out) || !al16(workspace) || !al16(cos_table) || !al16(sin_table) || (u_k && !al16(u_k)) ||
      (u_v && !al16(u_v)))
    return fail(PALU_EINVAL, "%s: 16-byte alignment required", who);
  const size_t need = palu_prefill_workspace_bytes(users, seq, n_heads, n_kv, n_groups, r_k, r_v);
  if (workspace_bytes < need)
    return fail(PALU_EINVAL, "%s: workspace of %zu bytes needed (palu_prefill_workspace_bytes), got %zu", who, need, workspace_bytes);

  PrefillArgs a{};
  a.x = static_cast<const __bf16*>(qkv);
  a.ldx = ld;
  a.U = users;
  a.S = seq;
  a.nkv = n_kv;
  a.rep = n_heads / n_kv;
  a.hpg = n_kv / n_groups;
  a.k_off = k_col_offset;
  a.k_gs = a.r_k = r_k;
  a.full_k = u_k == nullptr;
  a.v_off = v_col_offset;
  a.v_gs = a.r_v = r_v;
  a.u_k = static_cast<const __bf16*>(u_k);
  a.u_v = static_cast<const __bf16*>(u_v);
  a.cos_t = cos_table;
  a.sin_t = sin_table;
  a.table_rows = table_rows;
  a.qscale = scale * 1.44269504088896340736f;
  a.out = static_cast<__bf16*>(out);
  a.ldo = ld_out;
  a.nblk = (seq + 31) / 32;
  const bool split = !(per_head && r_v <= HD);
  a.tiles = PF_KTILES + v_tiles(n_kv, n_groups, r_v);
  a.rec = static_cast<__bf16*>(workspace);
  __bf16* uvt = a.rec + (size_t)users * n_kv * a.nblk * a.tiles * 512;
  a.uvt = (split || !u_v) ? nullptr : uvt;
  a.ksc = reinterpret_cast<float*>(uvt + (size_t)n_kv * 4 * 8 * 512);
  const dim3 grid((unsigned)(users * n_kv * ((a.nblk + 3) / 4)), 2);
  if (split) hipLaunchKernelGGL(palu_prefill_rebuild_kernel<true>, grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL(palu_prefill_rebuild_kernel<false>, grid, dim3(256), 0, stream, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(PALU_EHIP, "%s: rebuild launch: %s", who, hipGetErrorString(e));
  if (split) return launch_attn<8, true, false>(a, stream);
  if (!u_v) return launch_attn<8, false, false>(a, stream);
  switch (r_v / 16) {
    case 1: return launch_attn<1, false, true>(a, stream);
    case 2: return launch_attn<2, false, true>(a, stream);
    case 3: return launch_attn<3, false, true>(a, stream);
    case 4: return launch_attn<4, false, true>(a, stream);
    case 5: return launch_attn<5, false, true>(a, stream);
    case 6: return launch_attn<6, false, true>(a, stream);
    case 7: return launch_attn<7, false, true>(a, stream);
    default: return launch_attn<8, false, true>(a, stream);
  }
}

extern "C" int palu_latent_fill(void* cache, long long batch_stride, long long group_stride, const void* src,
                                long long src_row_stride, long long src_group_stride, int users, int n_groups, int n_pos,
                                int seq_len, int width, int cache_layout, const float* cos_table, const float* sin_table,
                                int table_rows, hipStream_t stream) {
  palu::g_err[0] = 0;
  const char* who = "palu_latent_fill";
  if (!cache || !src) return fail(PALU_EINVAL, "%s: a required pointer is null", who);
  if (users <= 0 || n_groups <= 0 || n_pos <= 0 || n_pos > seq_len)
    return fail(PALU_EINVAL, "%s: users %d, groups %d, %d positions of a cache of %d", who, users, n_groups, n_pos, seq_len);
  if (cache_layout != PALU_LAYOUT_ROWS && cache_layout != PALU_LAYOUT_TILED && cache_layout != PALU_LAYOUT_TILED_V)
    return fail(PALU_EINVAL, "%s: cache layout %d", who, cache_layout);
  if (width <= 0 || width % (cache_layout == PALU_LAYOUT_ROWS ? 8 : 16) || (cache_layout != PALU_LAYOUT_ROWS && seq_len % 32))
    return fail(PALU_EINVAL, "%s: width %d (multiples of 8, of 16 when tiled), seq_len %d (of 32 when tiled)", who, width, seq_len);
  if (src_row_stride < width || src_row_stride % 8 || src_group_stride % 8 || batch_stride % 8 || group_stride % 8)
    return fail(PALU_EINVAL, "%s: strides must be multiples of 8", who);
  if (!al16(cache) || !al16(src)) return fail(PALU_EINVAL, "%s: 16-byte alignment required", who);
  if ((cos_table == nullptr) != (sin_table == nullptr) ||
      (cos_table && (width != HD || table_rows < n_pos || cache_layout == PALU_LAYOUT_TILED_V)))
    return fail(PALU_EINVAL, "%s: rotation takes both tables, %d-wide K heads and a table row per position", who, HD);
  const FillArgs a{static_cast<__bf16*>(cache), batch_stride, group_stride, static_cast<const __bf16*>(src), src_row_stride,
                   src_group_stride, users, n_groups, n_pos, width, cos_table, sin_table, table_rows};
  const long long total = cache_layout == PALU_LAYOUT_TILED_V ? (long long)users * n_groups * ((n_pos + 7) / 8) * width
                                                               : (long long)users * n_groups * n_pos * (width / 8);
  const dim3 grid((unsigned)std::min<long long>((total + 255) / 256, 16384));
  if (cache_layout == PALU_LAYOUT_ROWS) hipLaunchKernelGGL(palu_latent_fill_kernel<PALU_LAYOUT_ROWS>, grid, dim3(256), 0, stream, a);
  else if (cache_layout == PALU_LAYOUT_TILED) hipLaunchKernelGGL(palu_latent_fill_kernel<PALU_LAYOUT_TILED>, grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL(palu_latent_fill_kernel<PALU_LAYOUT_TILED_V>, grid, dim3(256), 0, stream, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? PALU_OK : fail(PALU_EHIP, "%s launch: %s", who, hipGetErrorString(e));
}
