// Decode-step projections: y[m][c] = sum_k x[m][k] w[c][k] for the rows of one decode step (m <= 64),
// bf16 in, fp32 accumulate. Every weight byte is used once per step by all m rows, so each call is one
// stream of the weight matrix from HBM; the activations (at most 64 x k bf16, L2-resident) are re-read
// from L2 by every workgroup. No counterpart in the reference's op interface: these are the
// ttnn.linear calls of the reference model's decode step (palu_tt/attention.py:585-733, model.py),
// which the decoder issues for its QKV, output, gate/up, down and LM-head projections.
//
// Weights are stored tiled (palu_tt.decoder_ops.tile_weight): row tile rt (16 output columns) and k
// tile kt (32 inputs) form one 1 KB tile, the A operand of v_mfma_f32_16x16x32_bf16 for one wave, lane
// l = 16 g + n holding w[16 rt + n][32 kt + 8 g .. +7]. Row tiles form groups of RTW (the last group may
// be shorter) and a group's tiles are stored k tile by k tile ([kt][rt in group]), so the workgroup that
// owns a group (or one k slice of it) reads one sequential stream; every weight load of a wave is one
// aligned kilobyte. The activations come row-major (lane (g, n) of tile (kt, mt) reads 16 bytes of row
// 16 mt + n: sixteen half cache lines per tile) or tiled the same way as the weights with the 64 rows as
// four row tiles ([kt][mt], palu_tt.decoder_ops.tile_rows; one contiguous kilobyte per tile), which
// the decoder's RMSNorm and SwiGLU kernels write directly.
//
// Outputs (the epilogue, EPI): bf16 y [m][n] (split partials summed by a second launch); the fp32 split
// partials [KS][m][n] themselves, for a consumer that sums them (palu_rmsnorm's residual input,
// palu_qkv_post); for a gate / up weight interleaved eight rows at a time (tile_weight of
// palu_tt.decoder_ops.interleave_gate_up), silu(gate) * up in the tiled activation layout, optionally
// of the RMS-normalised x (the row scale rsqrt(mean(x^2) + eps) applied to the products, the norm's
// weight folded into the gate / up weight; the loop sums x^2 from the activation tiles it already
// loads); the residual update h += y, also written tiled for the next projection; or the decode step's
// QKV epilogue (q RoPE, K / V latent appends), in place of palu_qkv_post's second launch. The last three
// need KS = 1: the epilogue sees whole dot products.
//
// A workgroup owns one group and one of KS slices of the k tiles. Its 4 waves (one per SIMD, so each may
// use the whole 512-entry register file) take the slice's k tiles in turn (wave w: kt0 + w, kt0 + w + 4,
// ...). Per k tile a wave loads RTW weight tiles (nontemporal: read once per step) and the MT 16-row
// activation tiles there are rows for (1, 2 or 4; cached), and issues RTW x MT MFMAs into RTW x MT
// accumulators; the loads of the next NB - 1 k tiles are in flight meanwhile. The waves' partial sums meet
// in LDS, and each wave adds up and stores a quarter of the output tiles (bf16 y, fp32 split partials, or the
// SwiGLU activations). Up to 16 rows load a quarter of the 64-row call's activation tiles: an FFN of 12 rows takes
// 61.2 us against 65.1 with all four, of 32 rows (two tiles) 64.3 against 66.7, a two-layer model's step for one row 356
// against 393.
//
// Measured on MI355X (64 rows, weights rotated past the MALL, HIP-graph launches): the tiled activations
// take the gate/up projection (28672 x 4096) from 51.9 to 43.4 us, against 52.5 us for hipBLASLt; a
// copy of this loop with the MFMAs and activation loads removed streams the weights at 5.6-5.9 TB/s,
// and deeper buffering (6 or 8 steps) or 8 waves per workgroup did not raise it.
#pragma once

#include "palu_kernel.h"

namespace palu {

struct LinEpi {
  float eps, inv_k;                  // EPI_SWIGLU_NORM
  __bf16* h;                         // EPI_RESID: [m][n] bf16, rows ldh apart
  long long ldh;
  __bf16* h_tiled;                   //   and the 64-row tiled copy (or null)
  QkvEpi q;                          // EPI_QKV
};

// palu_linear_kernel for at most 16 / 32 rows (defined in palu_linear_m16.hip, palu_linear_m32.hip).
hipError_t linear_m16(int epi, int x_tiled, int rtw, const __bf16* x, long long ldx, int m, const __bf16* wt, int n16,
                      int kt_total, int ks, int ktps, __bf16* y, long long ldy, float* part, const LinEpi& ep,
                      hipStream_t s);
hipError_t linear_m32(int epi, int x_tiled, int rtw, const __bf16* x, long long ldx, int m, const __bf16* wt, int n16,
                      int kt_total, int ks, int ktps, __bf16* y, long long ldy, float* part, const LinEpi& ep,
                      hipStream_t s);

}  // namespace palu

namespace {

constexpr int LIN_MT = 4;                       // 16-row activation tiles of the tiled layout: m <= 64
constexpr int LIN_MAX_RTW = 8;

// Epilogues.
constexpr int EPI_OUT = 0;           // bf16 y, or the fp32 split partials
constexpr int EPI_SWIGLU = 1;        // silu(gate) * up, tiled
constexpr int EPI_SWIGLU_NORM = 2;   // the same over RMS-normalised x
constexpr int EPI_RESID = 3;         // h += y (row-major), and h tiled
constexpr int EPI_QKV = 4;           // q RoPE and latent appends (QkvEpi)

template <int RTW, int NW, int EPI, int MT>
struct LinSmem {
  static constexpr int SLOT = RTW * MT * 64;              // f32x4 per wave partial
  static constexpr int RED = NW * SLOT * 16;              // every wave's partial
  static constexpr int BYTES = RED + (EPI == EPI_SWIGLU_NORM ? NW * 64 * 4 : 0);   // + per-wave row sums of x^2
};

// Where the QKV epilogue sends columns col .. col + 3: kind 0 (q head gi), 1 / 2 (group gi's K / V
// slice) at column c of the head or slice, or -1 (a column no part reads).
__device__ __forceinline__ int qkv_part_of(const QkvEpi& e, int col, int& gi, int& c) {
  gi = 0;
  c = 0;
  if (col < e.nh * HD) {
    gi = col / HD;
    c = col - gi * HD;
    return 0;
  }
  if (col >= e.k_off && col < e.k_off + (e.G - 1) * e.k_gs + e.k_w) {
    const int d = col - e.k_off;
    gi = e.G > 1 ? d / e.k_gs : 0;
    c = d - gi * e.k_gs;
    return c < e.k_w ? 1 : -1;
  }
  if (col >= e.v_off && col < e.v_off + (e.G - 1) * e.v_gs + e.v_w) {
    const int d = col - e.v_off;
    gi = e.G > 1 ? d / e.v_gs : 0;
    c = d - gi * e.v_gs;
    return c < e.v_w ? 2 : -1;
  }
  return -1;
}

// NB register buffers per wave, so each step's loads are issued NB - 1 steps before its MFMAs. Weight
// and activation tiles of one step share a buffer: loads return in issue order, so an activation tile
// loaded later than the weights would make every wait a wait for those weights too. NW waves per
// workgroup (the launches use 4: one per SIMD, the whole register file each; 8, two per SIMD, was slower
// end to end for the one- and two-tile projections).
template <int RTW, int NB, int NW, bool XT, int EPI, int MT>
__global__ __launch_bounds__(NW * 64) void palu_linear_kernel(const __bf16* __restrict__ x, long long ldx, int m,
                                                              const __bf16* __restrict__ wt, int n16, int kt_total,
                                                              int ks_count, int kt_per_split,
                                                              __bf16* __restrict__ y, long long ldy,
                                                              float* __restrict__ part, const LinEpi ep) {
  using SM = LinSmem<RTW, NW, EPI, MT>;
  constexpr bool SWIGLU = EPI == EPI_SWIGLU || EPI == EPI_SWIGLU_NORM;
  constexpr int NT = (RTW * MT + NW - 1) / NW;       // output tiles each wave stores (at most)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  f32x4* red = reinterpret_cast<f32x4*>(smem);

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int mm = lane & 15, g = lane >> 4;
  const int ks = blockIdx.x % ks_count;
  const int rt0 = (blockIdx.x / ks_count) * RTW;
  const int rt_cnt = min(RTW, n16 - rt0);                 // uniform: the last group may be short
  const int kt_lo = ks * kt_per_split;
  const int kt_hi = min(kt_total, kt_lo + kt_per_split);

  // The epilogue's own global reads (the residual h, the rows' positions) are issued here, ahead of the
  // weight stream, so the epilogue does not start with a round trip to memory. Wave w stores output
  // tiles t = w, w + NW, ... (row tile t / 4, activation tile t % 4); lane (g, mm) of tile t holds
  // columns 16 (rt0 + t / 4) + 4 g .. + 3 of row 16 (t % 4) + mm.
  bf16x4 hpre[NT];
  int ppre[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int t = w + i * NW;
    const int r = t / MT, row = 16 * (t % MT) + mm;
    const bool ok = t < RTW * MT && r < rt_cnt && row < m;
    if constexpr (EPI == EPI_RESID) {
      const int col = 16 * (rt0 + (ok ? r : 0)) + 4 * g;
      hpre[i] = *reinterpret_cast<const bf16x4*>(ep.h + (ok ? row : 0) * ep.ldh + col);
    }
    if constexpr (EPI == EPI_QKV) ppre[i] = ep.q.pos[ok ? row : 0];
  }

  // Activation rows past m are replaced by zeros (row-major: they read row 0); their outputs are not
  // stored.
  const __bf16* xp[MT];
  bool xv[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = 16 * mt + mm;
    xv[mt] = r < m;
    xp[mt] = XT ? x + ((long long)mt * 64 + lane) * 8 : x + (long long)(xv[mt] ? r : 0) * ldx + 8 * g;
  }
  const bf16x8* wp = reinterpret_cast<const bf16x8*>(wt) + (long long)rt0 * kt_total * 64 + lane;

  f32x4 acc[RTW][MT];
#pragma unroll
  for (int r = 0; r < RTW; ++r)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[r][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss[MT] = {};              // EPI_SWIGLU_NORM: this lane's share of sum x^2 per row

  // Every load is issued on every path (row tiles past rt_cnt read the last row tile, k tiles past the
  // slice read the matrix's last k tile; their products are never stored), so each wait in the loop is
  // for exactly the loads of the buffer about to be used.
  bf16x8 wa[NB][RTW], xb[NB][MT];
  // Every workgroup reads the same activation tiles. Walked in the same order, all workgroups would
  // request the same few kilobytes at once; instead each group starts its slice at its own offset and
  // wraps around (32-layer decode step 5.21 -> 5.16 ms in a same-box A/B). i -> (i + krot) mod klen is
  // a permutation of the slice, so the waves together still cover each k tile once; the sums are the
  // same up to the order of the fp32 additions.
  const int klen = kt_hi - kt_lo;
  const int kper = klen / NW > 0 ? klen / NW : 1;
  const int krot = ((blockIdx.x / ks_count) * 37 % kper) * NW % (klen > 0 ? klen : 1);
  auto load = [&](int buf, int kt) {
    int i = kt - kt_lo;                                   // steps past the slice read its last tile
    i = i < klen ? (i + krot >= klen ? i + krot - klen : i + krot) : klen - 1;
    kt = klen > 0 ? min(kt_lo + i, kt_total - 1) : kt_total - 1;   // an empty slice reads the last tile
#pragma unroll
    for (int r = 0; r < RTW; ++r)
      wa[buf][r] = __builtin_nontemporal_load(wp + ((long long)kt * rt_cnt + min(r, rt_cnt - 1)) * 64);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      xb[buf][mt] = *reinterpret_cast<const bf16x8*>(xp[mt] + (XT ? (long long)kt * (LIN_MT * 512) : 32LL * kt));
  };
  auto compute = [&](int buf, bool live) {
    bf16x8 bz[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) bz[mt] = (xv[mt] && live) ? xb[buf][mt] : bf16x8{};
#pragma unroll
    for (int r = 0; r < RTW; ++r)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[r][mt] = mfma16(wa[buf][r], bz[mt], acc[r][mt]);
    if constexpr (EPI == EPI_SWIGLU_NORM) {
      // x^2 summed in pairs (v_dot2: the bf16 products are exact in fp32)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bf16x2 p2{bz[mt][2 * j], bz[mt][2 * j + 1]};
          ss[mt] = __builtin_amdgcn_fdot2_f32_bf16(p2, p2, ss[mt], false);
        }
    }
  };

  // The loop is unrolled by NB so that buffer indices are compile-time, and has no branch: steps past the
  // wave's count (the rest of the last round) load clamped tiles and multiply them by zero activations.
  // The scheduling barriers keep each step's loads ahead of the earlier step's MFMAs (left alone, the
  // compiler sinks every load to its first use and the wave has one tile in flight).
  // The prologue's loads keep their order (a scheduling barrier after each buffer): the loop-top wait
  // is computed from the load order on both paths into the loop, and a prologue reordered by the
  // scheduler made the compiler wait there for all but the newest loads, a drain every NB steps
  // (32-layer decode step 5.27 -> 5.23 ms in a same-box A/B).
  const int kt0 = kt_lo + w;
  const int nsteps = kt0 < kt_hi ? (kt_hi - kt0 + NW - 1) / NW : 0;   // uniform per wave
#pragma unroll
  for (int j = 0; j < NB - 1; ++j) {
    load(j, kt0 + j * NW);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int s = 0; s < nsteps; s += NB) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      load((j + NB - 1) % NB, kt0 + (s + j + NB - 1) * NW);
      __builtin_amdgcn_sched_barrier(0);
      compute(j, s + j < nsteps);
    }
  }

  // The waves' partials meet in LDS (slot layout [wave][r][mt][lane] of f32x4); each wave then sums
  // the NW slots of every NW-th (r, mt) tile and stores that tile, so the epilogue's arithmetic and
  // stores are spread over the SIMDs. Every LDS read of the sums is issued before the first is used and
  // the tiles are stored under a predicate rather than a branch per tile: the epilogue sits between the
  // last weight load and the end of the launch, and one round trip to LDS per tile (its reads, then the
  // next tile's) made it 1.2 us longer for the gate / up shape.
#pragma unroll
  for (int r = 0; r < RTW; ++r)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[w * SM::SLOT + (r * MT + mt) * 64 + lane] = acc[r][mt];
  float* rss = reinterpret_cast<float*>(smem + SM::RED);   // [wave][row] sums of x^2
  if constexpr (EPI == EPI_SWIGLU_NORM) {
    // lanes (g, mm), g = 0..3, hold columns 8 g .. 8 g + 7 of every k tile of row 16 mt + mm
    float s16[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) s16[mt] = ss[mt] + __shfl_xor(ss[mt], 16, 64);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) ss[mt] = s16[mt] + __shfl_xor(s16[mt], 32, 64);
    if (g == 0) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) rss[w * 64 + 16 * mt + mm] = ss[mt];
    }
  }
  __syncthreads();

  // Wave w's tiles t = w + i NW, i < NT (clamped to the last tile for the loads; tiles past it are not
  // stored). Lane (g, mm) of tile (r, mt) holds y^T[16 (rt0 + r) + 4 g + i][16 mt + mm], i < 4: four
  // consecutive output columns of activation row 16 mt + mm.
  f32x4 v[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int t = min(w + i * NW, RTW * MT - 1);
    v[i] = red[t * 64 + lane];
#pragma unroll
    for (int q = 1; q < NW; ++q) v[i] += red[q * SM::SLOT + t * 64 + lane];
  }
  if constexpr (EPI == EPI_SWIGLU_NORM) {
    // the row scale rsqrt(mean x^2 + eps): with NW a multiple of MT (asserted below) every tile of
    // wave w lies in activation tile w % MT, one row per lane
    const int row = 16 * (w % MT) + mm;
    float tot = 0.f;
#pragma unroll
    for (int q = 0; q < NW; ++q) tot += rss[q * 64 + row];
    const float sc = rsqrtf(tot * ep.inv_k + ep.eps);
#pragma unroll
    for (int i = 0; i < NT; ++i) v[i] *= sc;
  }
  if constexpr (SWIGLU) {
    static_assert(NW % MT == 0, "the SwiGLU epilogue pairs tiles of one activation tile");
    // Gate / up pairs: rows 0-7 of row tile rt are gate columns 8 rt .. 8 rt + 7 and rows 8-15 the up
    // columns of the same outputs (tile_weight of the interleaved weight), so lanes g < 2 of a tile hold
    // gate values and lanes g + 2, 32 lanes on, the matching up values. Tiles i and i + 1 of a wave
    // share their activation rows; one v_permlane32_swap of the upper half of tile i with the lower half
    // of tile i + 1 puts the gates of both in one register and the ups in the other, so that every lane
    // computes and stores one output of one of the two tiles (lanes 32-63: tile i + 1, output columns
    // 8 rt + 4 (g - 2) .. + 3). out = silu(gate) * up, stored in the tiled activation layout (64 rows x
    // n / 2) the next projection reads.
    const int row = 16 * (w % MT) + mm;
#pragma unroll
    for (int i = 0; i < NT; i += 2) {
      const int j = i + 1 < NT ? i + 1 : i;
      f32x4 gv, uv;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i][k]), __float_as_uint(v[j][k]), false, false);
        gv[k] = __uint_as_float(sw[0]);
        uv[k] = __uint_as_float(sw[1]);
      }
      bf16x4 o;
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] = (__bf16)((gv[k] / (1.f + __expf(-gv[k]))) * uv[k]);
      const int t = w + (g < 2 ? i : j) * NW, r = t / MT;
      if (t < RTW * MT && r < rt_cnt && row < m && (g < 2 || j != i))
        *reinterpret_cast<bf16x4*>(y + tiled_row_offset(row, 8 * (rt0 + r) + 4 * (g & 1))) = o;
    }
  } else {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int t = w + i * NW;
      const int r = t / MT, row = 16 * (t % MT) + mm;
      const bool ok = t < RTW * MT && r < rt_cnt && row < m;
      if constexpr (EPI == EPI_RESID) {
        // h + y rounded to bf16 once (the residual stream), in place and in the tiled layout
        if (ok) {
          const int col = 16 * (rt0 + r) + 4 * g;
          bf16x4 o;
#pragma unroll
          for (int k = 0; k < 4; ++k) o[k] = (__bf16)((float)hpre[i][k] + v[i][k]);
          *reinterpret_cast<bf16x4*>(ep.h + row * ep.ldh + col) = o;
          if (ep.h_tiled) *reinterpret_cast<bf16x4*>(ep.h_tiled + tiled_row_offset(row, col)) = o;
        }
      } else if constexpr (EPI == EPI_QKV) {
        // Columns col .. col + 3 of QKV row `row` lie in one q head or one group's K or V slice (the
        // entry point checks that the three ranges do not overlap and start on multiples of 8).
        int gi, c;
        const int kind = ok ? qkv_part_of(ep.q, 16 * (rt0 + r) + 4 * g, gi, c) : -1;
        if (kind >= 0) {
          float vv[4] = {v[i][0], v[i][1], v[i][2], v[i][3]};
          qkv_store<4>(ep.q, row, ppre[i], kind, gi, c, vv);
        }
      } else {
        if (ok) {
          const long long col = 16LL * (rt0 + r) + 4 * g;
          if (part) {
            *reinterpret_cast<f32x4*>(part + ((long long)ks * m + row) * (16LL * n16) + col) = v[i];
          } else {
            bf16x4 o;
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = (__bf16)v[i][k];
            *reinterpret_cast<bf16x4*>(y + row * ldy + col) = o;
          }
        }
      }
    }
  }
}

// Register buffers per wave: NB = 4 for every width. Workgroups of one or two row tiles load more
// activation than weight bytes per k tile (4 KB against 1-2 KB), and deeper rings only queue more of
// those L2 reads ahead of the weights: in graph-captured probes the QKV shape (two row tiles) took 16.4 us
// at NB 4 against 17.0 at 8 and 18.2 at 12, the output projection's (one row tile) 7.9 against 8.2 us at 8,
// and the 32-layer decode step 5.02 against 5.06 ms (same-box A/B, three runs each). With the fewer activation tiles of
// up to 32 rows the same holds: a two-layer model's step for one row 355 us at NB 4, 355 with 8 for one and two row
// tiles, 363 with 8 for all; an FFN of 12 rows 61.1 at NB 4, 63.1 at 8.

template <int RTW, bool XT, int EPI, int MT>
hipError_t launch_cfg(const __bf16* x, long long ldx, int m, const __bf16* wt, int n16, int kt_total, int ks,
                      int ktps, __bf16* y, long long ldy, float* part, const LinEpi& ep, hipStream_t s) {
  constexpr int NB = 4;
  constexpr int NW = 4;                                   // one wave per SIMD (8 measured slower end to end)
  auto kern = palu_linear_kernel<RTW, NB, NW, XT, EPI, MT>;
  constexpr int lds = LinSmem<RTW, NW, EPI, MT>::BYTES;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  const int groups = (n16 + RTW - 1) / RTW;
  hipLaunchKernelGGL(kern, dim3(groups * ks), dim3(NW * 64), lds, s, x, ldx, m, wt, n16, kt_total, ks, ktps, y,
                     ldy, part, ep);
  return hipGetLastError();
}

template <bool XT, int EPI, int MT>
hipError_t launch_rtw(int rtw, const __bf16* x, long long ldx, int m, const __bf16* wt, int n16, int kt_total, int ks,
                      int ktps, __bf16* y, long long ldy, float* part, const LinEpi& ep, hipStream_t s) {
  switch (rtw) {
    case 1: return launch_cfg<1, XT, EPI, MT>(x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    case 2: return launch_cfg<2, XT, EPI, MT>(x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    case 3: return launch_cfg<3, XT, EPI, MT>(x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    case 4: return launch_cfg<4, XT, EPI, MT>(x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    case 5: return launch_cfg<5, XT, EPI, MT>(x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    case 6: return launch_cfg<6, XT, EPI, MT>(x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    case 7: return launch_cfg<7, XT, EPI, MT>(x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    default: return launch_cfg<8, XT, EPI, MT>(x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
  }
}

template <int EPI, int MT>
hipError_t launch_epi(int x_tiled, int rtw, const __bf16* x, long long ldx, int m, const __bf16* wt, int n16,
                      int kt_total, int ks, int ktps, __bf16* y, long long ldy, float* part, const LinEpi& ep,
                      hipStream_t s) {
  return x_tiled ? launch_rtw<true, EPI, MT>(rtw, x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s)
                 : launch_rtw<false, EPI, MT>(rtw, x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
}

template <int MT>
hipError_t launch_mt(int epi, int x_tiled, int rtw, const __bf16* x, long long ldx, int m, const __bf16* wt, int n16,
                     int kt_total, int ks, int ktps, __bf16* y, long long ldy, float* part, const LinEpi& ep,
                     hipStream_t s) {
  switch (epi) {
    case EPI_SWIGLU: return launch_epi<EPI_SWIGLU, MT>(x_tiled, rtw, x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    case EPI_SWIGLU_NORM:
      return launch_epi<EPI_SWIGLU_NORM, MT>(x_tiled, rtw, x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    case EPI_RESID: return launch_epi<EPI_RESID, MT>(x_tiled, rtw, x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    case EPI_QKV: return launch_epi<EPI_QKV, MT>(x_tiled, rtw, x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
    default: return launch_epi<EPI_OUT, MT>(x_tiled, rtw, x, ldx, m, wt, n16, kt_total, ks, ktps, y, ldy, part, ep, s);
  }
}

}  // namespace
