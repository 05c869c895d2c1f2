// Prefill projections: y[m][c] = sum_k x[m][k] w[c][k] for many rows (more than the 64 of a decode step), over the
// weight as the decode step holds it: 16 x 32 tiles of 1 KB, each the A operand of v_mfma_f32_16x16x32_bf16 as it
// stands, row tiles in groups of rtw stored [k tile][row tile in group] (palu_linear.hip). The prefill used to copy
// every weight back to the nn.Linear layout on each call and multiply with the library GEMM: the copy moved the
// weight about six times, more than the product itself up to some thousand rows. No counterpart in the
// reference's op interface (its ttnn.linear calls, palu_tt/attention.py:380-480 and model.py).
//
// A workgroup owns 128 activation rows (MT 16-row tiles) and 64 RPW output columns, its 4 waves RPW row tiles of the
// weight each. A weight tile is used by exactly one wave, so it goes from memory straight to that wave's registers; the
// activations, which all four waves read, are copied straight to LDS (global_load_lds: lane l's 16 bytes land at 16 l of
// the tile's kilobyte, which is the operand order), three 64-deep k stages ahead. An activation tile read from
// LDS feeds RPW MFMAs and a weight tile MT. Two workgroups share a CU.
//
// Bound: MFMA from some 500 rows on, the weight stream below. Measured (MI355X, weights rotated past the caches; the
// library GEMM on an nn.Linear-layout copy, without the time to make the copy and without SwiGLU, in brackets; two boxes
// where they differ): 2048 x 28672 x 4096 with SwiGLU 428 us = 1.13 PFLOP/s (355 to 391), 2048 x 4096 x 14336 220 (208
// to 222), 4096 x 5120 x 4096 182 (145), 1554 x 5376 x 4096 107 (72), 512 x 28672 x 4096 129 (100), 128 x 28672 x 4096
// 56 (56), 300 x 4096 x 14336 62 (74), 100 x 4096 x 14336 34 (51). So the library's product is the faster one at full
// shapes; the copy it needs takes longer than the difference. First forms: activations through registers (one stage
// ahead) 535 us at the first shape; 256-row workgroups with one wave per SIMD 653 to 740 us (the 256 accumulators and
// the stages do not fit without copies); waits left to the compiler 543 us.
//
// Work order: the workgroups that share a weight column block run next to each other on one XCD (ids 8 apart), so the
// weight comes from memory once and from that XCD's L2 for the other row blocks.
//
// Outputs: bf16 rows; fp32 partial sums of ks k slices (summed by palu_rows_reduce_kernel); or, for a gate / up weight
// interleaved eight rows at a time, silu(gate) * up rows: the gate / up product itself is never written.
#include "palu_kernel.h"

#include <algorithm>

namespace {

struct RowsArgs {
  const __bf16* x;
  long long ldx;
  int m;
  const __bf16* wt;
  int rtw, n16, kt_total, ks, ktps;      // k slices of ktps k tiles
  int ncol, mblk;                         // column blocks x k slices, row blocks
  __bf16* y;
  long long ldy;
  float* part;                            // [ks][m][n] when ks > 1
};

typedef __attribute__((address_space(1))) const void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

constexpr int XS = 4;                     // activation stages in LDS
constexpr int ROWS_MT = 8;                // 16-row activation tiles of a workgroup
constexpr int ROWS_PER_CU = 2;            // workgroups that share a CU

template <int MT, int RPW, bool SWIGLU>
__global__ __launch_bounds__(256, 2) void palu_rows_kernel(const RowsArgs a) {
  static_assert(MT % 4 == 0 && RPW >= 1, "whole activation tiles per wave");
  constexpr int XPW = MT / 2;             // activation tiles a wave copies per k stage (2 MT tiles, 4 waves)
  constexpr int WS = RPW >= 4 ? 2 : 4;    // weight stages in registers
  // One array per stage: the compiler then knows that a copy into one stage is no store to the stage being read.
  __shared__ bf16x8 xs0[2 * MT * 64], xs1[2 * MT * 64], xs2[2 * MT * 64], xs3[2 * MT * 64];
  const int tid = threadIdx.x, lane = tid & 63, mm = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xj = blockIdx.x >> 3;
  const int mb = xj % a.mblk, col = (xj / a.mblk) * 8 + (blockIdx.x & 7);
  if (col >= a.ncol) return;              // padding workgroup (uniform)
  const int ks = col % a.ks, rt0 = (col / a.ks) * 4 * RPW + w * RPW;
  const int kt_lo = ks * a.ktps, kt_hi = min(a.kt_total, kt_lo + a.ktps);
  const int nst = (kt_hi - kt_lo) >> 1;                   // stages of two k tiles
  const int row0 = mb * 16 * MT;

  // Weight streams: row tile rt of group gi lies at ((gi rtw) kt_total + kt cnt + r) KB. Row tiles past the matrix read
  // its last one (their outputs are not stored).
  const bf16x8* wp[RPW];
  int ws[RPW];
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    const int rt = min(rt0 + i, a.n16 - 1), gi = rt / a.rtw;
    ws[i] = min(a.rtw, a.n16 - gi * a.rtw) * 64;
    wp[i] = reinterpret_cast<const bf16x8*>(a.wt) + ((long long)gi * a.rtw * a.kt_total + (rt - gi * a.rtw)) * 64 +
            (long long)kt_lo * ws[i];
  }
  // Activation tiles of this wave: t = w XPW + i is (row tile t / 2, k tile t % 2 of the stage), so a wave reads both
  // 64-byte halves of a row's 128-byte line.
  const __bf16* xp[XPW / 2];
#pragma unroll
  for (int i = 0; i < XPW / 2; ++i) {
    const int r = min(row0 + 16 * (w * (XPW / 2) + i) + mm, a.m - 1);
    xp[i] = a.x + (long long)r * a.ldx + 32LL * kt_lo + 8 * g;
  }

  f32x4 acc[RPW][MT];
#pragma unroll
  for (int i = 0; i < RPW; ++i)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 wr[WS][2][RPW];
  const int kt_n = kt_hi - kt_lo;
  auto load_w = [&](int par, int kth, int s) {
    const long long kt = min(2 * s + kth, kt_n - 1);
#pragma unroll
    for (int i = 0; i < RPW; ++i) wr[par][kth][i] = wp[i][kt * ws[i] + lane];
  };
  // Stage s of this wave's activation tiles straight to LDS (lane l's 16 bytes land at 16 l of the tile's kilobyte).
  auto load_x = [&](bf16x8* buf, int s) {
#pragma unroll
    for (int i = 0; i < XPW; ++i) {
      const int kt = min(2 * s + (i & 1), kt_n - 1);
      __builtin_amdgcn_global_load_lds((gvoid*)(xp[i >> 1] + 32LL * kt),
                                       (lvoid*)(buf + ((i & 1) * MT + w * (XPW / 2) + (i >> 1)) * 64), 16, 0, 0);
    }
  };
  // `tail`: one of the last nst % 4 stages (a constant where it is called), whose copies ahead would be past the slice.
  auto stage = [&](const bf16x8* cur, bf16x8* nxt, int j, int s, bool tail) __attribute__((always_inline)) {
    // The stage's activation tiles in pairs, each pair read from LDS while the one before it is multiplied (left to the
    // compiler every read stood right before its use), and the products ahead of the other workgroup's address work: 2048 x
    // 28672 x 4096 434 -> 427 us, 2048 x 4096 x 14336 223 -> 220.
    bf16x8 b[2][2];
    auto read = [&](int q) {
#pragma unroll
      for (int i = 0; i < 2; ++i) b[q & 1][i] = cur[(2 * q + i) * 64 + lane];
    };
    read(0);
    if (!tail) load_x(nxt, s + XS - 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < MT; ++q) {        // k tile q / (MT / 2), row tiles 2 q % MT and the next
      const int kth = q / (MT / 2);
      if (q + 1 < MT) read(q + 1);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < RPW; ++i)
          acc[i][(2 * q + h) % MT] = mfma16(wr[j % WS][kth][i], b[q & 1][h], acc[i][(2 * q + h) % MT]);
      __builtin_amdgcn_s_setprio(0);
      if (q % (MT / 2) == MT / 2 - 1) load_w(j % WS, kth, s + WS);
      __builtin_amdgcn_sched_barrier(0);
    }
    // Loads complete in order. The next stage's activations were asked for XS - 2 stages ago and its weights WS - 1
    // stages ago, so once no more than the loads of that many stages are outstanding, both have arrived, and past the
    // barrier in every wave. (Left to the compiler the weights' wait was for every load.) That count holds where every
    // stage issues all its loads; a tail stage does not (it copies nothing, and the compiler drops weight loads that no
    // stage uses), so it waits for everything.
    __builtin_amdgcn_sched_barrier(0);
    constexpr int V = (WS - 1 < XS - 2 ? WS - 1 : XS - 2) * (XPW + 2 * RPW);
    static_assert(V < 64, "the wait counter");
    if (tail) __builtin_amdgcn_s_waitcnt(0x0F70);
    else __builtin_amdgcn_s_waitcnt(0x0F70 | (V & 15) | ((V >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  if (nst > 0) {
#pragma unroll
    for (int j = 0; j < WS; ++j) {
      load_w(j, 0, j);
      load_w(j, 1, j);
    }
    load_x(xs0, 0);
    load_x(xs1, 1);
    __builtin_amdgcn_sched_barrier(0);                    // stage 2's copies last: the wait below is for all but them
    load_x(xs2, 2);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70 | XPW);             // the loop counts on loads in steady order
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    int s = 0;
    for (; s + 4 <= nst; s += 4) {
      stage(xs0, xs3, 0, s, false);
      stage(xs1, xs0, 1, s + 1, false);
      stage(xs2, xs1, 2, s + 2, false);
      stage(xs3, xs2, 3, s + 3, false);
    }
    if (s < nst) stage(xs0, xs3, 0, s, true);
    if (s + 1 < nst) stage(xs1, xs0, 1, s + 1, true);
    if (s + 2 < nst) stage(xs2, xs1, 2, s + 2, true);
  }
  if (kt_n & 1) {                         // an odd slice's last k tile, straight from memory
    const int kt = kt_n - 1;
    bf16x8 wl[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) wl[i] = wp[i][(long long)kt * ws[i] + lane];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int r = min(row0 + 16 * t + mm, a.m - 1);
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(a.x + (long long)r * a.ldx + 32LL * (kt_lo + kt) + 8 * g);
#pragma unroll
      for (int i = 0; i < RPW; ++i) acc[i][t] = mfma16(wl[i], b, acc[i][t]);
    }
  }

  // Lane (g, mm) of tile (i, t): columns 16 (rt0 + i) + 4 g .. + 3 of row row0 + 16 t + mm.
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int row = row0 + 16 * t + mm;
    if constexpr (SWIGLU) {
      static_assert(MT % 2 == 0, "row tiles are paired");
      if (t & 1) continue;
      // Lanes g < 2 hold gate columns, lanes g + 2 the up columns of the same outputs; one v_permlane32_swap of row
      // tiles t and t + 1 leaves every lane a gate and its up: lanes g < 2 of row tile t, g >= 2 of t + 1.
#pragma unroll
      for (int i = 0; i < RPW; ++i) {
        bf16x4 o;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i][t][k]), __float_as_uint(acc[i][t + 1][k]),
                                                           false, false);
          const float gv = __uint_as_float(sw[0]), uv = __uint_as_float(sw[1]);
          o[k] = (__bf16)((gv / (1.f + __expf(-gv))) * uv);
        }
        const int r = row + (g < 2 ? 0 : 16);
        if (r < a.m && rt0 + i < a.n16) *reinterpret_cast<bf16x4*>(a.y + r * a.ldy + 8 * (rt0 + i) + 4 * (g & 1)) = o;
      }
    } else {
#pragma unroll
      for (int i = 0; i < RPW; ++i) {
        if (row < a.m && rt0 + i < a.n16) {
          const int c = 16 * (rt0 + i) + 4 * g;
          if (a.part) {
            *reinterpret_cast<f32x4*>(a.part + ((long long)ks * a.m + row) * (16LL * a.n16) + c) = acc[i][t];
          } else {
            bf16x4 o;
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = (__bf16)acc[i][t][k];
            *reinterpret_cast<bf16x4*>(a.y + row * a.ldy + c) = o;
          }
        }
      }
    }
  }
}

// y[r][c] = bf16(sum over the k slices, in order); 4 columns per thread.
__global__ __launch_bounds__(256) void palu_rows_reduce_kernel(const float* __restrict__ part, int ks, int m, int n,
                                                               __bf16* __restrict__ y, long long ldy) {
  const long long quads = (long long)m * (n / 4);
  for (long long e = blockIdx.x * 256LL + threadIdx.x; e < quads; e += (long long)gridDim.x * 256) {
    const int r = (int)(e / (n / 4)), c = (int)(e % (n / 4)) * 4;
    f32x4 s = *reinterpret_cast<const f32x4*>(part + (long long)r * n + c);
    for (int k = 1; k < ks; ++k) s += *reinterpret_cast<const f32x4*>(part + ((long long)k * m + r) * n + c);
    bf16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (__bf16)s[i];
    *reinterpret_cast<bf16x4*>(y + r * ldy + c) = o;
  }
}

template <int MT, int RPW, bool SWIGLU>
int launch_rows(const RowsArgs& a0, hipStream_t s) {
  RowsArgs a = a0;
  a.mblk = (a.m + 16 * MT - 1) / (16 * MT);
  a.ncol = (a.n16 + 4 * RPW - 1) / (4 * RPW) * a.ks;
  auto kern = palu_rows_kernel<MT, RPW, SWIGLU>;
  hipLaunchKernelGGL(kern, dim3((unsigned)((a.ncol + 7) / 8 * 8 * a.mblk)), dim3(256), 0, s, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? PALU_OK : fail(PALU_EHIP, "palu_linear_rows launch: %s", hipGetErrorString(e));
}

struct RowsPlan {
  int rpw, ks;
};

// Columns per workgroup (64 RPW) and k slices: the pair whose busiest CU finishes first, from a model in clocks. Per k
// tile a workgroup's MFMAs take 16 MT RPW clocks and its loads about 40 bytes a clock; RPW 4 moves fewer bytes per product
// (2048 x 28672 x 4096: 437 against 581 us), RPW 2 makes twice the workgroups and keeps twice as many stages in flight,
// which wins where there is one row block (128 rows: 59.5 against 79.3 us). A k split costs its partial sums' round
// trip and a launch: 100 x 4096 x 14336 takes 139 us whole, 33.7 in 8 slices, 41.8 in 16; 2048 rows 226 whole, 234 in 2.
// The model's pick was the fastest or within 4 % of it at 15 of 17 measured shapes (12 % off at the worst).
RowsPlan rows_plan(int m, int n16, int kt_total, bool swiglu) {
  RowsPlan best{4, 1};
  double cost = 1e300;
  for (const int rpw : {4, 2}) {
    const long long mblk = (m + 16 * ROWS_MT - 1) / (16 * ROWS_MT), ncol = (n16 + 4 * rpw - 1) / (4 * rpw);
    for (int ks = 1; ks <= (swiglu ? 1 : 16); ks *= 2) {
      const int ktps = (kt_total + ks - 1) / ks;
      if (ks > 1 && ktps < 16) break;
      const long long units = mblk * ncol * ks, slots = 256LL * ROWS_PER_CU;
      const double mfma = 16.0 * ROWS_MT * rpw, mem = (4.0 * rpw + ROWS_MT) * 1024.0 / 40.0;
      const double rounds = units <= 256 ? 1.0 : (double)((units + slots - 1) / slots) * ROWS_PER_CU;
      const double t = rounds * (ktps * (mfma > mem ? mfma : mem) + 3000.0) + (ks > 1 ? 6000.0 + 2.0 * ks * m * n16 * 64 / 2000.0 : 0.0);
      if (t < cost * 0.999) {
        cost = t;
        best = RowsPlan{rpw, ks};
      }
    }
  }
  return best;
}

template <bool SWIGLU>
int dispatch_rows(const RowsPlan& p, const RowsArgs& a, hipStream_t s) {
  return p.rpw == 4 ? launch_rows<ROWS_MT, 4, SWIGLU>(a, s) : launch_rows<ROWS_MT, 2, SWIGLU>(a, s);
}

bool rows_shape_ok(int m, int n, int k) { return m > 0 && n > 0 && n % 16 == 0 && k > 0 && k % 32 == 0; }

}  // namespace

extern "C" size_t palu_linear_rows_workspace_bytes(int m, int n, int k, int y_mode) {
  if (!rows_shape_ok(m, n, k) || y_mode != PALU_LINEAR_BF16) return 0;
  const RowsPlan p = rows_plan(m, n / 16, k / 32, false);
  return p.ks > 1 ? (size_t)p.ks * m * n * sizeof(float) : 0;
}

extern "C" int palu_linear_rows(const void* x, long long ldx, int m, const void* w_tiled, int n, int k, int rtw, void* y,
                                long long ldy, int y_mode, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  palu::g_err[0] = 0;
  const char* who = "palu_linear_rows";
  if (!x || !w_tiled || !y) return fail(PALU_EINVAL, "%s: a required pointer is null", who);
  if (!rows_shape_ok(m, n, k)) return fail(PALU_EINVAL, "%s: m = %d, n = %d (multiple of 16), k = %d (multiple of 32)", who, m, n, k);
  if (y_mode != PALU_LINEAR_BF16 && y_mode != PALU_LINEAR_SWIGLU_ROWS)
    return fail(PALU_EINVAL, "%s: y_mode = %d is not PALU_LINEAR_BF16 or PALU_LINEAR_SWIGLU_ROWS", who, y_mode);
  const bool swiglu = y_mode == PALU_LINEAR_SWIGLU_ROWS;
  if (ldx < k || ldx % 8 || ldy < (swiglu ? n / 2 : n) || ldy % 4)
    return fail(PALU_EINVAL, "%s: row strides ldx = %lld (multiple of 8), ldy = %lld (of 4)", who, ldx, ldy);
  if (rtw < 1 || rtw > 8) return fail(PALU_EINVAL, "%s: rtw = %d (1..8, as the weight was tiled)", who, rtw);
  if (((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w_tiled)) & 15) || (reinterpret_cast<uintptr_t>(y) & 7))
    return fail(PALU_EINVAL, "%s: x and w_tiled must be 16-byte, y 8-byte aligned", who);
  const RowsPlan p = rows_plan(m, n / 16, k / 32, swiglu);
  const size_t need = palu_linear_rows_workspace_bytes(m, n, k, y_mode);
  if (need && (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15)))
    return fail(PALU_EINVAL, "%s: workspace of %zu bytes (16-byte aligned) needed, got %zu", who, need, workspace_bytes);
  if (((long long)m + 127) / 128 * ((n / 16 + 7) / 8 * 16LL + 8) > 0x7fffffffLL) return fail(PALU_EUNSUPPORTED, "%s: grid too large", who);
  RowsArgs a{static_cast<const __bf16*>(x), ldx, m, static_cast<const __bf16*>(w_tiled), rtw, n / 16, k / 32, p.ks,
             (k / 32 + p.ks - 1) / p.ks, 0, 0, static_cast<__bf16*>(y), ldy, p.ks > 1 ? static_cast<float*>(workspace) : nullptr};
  a.ks = (a.kt_total + a.ktps - 1) / a.ktps;              // no empty slice
  if (int rc = swiglu ? dispatch_rows<true>(p, a, stream) : dispatch_rows<false>(p, a, stream)) return rc;
  if (a.part) {
    const long long quads = (long long)m * (n / 4);
    hipLaunchKernelGGL(palu_rows_reduce_kernel, dim3((unsigned)std::min<long long>((quads + 255) / 256, 4096)), dim3(256), 0,
                       stream, a.part, a.ks, m, n, a.y, ldy);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(PALU_EHIP, "%s reduce launch: %s", who, hipGetErrorString(e));
  }
  return PALU_OK;
}
