// The naive decode of per-head latents (PaluRuntime.use_fused_k off, the reference's default; palu_tt/attention.py:
// 657-710): every attended key is rebuilt and written out, K[p] = RoPE_p(lat[p] u_k), and the stock flash-decode runs
// over those keys and the V latent. The rebuild kernel reads the latent cache in the layout it has and writes
// the keys in the same layout, ready for the flash-decode; V is read where it lies.
#include "palu_kernel.h"

#include <algorithm>

namespace {

struct RebuildArgs {
  const __bf16* lat;                      // [B][n_kv][cache_len][r], row-major or K tiles
  const __bf16* u_k;                      // [n_kv][r][128]
  const float* cos_t;                     // [table_rows][128], Meta-interleaved
  const float* sin_t;
  const int32_t* cur_pos;
  __bf16* k;                              // [B][n_kv][S][128], the layout of lat
  int n_kv, cache_len, S, table_rows, chunks, per_wave;
};

// A workgroup takes `per_wave` 32-position blocks per wave of one (row, KV head); blocks past the row's position are
// skipped. u_k^T sits in LDS ([dim][rank], rows padded by 16 bytes), a latent block in registers as the MFMA's B
// operand (the K-tile order; row-major caches are read in it), and the accumulators leave lane (n, g) with dims
// 16 t + 4 g .. + 3 of one position: the RoPE pairs are in the lane, and the rotated key, rounded to bf16 once, is four
// consecutive width-indices of the K tile (eight-byte stores, 512 contiguous bytes per instruction).
// Bound by memory and latency: the latents in, 256 bytes per key and head out (from L2 again for the flash-decode), and
// the fp32 table rows, once per head (from L2). Four rows of 2000 positions at r 64 / 64: rebuild 16 us, flash-decode
// 13.5, a layer's step 43 us against 120 with the chain of torch launches before (tiles to rows, copies, GEMM, rotation).
// Loading a block's table rows ahead of its products took 22 us (the last block's loads of a next one are lost).
template <bool TILED, int R>
__global__ __launch_bounds__(256) void palu_rebuild_kernel(const RebuildArgs a) {
  static_assert(R % 16 == 0 && R <= HD && (TILED || R % 32 == 0), "half K tiles exist in the tiled layout only");
  constexpr int KBF = R / 32, KB = (R + 31) / 32, US = R + 8;
  __shared__ __attribute__((aligned(16))) __bf16 ut[HD * US];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int item = blockIdx.x / a.chunks, b = item / a.n_kv, h = item - b * a.n_kv;
  const int blk0 = (blockIdx.x - item * a.chunks) * 4 * a.per_wave;
  const int len = max(0, min(a.S, load_uniform(a.cur_pos, b) + 1));
  const int nblk = (len + BLK - 1) / BLK;
  if (blk0 >= nblk) return;               // uniform, before the barrier

  const __bf16* lat = a.lat + (long long)item * a.cache_len * R;
  __bf16* k = a.k + (long long)item * a.S * HD;
  const int t0 = 8 * (n >> 2) + (n & 3);  // this lane's position in half-block 0
  // Block j's latents (past the row's last block: that one again, unused). No load sits under a branch: the wait at its
  // end would be for every load before it.
  bf16x8 x[2][KB];
  auto load = [&](int j) {
    j = min(j, nblk - 1);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if constexpr (TILED) {
        const __bf16* t = lat + (long long)j * 32 * R + c * 16 * R;
#pragma unroll
        for (int kb = 0; kb < KBF; ++kb) x[c][kb] = *reinterpret_cast<const bf16x8*>(t + kb * 512 + lane * 8);
        if constexpr (KB > KBF) x[c][KBF] = low4(*reinterpret_cast<const bf16x4*>(t + KBF * 512 + lane * 4));
      } else {
        const __bf16* t = lat + (long long)min(32 * j + t0 + 4 * c, a.cache_len - 1) * R + 8 * g;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) x[c][kb] = *reinterpret_cast<const bf16x8*>(t + 32 * kb);
      }
    }
  };
  load(blk0 + w);
  constexpr int UPT = (R * (HD / 8) + 255) / 256;
  bf16x8 uv[UPT];
#pragma unroll
  for (int i = 0; i < UPT; ++i) {
    const int e = min(tid + i * 256, R * (HD / 8) - 1);
    uv[i] = *reinterpret_cast<const bf16x8*>(a.u_k + ((long long)h * R + e % R) * HD + (e / R) * 8);
  }
#pragma unroll
  for (int i = 0; i < UPT; ++i) {
    const int e = min(tid + i * 256, R * (HD / 8) - 1);    // threads past the end store the last piece again
#pragma unroll
    for (int q = 0; q < 8; ++q) ut[((e / R) * 8 + q) * US + e % R] = uv[i][q];
  }
  __syncthreads();

  for (int i = 0; i < a.per_wave; ++i) {
    const int j = blk0 + i * 4 + w;
    if (j >= nblk) return;                // uniform per wave; no barrier follows
    f32x4 acc[2][8];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int t = 0; t < 8; ++t) acc[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        bf16x8 u;
        if (kb < KBF) u = *reinterpret_cast<const bf16x8*>(ut + (16 * t + n) * US + 32 * kb + 8 * g);
        else u = low4(*reinterpret_cast<const bf16x4*>(ut + (16 * t + n) * US + 32 * kb + 4 * g));
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[c][t] = mfma16(u, x[c][kb], acc[c][t]);
      }
    if (i + 1 < a.per_wave) load(j + 4);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int p = 32 * j + t0 + 4 * c;
      const long long row = (long long)min(p, a.table_rows - 1) * HD + 4 * g;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const f32x4 cs = *reinterpret_cast<const f32x4*>(a.cos_t + row + 16 * t);
        const f32x4 sn = *reinterpret_cast<const f32x4*>(a.sin_t + row + 16 * t);
        bf16x4 o;
#pragma unroll
        for (int q = 0; q < 4; q += 2) {
          const float x0 = acc[c][t][q], x1 = acc[c][t][q + 1];
          o[q] = (__bf16)fmaf(x0, cs[q], -(x1 * sn[q]));
          o[q + 1] = (__bf16)fmaf(x1, cs[q], x0 * sn[q]);
        }
        if constexpr (TILED) {
          *reinterpret_cast<bf16x4*>(k + tiled_k_offset(p, 16 * t + 4 * g, HD)) = o;
        } else if (p < a.S) {
          *reinterpret_cast<bf16x4*>(k + (long long)p * HD + 16 * t + 4 * g) = o;
        }
      }
    }
  }
}

template <bool TILED>
int launch_rebuild(int r, const RebuildArgs& a, dim3 grid, hipStream_t s) {
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PALU_OK : fail(PALU_EHIP, "palu_naive_decode: rebuild launch: %s", hipGetErrorString(e));
  };
  switch (r) {
    case 32: return go(palu_rebuild_kernel<TILED, 32>);
    case 64: return go(palu_rebuild_kernel<TILED, 64>);
    case 96: return go(palu_rebuild_kernel<TILED, 96>);
    case 128: return go(palu_rebuild_kernel<TILED, 128>);
  }
  if constexpr (TILED) {
    switch (r) {
      case 16: return go(palu_rebuild_kernel<TILED, 16>);
      case 48: return go(palu_rebuild_kernel<TILED, 48>);
      case 80: return go(palu_rebuild_kernel<TILED, 80>);
      case 112: return go(palu_rebuild_kernel<TILED, 112>);
    }
  }
  return fail(PALU_EUNSUPPORTED, "palu_naive_decode: r_k %d", r);
}

size_t key_bytes(int batch, int n_kv, int recon_len) { return ((size_t)batch * n_kv * recon_len * HD * 2 + 255) & ~(size_t)255; }

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

extern "C" size_t palu_naive_workspace_bytes(int batch, int n_kv, int recon_len, int r_v) {
  if (batch <= 0 || n_kv <= 0 || recon_len <= 0 || r_v <= 0 || (long long)batch * n_kv > 65535) return 0;
  return key_bytes(batch, n_kv, recon_len) + decode_ws_bytes(batch * n_kv, r_v);
}

extern "C" int palu_naive_decode(const void* q, const void* k_latent, const void* u_k, const float* cos_table,
                                 const float* sin_table, int table_rows, const void* v_latent, const int32_t* cur_pos,
                                 void* out, float scale, int batch, int n_q, int n_kv, int seq_len, int recon_len, int r_k,
                                 int r_v, int out_dtype, int cache_layout, int deterministic, void* workspace,
                                 size_t workspace_bytes, hipStream_t stream) {
  palu::g_err[0] = 0;
  const char* who = "palu_naive_decode";
  const bool tiled = cache_layout == PALU_LAYOUT_TILED;
  if (!u_k || !cos_table || !sin_table || !workspace) return fail(PALU_EINVAL, "%s: a required pointer is null", who);
  if (recon_len <= 0 || recon_len > seq_len || (tiled && (recon_len % 32 || seq_len % 32)))
    return fail(PALU_EINVAL, "%s: recon_len %d of a cache of %d positions (multiples of 32 when tiled)", who, recon_len, seq_len);
  if (r_k <= 0 || r_k > HD || r_k % (tiled ? 16 : 32))
    return fail(PALU_EINVAL, "%s: r_k %d (multiples of 32 up to %d; of 16 for tiled caches)", who, r_k, HD);
  if (batch <= 0 || n_kv <= 0) return fail(PALU_EINVAL, "%s: batch and head counts must be positive", who);
  if ((long long)batch * n_kv > 65535) return fail(PALU_EUNSUPPORTED, "%s: batch * n_kv exceeds the grid limit", who);
  // The flash-decode's V widths, checked ahead of the rebuild's launch: the workspace's size depends on a valid one.
  if (r_v < 32 || r_v > HD || r_v % (tiled ? 16 : 32))
    return fail(PALU_EUNSUPPORTED, "%s: r_v %d (multiples of 32 up to %d; of 16 from 32 on for tiled caches)", who, r_v, HD);
  if (table_rows < recon_len) return fail(PALU_EINVAL, "%s: %d table rows for %d positions", who, table_rows, recon_len);
  if (!al16(u_k) || !al16(cos_table) || !al16(sin_table) || !al16(workspace))
    return fail(PALU_EINVAL, "%s: 16-byte alignment required", who);
  const size_t need = palu_naive_workspace_bytes(batch, n_kv, recon_len, r_v);
  if (workspace_bytes < need)
    return fail(PALU_EINVAL, "%s: workspace of %zu bytes needed (palu_naive_workspace_bytes), got %zu", who, need, workspace_bytes);
  DecodeArgs a;
  const size_t kb = key_bytes(batch, n_kv, recon_len);
  if (int rc = palu::flash_setup(a, q, workspace, v_latent, cur_pos, out, scale, batch, n_q, n_kv, recon_len, r_v, out_dtype,
                                 cache_layout, deterministic, static_cast<char*>(workspace) + kb, workspace_bytes - kb, who))
    return rc;
  if (!k_latent || !al16(k_latent)) return fail(PALU_EINVAL, "%s: k_latent must be a 16-byte aligned cache", who);
  a.k_sg = (long long)recon_len * HD;
  a.k_sb = a.k_sg * n_kv;
  a.v_sg = (long long)seq_len * r_v;
  a.v_sb = a.v_sg * n_kv;
  // One block per wave until that gives two workgroups a CU, then more blocks per staged u_k^T.
  const int nblk = (recon_len + BLK - 1) / BLK;
  const long long groups = (long long)batch * n_kv * ((nblk + 3) / 4);
  const int per_wave = (int)std::min<long long>(8, std::max<long long>(1, groups / 512));
  const int chunks = (nblk + 4 * per_wave - 1) / (4 * per_wave);
  const RebuildArgs ra{static_cast<const __bf16*>(k_latent), static_cast<const __bf16*>(u_k), cos_table, sin_table, cur_pos,
                       static_cast<__bf16*>(workspace), n_kv, seq_len, recon_len, table_rows, chunks, per_wave};
  const dim3 grid((unsigned)(batch * n_kv) * (unsigned)chunks);
  if (int rc = tiled ? launch_rebuild<true>(r_k, ra, grid, stream) : launch_rebuild<false>(r_k, ra, grid, stream)) return rc;
  return dispatch_full(a, tiled, false, r_v, out_dtype == PALU_DTYPE_F32, stream);
}
