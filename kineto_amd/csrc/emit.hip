/*
 * emit.hip — stage 4b: the activities formatted into the document, for traces of any size beyond the small
 * ones (small.hip).  A file of its own because it takes twice as long to compile as everything else together.
 */
#include "gpu_common.h"

namespace ktj {
namespace gpu {

/* ------------------------------------------------------------------------------------------ */
/* stage 4b: emit.  Workgroup k owns the output bytes [k*T, (k+1)*T) of the whole document      */
/* (clipped to the activity section), so every global store is an aligned 16-byte store.  The    */
/* first activity of every tile is found once by k_tile_starts (binary search in the offsets);   */
/* the emit workgroup formats one activity per lane into LDS through a 64-bit accumulator        */
/* (literals are immediates, digits are packed arithmetically, no per-byte loads), with clipping */
/* (an activity straddling a tile boundary is formatted by both tiles), copies dictionary        */
/* strings with whole wavefronts, and flushes the tile.  T is chosen by the host so that a tile  */
/* holds about as many activities as the workgroup has lanes.                                    */
/* ------------------------------------------------------------------------------------------ */
#define EMIT_THREADS 128
#define EMIT_MAX_JOBS 512

__global__ void k_tile_starts(const uint64_t* offs, uint64_t n, uint64_t prefix_len, uint32_t tile, uint64_t first_tile,
                              uint32_t n_tiles, uint32_t* start) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t > n_tiles) return;
  if (t == n_tiles) { start[t] = (uint32_t)n; return; }
  const uint64_t t0 = (first_tile + t) * (uint64_t)tile;
  const uint64_t lo = (t0 > prefix_len ? t0 : prefix_len) - prefix_len;
  uint64_t a = 0, b = n; /* first record with offs[r + 1] > lo */
  while (a < b) { const uint64_t m = (a + b) >> 1; if (offs[m + 1] > lo) b = m; else a = m + 1; }
  start[t] = (uint32_t)a;
}

__global__ void __launch_bounds__(EMIT_THREADS)
k_emit(const MatRow* mat, const uint32_t* perm, const uint64_t* offs, uint64_t n, EmitCtx ctx, char* out,
       uint64_t prefix_len, uint64_t act_bytes, uint32_t tile, uint64_t first_tile, const uint32_t* start) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* buf = smem;                                                   /* tile bytes */
  CopyJob* jobs = reinterpret_cast<CopyJob*>(smem + tile);            /* EMIT_MAX_JOBS */
  uint32_t* n_jobs = reinterpret_cast<uint32_t*>(smem + tile + EMIT_MAX_JOBS * sizeof(CopyJob));

  const uint64_t t0 = (first_tile + blockIdx.x) * (uint64_t)tile;     /* absolute, multiple of the tile size */
  const uint64_t abs_lo = t0 > prefix_len ? t0 : prefix_len;
  const uint64_t abs_end = prefix_len + act_bytes;
  const uint64_t abs_hi = t0 + tile < abs_end ? t0 + tile : abs_end;
  if (abs_lo >= abs_hi) return;
  const int32_t lo = (int32_t)(abs_lo - t0), hi = (int32_t)(abs_hi - t0); /* tile-local */

  const uint64_t r0 = start[blockIdx.x];
  uint64_t r1 = start[blockIdx.x + 1];
  if (r1 < n && offs[r1] + prefix_len < abs_hi) ++r1;                  /* the straddler at the upper edge */

  if (threadIdx.x == 0) *n_jobs = 0;
  {
    uint4* z = reinterpret_cast<uint4*>(buf);
    const uint4 zero = make_uint4(0, 0, 0, 0);
    for (uint32_t k = threadIdx.x; k < tile / 16u; k += EMIT_THREADS) z[k] = zero;
  }
  __syncthreads();
  for (uint64_t r = r0 + threadIdx.x; r < r1; r += EMIT_THREADS) {
    const uint64_t o = offs[r];
    if (offs[r + 1] == o) continue; /* dropped or empty */
    const MatRow m = mat[perm[r]];
    TileWriter w;
    w.buf = buf; w.size = tile;
    w.jobs = jobs; w.n_jobs = n_jobs; w.max_jobs = EMIT_MAX_JOBS;
    w.begin((int32_t)((int64_t)(o + prefix_len) - (int64_t)t0));
    format_activity(w, m, ctx);
    w.end();
  }
  __syncthreads();
  {
    /* string copies: one job per 16-lane group; aligned 8-byte words in the middle (two aligned
     * global loads funnel-shifted into one aligned LDS store), single bytes at both ends */
    const uint32_t nj = *n_jobs < EMIT_MAX_JOBS ? *n_jobs : EMIT_MAX_JOBS;
    const uint32_t group = threadIdx.x >> 4, gl = threadIdx.x & 15u;
    for (uint32_t j = group; j < nj; j += (EMIT_THREADS >> 4)) {
      const CopyJob job = jobs[j];
      uint32_t headb = (8u - ((uint32_t)job.dst & 7u)) & 7u;
      if (headb > job.len) headb = job.len;
      if (gl < headb) buf[job.dst + (int32_t)gl] = job.src[gl];
      const uint32_t words = (job.len - headb) >> 3;
      const uintptr_t sa = (uintptr_t)(job.src + headb);
      const uint32_t sh = (uint32_t)(sa & 7u) * 8u;
      const uint64_t* sp = reinterpret_cast<const uint64_t*>(sa & ~(uintptr_t)7);
      uint64_t* dp = reinterpret_cast<uint64_t*>(buf + job.dst + (int32_t)headb);
      for (uint32_t k = gl; k < words; k += 16u) {
        uint64_t v = sp[k];
        if (sh) v = (v >> sh) | (sp[k + 1] << (64u - sh));
        dp[k] = v;
      }
      const uint32_t done = headb + words * 8u;
      if (gl < job.len - done) buf[job.dst + (int32_t)(done + gl)] = job.src[done + gl];
    }
  }
  __syncthreads();
  /* flush: unaligned head bytes (first tile only), 16-byte body, tail bytes */
  char* g = out + abs_lo;
  const char* s = buf + lo;
  const uint32_t nbytes = (uint32_t)(hi - lo);
  uint32_t pre = (uint32_t)((16u - (uint32_t)((uintptr_t)g & 15u)) & 15u);
  if (pre > nbytes) pre = nbytes;
  for (uint32_t k = threadIdx.x; k < pre; k += EMIT_THREADS) g[k] = s[k];
  const uint32_t body = (nbytes - pre) / 16u;
  {
    uint4* gv = reinterpret_cast<uint4*>(g + pre);
    const uint4* sv = reinterpret_cast<const uint4*>(s + pre);
    for (uint32_t k = threadIdx.x; k < body; k += EMIT_THREADS) gv[k] = sv[k];
  }
  for (uint32_t k = pre + body * 16u + threadIdx.x; k < nbytes; k += EMIT_THREADS) g[k] = s[k];
}

/* Direct variant: one lane per activity; blocks of 16 bytes, aligned in the document (see
 * BlockWriter for who writes the blocks that two activities share).  Finished blocks wait in the
 * lane's stage in LDS, one 128-byte line of the document and the beginning of the next, and a line
 * leaves when it is complete (a line written in pieces some microseconds apart leaves the L2 cache
 * once per piece): at the points where the whole wavefront meets — after the head of the event,
 * after its args if some lane's stage is full by then, and after the flow event — the four lanes
 * of a quad store each other's blocks, 64 contiguous bytes per quad and instruction, and in between
 * a lane whose stage is nearly full stores its line itself (BlockWriter::relief).  Lanes without an activity stay until the end
 * for the quads' sake.  The document's prefix and suffix are already in place when this kernel
 * runs; the first and the last activity merge with them. */
template <bool LIST> /* only the activities on the list, or all where the weaver prints none */
__global__ void __launch_bounds__(KTJ_BLOCK) __attribute__((amdgpu_waves_per_eu(3)))
k_emit_direct(const char* rows, const uint32_t* perm, const uint64_t* offs, const uint8_t* kind_sorted,
              EmitCtx ctx, char* out, uint64_t prefix_len, const Scalars* sc, const uint32_t* left) {
  const bool all = !LIST || sc->no_text;
  const uint64_t n_rows = sc->emit_rows, n_mine = all ? n_rows : n_rows ? sc->n_left : 0u;
  if ((uint64_t)blockIdx.x * blockDim.x >= n_mine) return;
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, o = 0;
  uint32_t row = 0;
  bool active = i < n_mine;
  if (!all && active) i = left[i];
  /* A wavefront that has just started comes first on its SIMD until the loads of its joined row are
   * on their way (two dependent loads with a few instructions between them, which would otherwise
   * queue behind the formatting of the two older wavefronts): config 3 4.70 -> 4.61 ms, config 4
   * 2.12 -> 2.07 ms.  Priority 1, 2 or 3: the same.  Kept up until the name is copied, lowered in
   * steps, lowered behind the branch below or before the row's loads: slower or no gain; a
   * scheduling barrier in place of the priority: no gain. */
  __builtin_amdgcn_s_setprio(3);
  if (active) { row = perm[i]; o = offs[i]; active = offs[i + 1] != o; } /* one wait for both */
  MatRow m;
  BlockWriter w;
  w.stage_init((uint32_t)threadIdx.x * (KTJ_STAGE_BLOCKS * 16u));
  ActivityParts<BlockWriter> parts;
  if (active) {
    m = *reinterpret_cast<const MatRow*>(rows + (uint64_t)row * (LIST ? sizeof(weave::TextRow) : sizeof(MatRow)));
    __builtin_amdgcn_s_setprio(0); /* (a wavefront without any activity keeps it: it ends at once) */
    w.begin(out, prefix_len + o, !i ? 0u : LIST ? tail_kind_at(kind_sorted, reinterpret_cast<const weave::TextRow*>(rows), perm, i - 1, ctx) : kind_sorted[i - 1], i == 0);
    w.stage_follow();
    format_head(w, m, ctx, parts);
  }
  w.flush(false);
  if (active) format_args(w, m, ctx, parts);
  w.flush_if_full();
  if (active) {
    format_flow(w, m, ctx, parts);
    w.end(i + 1 == n_rows);
  }
  w.flush(true);
}
hipError_t emit_direct(const void* rows, const uint32_t* perm, const uint64_t* offs, const uint8_t* kind_sorted, uint64_t n_most, EmitCtx ctx,
                       char* out, uint64_t prefix_len, const Scalars* sc, const uint32_t* left, hipStream_t st) {
  if (n_most == 0) return hipSuccess;
  const size_t stage_lds = (size_t)KTJ_BLOCK * KTJ_STAGE_BLOCKS * 16u;
  hipLaunchKernelGGL(left ? k_emit_direct<true> : k_emit_direct<false>, dim3(grid_for(n_most, KTJ_BLOCK)), dim3(KTJ_BLOCK), stage_lds, st, static_cast<const char*>(rows), perm, offs,
                     kind_sorted, ctx, out, prefix_len, sc, left);
  return KTJ_LAUNCH_CHECK();
}

uint32_t emit_tile_bytes(uint64_t act_bytes, uint64_t n_rows) {
  /* about 0.85 activities per lane, in steps of 4 KiB, between 8 and 40 KiB */
  const uint64_t avg = n_rows ? act_bytes / n_rows : 512;
  uint64_t t = (avg * EMIT_THREADS * 85 / 100 + 4095) / 4096 * 4096;
  if (t < 8192) t = 8192;
  if (t > 40960) t = 40960;
  return (uint32_t)t;
}
uint64_t emit_tile_count(uint64_t prefix_len, uint64_t act_bytes, uint32_t tile) {
  if (act_bytes == 0) return 0;
  return (prefix_len + act_bytes - 1) / tile - prefix_len / tile + 1;
}

hipError_t emit(const MatRow* mat, const uint32_t* perm, const uint64_t* offs, uint64_t n, EmitCtx ctx, char* out,
                uint64_t prefix_len, uint64_t act_bytes, uint32_t tile, uint32_t* tile_start, hipStream_t st) {
  if (act_bytes == 0) return hipSuccess;
  const uint64_t first_tile = prefix_len / tile;
  const uint32_t tiles = (uint32_t)emit_tile_count(prefix_len, act_bytes, tile);
  hipLaunchKernelGGL(k_tile_starts, dim3(grid_for((uint64_t)tiles + 1, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, offs, n,
                     prefix_len, tile, first_tile, tiles, tile_start);
  const size_t lds = (size_t)tile + EMIT_MAX_JOBS * sizeof(CopyJob) + 16;
  hipLaunchKernelGGL(k_emit, dim3(tiles), dim3(EMIT_THREADS), lds, st, mat, perm, offs, n, ctx, out, prefix_len,
                     act_bytes, tile, first_tile, (const uint32_t*)tile_start);
  return KTJ_LAUNCH_CHECK();
}

}  // namespace gpu
}  // namespace ktj
