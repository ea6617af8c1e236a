/*
 * kernels.hip — HIP kernels of the trace post-processing engine, written for gfx950 (CDNA4):
 * 64-wide wavefronts, ballot/popcount based ranking, LDS-staged tiles, 16-byte lanes.
 *
 * Nothing here is a dense contraction, so there is no MFMA; every kernel is bound by HBM (or,
 * for the hash joins, by random 64-byte sector access).  Stage by stage:
 *   0  dictionary   strings → name view (logger's name pipeline) and arg view (sanitised)
 *   1  decode       packed activity records → columns, through LDS so that global reads are
 *                   lane-consecutive 16-byte loads
 *   2  convert/join clock model, window filter, external-correlation join, runtime↔device join,
 *                   stream back-fill with dense per-device stream indices
 *   3  order        dense ranks of (device, resource), 64-bit composite keys, stable LSD radix sort
 *   4  size/emit    exact byte length per activity, device-wide exclusive scan, output-partitioned
 *                   tiles formatted in LDS and flushed with aligned 16-byte stores
 */
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <mutex>

#include "gpu_common.h"

namespace ktj {
namespace gpu {

/* Returns the slot holding `key`, inserting it if absent; KTJ_NOSLOT when no free slot lies within
 * KTJ_TABLE_PROBES slots of the key's home slot (a table that is at most half full never gets
 * there; one that is close to full does at once, so that an input with far too many distinct keys
 * costs a bounded number of probes per row and is reported instead of crawling). */
__device__ uint32_t table_insert(uint64_t* keys, uint32_t mask, uint64_t key) {
  if (key == KTJ_EMPTY_KEY) { keys[mask + 1u] = 0; return mask + 1u; }
  uint32_t slot = (uint32_t)hash64(key) & mask;
  for (uint32_t probe = 0; probe <= mask && probe < KTJ_TABLE_PROBES; ++probe) {
    uint64_t cur = keys[slot];
    if (cur == key) return slot;
    if (cur == KTJ_EMPTY_KEY) {
      unsigned long long prev = atomicCAS((unsigned long long*)&keys[slot], (unsigned long long)KTJ_EMPTY_KEY,
                                          (unsigned long long)key);
      if (prev == KTJ_EMPTY_KEY || prev == key) return slot;
    }
    slot = (slot + 1u) & mask;
  }
  return KTJ_NOSLOT;
}
/* table_insert for a table with a documented limit on its distinct keys: the key that would be
 * number `limit` + 1 is refused (KTJ_NOSLOT), whatever room the table still has, so that a trace is
 * accepted or refused by the count the limit names and not by how its keys happen to hash. */
__device__ uint32_t table_insert_counted(uint64_t* keys, uint32_t mask, uint64_t key, unsigned int* count, uint32_t limit) {
  if (key == KTJ_EMPTY_KEY) {
    if (atomicExch((unsigned long long*)&keys[mask + 1u], 0ULL) != 0ULL && atomicAdd(count, 1u) >= limit) return KTJ_NOSLOT;
    return mask + 1u;
  }
  uint32_t slot = (uint32_t)hash64(key) & mask;
  for (uint32_t probe = 0; probe <= mask && probe < KTJ_TABLE_PROBES; ++probe) {
    uint64_t cur = keys[slot];
    if (cur == key) return slot;
    if (cur == KTJ_EMPTY_KEY) {
      if (*(volatile unsigned int*)count >= limit) return KTJ_NOSLOT; /* full by count: take no further slot */
      unsigned long long prev = atomicCAS((unsigned long long*)&keys[slot], (unsigned long long)KTJ_EMPTY_KEY,
                                          (unsigned long long)key);
      if (prev == KTJ_EMPTY_KEY) return atomicAdd(count, 1u) >= limit ? KTJ_NOSLOT : slot;
      if (prev == key) return slot;
    }
    slot = (slot + 1u) & mask;
  }
  return KTJ_NOSLOT;
}
__device__ uint32_t table_find(const uint64_t* keys, uint32_t mask, uint64_t key) {
  if (key == KTJ_EMPTY_KEY) return keys[mask + 1u] == 0 ? mask + 1u : KTJ_NOSLOT;
  uint32_t slot = (uint32_t)hash64(key) & mask;
  for (uint32_t probe = 0; probe <= mask && probe < KTJ_TABLE_PROBES; ++probe) {
    uint64_t cur = keys[slot];
    if (cur == key) return slot;
    if (cur == KTJ_EMPTY_KEY) return KTJ_NOSLOT;
    slot = (slot + 1u) & mask;
  }
  return KTJ_NOSLOT;
}

/* Join tables (Table).  Direct mode: slot = key - base.  Hash mode: slots are grouped in runs of
 * sixteen; a key lives at position (key + rotation) & 15 of a run, where the rotation and the
 * probe sequence over runs (double hashing) depend only on the remaining key bits.  Sixteen
 * consecutive ids therefore share one run, while strided or clustered ids still spread like under
 * a full hash and a collision costs one probe in another run rather than a walk through a full one. */
struct ProbeSeq {
  uint32_t run, step, low, runs;
  __device__ __forceinline__ ProbeSeq(uint64_t key, uint32_t n_runs) {
    const uint64_t h = hash64(key >> 4);
    runs = n_runs;
    run = __umulhi((uint32_t)h, runs);
    step = 1u + 2u * __umulhi((uint32_t)(h >> 32), runs >> 1); /* odd and below `runs`: visits every run, whose number is a power of two or a prime */
    low = ((uint32_t)key + (uint32_t)((h * 0x9E3779B97F4A7C15ULL) >> 60)) & 15u; /* ids sharing low bits still use all positions */
  }
  __device__ __forceinline__ uint32_t slot() const { return (run << 4) | low; }
  __device__ __forceinline__ void next() { run += step; run = run >= runs ? run - runs : run; }
};
/* A table as its plan has it, read once: the stores of a pass over rows would have it read again for each (11 million kernels: links 388 -> 373 us). */
struct TableView { uint64_t* keys; uint32_t mask, runs, keyed_direct, direct, no_heads; uint64_t base, span; };
__device__ __forceinline__ TableView view(const Table& t) { return TableView{t.keys, t.mask, t.runs, t.keyed_direct, t.ctl->direct, t.ctl->no_heads, t.ctl->base, t.ctl->span}; }
/* Returns the slot of `key`, inserting it if absent; KTJ_NOSLOT when the table is full (hash
 * mode) or the key lies outside the planned range (direct mode; cannot happen for keys that were
 * part of the range computation). */
__device__ uint32_t slot_insert(const TableView& t, uint64_t key) {
  if (t.direct) {
    if (t.keyed_direct && key == KTJ_EMPTY_KEY) { t.keys[t.mask + 1u] = 0; return t.mask + 1u; }
    const uint64_t idx = key - t.base;
    if (idx > t.span) return KTJ_NOSLOT;
    if (t.keyed_direct && t.keys[idx] != key) t.keys[idx] = key; /* every writer stores the same value */
    return (uint32_t)idx;
  }
  if (key == KTJ_EMPTY_KEY) { t.keys[t.mask + 1u] = 0; return t.mask + 1u; }
  ProbeSeq p(key, t.runs);
  for (uint32_t probe = 0; probe < t.runs; ++probe, p.next()) {
    const uint32_t slot = p.slot();
    uint64_t cur = t.keys[slot];
    if (cur == key) return slot;
    if (cur == KTJ_EMPTY_KEY) {
      unsigned long long prev = atomicCAS((unsigned long long*)&t.keys[slot], (unsigned long long)KTJ_EMPTY_KEY,
                                          (unsigned long long)key);
      if (prev == KTJ_EMPTY_KEY || prev == key) return slot;
    }
  }
  return KTJ_NOSLOT;
}
/* In direct mode without stored keys every id inside the range has a slot; one that was never
 * inserted reads as empty per-slot values. */
__device__ uint32_t slot_find(const TableView& t, uint64_t key) {
  if (t.direct) {
    if (t.keyed_direct && key == KTJ_EMPTY_KEY) return t.keys[t.mask + 1u] == 0 ? t.mask + 1u : KTJ_NOSLOT;
    const uint64_t idx = key - t.base;
    if (idx > t.span) return KTJ_NOSLOT;
    if (t.keyed_direct && t.keys[idx] != key) return KTJ_NOSLOT;
    return (uint32_t)idx;
  }
  if (key == KTJ_EMPTY_KEY) return t.keys[t.mask + 1u] == 0 ? t.mask + 1u : KTJ_NOSLOT;
  ProbeSeq p(key, t.runs);
  for (uint32_t probe = 0; probe < t.runs; ++probe, p.next()) {
    const uint32_t slot = p.slot();
    uint64_t cur = t.keys[slot];
    if (cur == key) return slot;
    if (cur == KTJ_EMPTY_KEY) return KTJ_NOSLOT;
  }
  return KTJ_NOSLOT;
}

__device__ __forceinline__ uint32_t slot_insert(const Table& t, uint64_t key) { return slot_insert(view(t), key); }
__device__ __forceinline__ uint32_t slot_find(const Table& t, uint64_t key) { return slot_find(view(t), key); }

/* Sums a per-thread count over the workgroup and adds it to a global counter with one atomic per
 * workgroup (a single hot address serialises atomics in L2, so they must be rare).  Must be
 * reached by every thread of the workgroup.  block_add_to: a counter of its own address, for counts
 * that are zero in nearly every workgroup; block_add: one of the sharded counters of Scalars. */
__device__ __forceinline__ uint32_t block_sum(uint32_t mine) { /* the sum, in thread 0 */
  __shared__ uint32_t partial[16]; /* of up to 1024 threads */
  const uint32_t w = wave_sum_u32(mine);
  __syncthreads();
  if (lane_id() == 0) partial[threadIdx.x >> 6] = w;
  __syncthreads();
  uint32_t t = 0;
  if (threadIdx.x == 0)
    for (uint32_t k = 0; k < (blockDim.x >> 6); ++k) t += partial[k];
  return t;
}
__device__ __forceinline__ void block_add_to(unsigned long long* counter, uint32_t mine) {
  const uint32_t t = block_sum(mine);
  if (threadIdx.x == 0 && t) atomicAdd(counter, (unsigned long long)t);
}
__device__ __forceinline__ void block_add(Scalars* sc, int which, uint32_t mine) {
  const uint32_t t = block_sum(mine);
  if (threadIdx.x == 0 && t) atomicAdd(&sc->shard[blockIdx.x & (KTJ_COUNTER_SHARDS - 1u)][which], (unsigned long long)t);
}

/* two of them that are one or none per thread */
__device__ __forceinline__ void block_add_two(Scalars* sc, int which, bool mine, int which2, bool mine2) {
  const uint32_t t = block_sum((mine ? 1u : 0u) | (mine2 ? 0x10000u : 0u));
  if (threadIdx.x == 0 && t) {
    unsigned long long* const counter = sc->shard[blockIdx.x & (KTJ_COUNTER_SHARDS - 1u)];
    if (t & 0xFFFFu) atomicAdd(&counter[which], (unsigned long long)(t & 0xFFFFu));
    if (t >> 16) atomicAdd(&counter[which2], (unsigned long long)(t >> 16));
  }
}

__global__ void k_fill_u64(uint64_t* p, uint64_t v, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
hipError_t fill_u64(uint64_t* p, uint64_t v, uint64_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(n, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, p, v, n);
  return KTJ_LAUNCH_CHECK();
}
hipError_t fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, p, v, n);
  return KTJ_LAUNCH_CHECK();
}
/* What a pass needs before its records are looked at, in one launch: the scalars (first workgroup), the
 * dictionary views (a wavefront per string) and the fills of the small tables (the last workgroups). */
#define BEGIN_FILL_BLOCKS 128u
__global__ void __launch_bounds__(KTJ_BLOCK)
k_begin(Scalars* s, FillJobs jobs, const char* blob, const uint64_t* off, uint32_t n_strings, uint32_t dict_blocks, DictEntry* entries,
        char* name_blob, char* arg_blob) {
  if (blockIdx.x == 0) {
    for (uint32_t k = threadIdx.x; k < KTJ_COUNTER_SHARDS * 16u; k += KTJ_BLOCK) {
      s->shard[k / 16u][k % 16u] = 0;
      s->range_shard[k / 16u][k % 16u] = k % 2u ? 0 : ~0ULL; /* lo, hi of each range: empty */
    }
    if (threadIdx.x == 0) {
      s->ts_min_biased = ~0ULL; s->ts_max_biased = 0;
      s->out_of_range = 0; s->out_of_order = 0; s->n_flow = 0; s->n_linked = 0; s->n_blank_names = 0; s->n_valid = 0;
      s->n_unresolved = 0; s->n_sync_typed = 0; s->n_device_orphans = 0; s->error = 0; s->have_stream_src = 0; s->n_dev_ranks = 0; s->n_res_ranks = 0; s->n_dense = 0; s->runtime_ids_repeat = 0;
      s->n_queues = 0; s->n_sync_rows = 0; s->ext_ids_repeat = 0; s->n_plain = 0; s->n_left = 0; s->no_text = 0;
      s->sort.ts_bits = s->sort.res_bits = s->sort.key_bits = s->sort.low_bits = s->sort.n_dev = 0;
      for (int k = 0; k < KTJ_DONE_COUNT; ++k) s->done[k] = 0;
      for (uint32_t k = 0; k < KTJ_PART_SLOTS; ++k) s->part_done[k] = 0;
      for (int k = 0; k < KTJ_CLOCK_COUNT; ++k) s->clock[k] = 0;
      stage_clock(s, KTJ_CLOCK_BEGIN);
    }
  } else if (blockIdx.x <= dict_blocks) {
    const uint32_t id = (blockIdx.x - 1u) * (KTJ_BLOCK >> 6) + (threadIdx.x >> 6);
    if (id < n_strings) dict_string(blob, off, id, entries, name_blob, arg_blob);
  } else {
    const uint32_t b = blockIdx.x - 1u - dict_blocks;
    for (uint32_t j = 0; j < jobs.count; ++j) {
      const uint64_t n = jobs.n[j], v = jobs.value[j];
      if (jobs.bytes_each[j] == 8) {
        uint64_t* p = static_cast<uint64_t*>(jobs.p[j]);
        for (uint64_t i = (uint64_t)b * KTJ_BLOCK + threadIdx.x; i < n; i += BEGIN_FILL_BLOCKS * KTJ_BLOCK) p[i] = v;
      } else {
        uint32_t* p = static_cast<uint32_t*>(jobs.p[j]);
        for (uint64_t i = (uint64_t)b * KTJ_BLOCK + threadIdx.x; i < n; i += BEGIN_FILL_BLOCKS * KTJ_BLOCK) p[i] = (uint32_t)v;
      }
    }
  }
}
hipError_t begin_pass(Scalars* s, const FillJobs& jobs, const char* blob, const uint64_t* off, uint32_t n_strings, DictEntry* entries,
                      char* name_blob, char* arg_blob, hipStream_t st) {
  static_assert((KTJ_COUNTER_SHARDS & (KTJ_COUNTER_SHARDS - 1u)) == 0, "a workgroup's copy is its index modulo the number of copies");
  const uint32_t dict_blocks = grid_for(n_strings, KTJ_BLOCK >> 6);
  hipLaunchKernelGGL(k_begin, dim3(1u + dict_blocks + BEGIN_FILL_BLOCKS), dim3(KTJ_BLOCK), 0, st, s, jobs, blob, off, n_strings, dict_blocks,
                     entries, name_blob, arg_blob);
  return KTJ_LAUNCH_CHECK();
}

/* ------------------------------------------------------------------------------------------ */
/* static scratch array: the working memory of ktj_process_noalloc.  Every GPU the library runs  */
/* on holds its own copy, at its own address, until the process ends.  In host code the array's  */
/* name is only a handle for hipGetSymbolAddress; everything else uses the looked-up address.    */
/* ------------------------------------------------------------------------------------------ */
static __device__ __align__(256) unsigned char scratch[KTJ_NOALLOC_SCRATCH_BYTES];
#define KTJ_MAX_DEVICES 64
static void* g_scratch_ptr[KTJ_MAX_DEVICES];
static std::mutex g_scratch_lock;

hipError_t scratch_address(int device, void** ptr, size_t* bytes) {
  *ptr = nullptr;
  *bytes = 0;
  if (device < 0 || device >= KTJ_MAX_DEVICES) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> guard(g_scratch_lock);
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    const hipError_t rc = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (rc != hipSuccess) return rc;
    g_scratch_ptr[device] = p;
  }
  *ptr = g_scratch_ptr[device];
  *bytes = KTJ_NOALLOC_SCRATCH_BYTES;
  return hipSuccess;
}

/* ------------------------------------------------------------------------------------------ */
/* exclusive scan: per-block sums → scan of the sums (one block) → per-block scan               */
/* ------------------------------------------------------------------------------------------ */
#define SCAN_ITEMS 8
#define SCAN_TILE (KTJ_BLOCK * SCAN_ITEMS)

#define SCAN_MAX_WAVES 16 /* workgroups of up to 1024 lanes */
/* a lane's SCAN_ITEMS consecutive values: two 16-byte loads where the whole run is inside the input
 * (the inputs are 16-byte aligned device buffers), single values at the end */
__device__ __forceinline__ void scan_load_items(const uint32_t* in, uint64_t n, uint64_t base, uint32_t (&v)[SCAN_ITEMS]) {
  static_assert(SCAN_ITEMS == 8, "two uint4 per lane");
  if (base + SCAN_ITEMS <= n) {
    const uint4 a = *reinterpret_cast<const uint4*>(in + base), b = *reinterpret_cast<const uint4*>(in + base + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
    for (int k = 0; k < SCAN_ITEMS; ++k) v[k] = base + k < n ? in[base + k] : 0u;
  }
}
__device__ __forceinline__ uint64_t block_exclusive_scan_u64(uint64_t v, uint64_t* lds_wave /* SCAN_MAX_WAVES */, uint64_t* total) {
  /* inclusive scan inside the wave */
  unsigned long long x = v;
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long y = __shfl_up(x, (unsigned)o);
    if ((int)lane_id() >= o) x += y;
  }
  const uint32_t w = threadIdx.x >> 6;
  if (lane_id() == 63) lds_wave[w] = x;
  __syncthreads();
  uint64_t base = 0, tot = 0;
  for (uint32_t k = 0; k < (blockDim.x >> 6); ++k) {
    const uint64_t s = lds_wave[k];
    if (k < w) base += s;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return base + x - v;
}

__global__ void k_scan_sums(const uint32_t* in, uint64_t n, uint64_t* sums) {
  __shared__ uint64_t lds_wave[SCAN_MAX_WAVES];
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
  uint32_t v[SCAN_ITEMS];
  scan_load_items(in, n, base, v);
  uint64_t s = 0;
  for (int k = 0; k < SCAN_ITEMS; ++k) s += v[k];
  uint64_t tot;
  block_exclusive_scan_u64(s, lds_wave, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}
/* one block: sums[0..m) → exclusive prefix in place, grand total → sums[m] */
__global__ void k_scan_of_sums(uint64_t* sums, uint64_t m) {
  __shared__ uint64_t lds_wave[SCAN_MAX_WAVES];
  uint64_t carry = 0;
  for (uint64_t base = 0; base < m; base += 8u * (uint64_t)blockDim.x) { /* eight neighbours per thread (one: 10 743 of them 20 us, now 13) */
    const uint64_t i = base + 8u * (uint64_t)threadIdx.x;
    uint64_t v[8], all = 0, tot;
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k) v[k] = sums[i + k < m ? i + k : m - 1];
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k) { v[k] = i + k < m ? v[k] : 0u; all += v[k]; }
    uint64_t ex = carry + block_exclusive_scan_u64(all, lds_wave, &tot);
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k) { if (i + k < m) sums[i + k] = ex; ex += v[k]; }
    carry += tot;
  }
  if (threadIdx.x == 0) sums[m] = carry;
}
template <typename OutT>
__global__ void k_scan_final(const uint32_t* in, uint64_t n, const uint64_t* sums, OutT* out) {
  __shared__ uint64_t lds_wave[SCAN_MAX_WAVES];
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
  uint32_t v[SCAN_ITEMS];
  scan_load_items(in, n, base, v);
  uint64_t s = 0;
  for (int k = 0; k < SCAN_ITEMS; ++k) s += v[k];
  uint64_t tot;
  uint64_t ex = block_exclusive_scan_u64(s, lds_wave, &tot) + sums[blockIdx.x];
  if (base + SCAN_ITEMS <= n) { /* the lane's run as 16-byte stores (the outputs are 16-byte aligned device buffers) */
    OutT r[SCAN_ITEMS];
    for (int k = 0; k < SCAN_ITEMS; ++k) { r[k] = (OutT)ex; ex += v[k]; }
    constexpr int PER = 16 / sizeof(OutT);
    typedef OutT vec __attribute__((ext_vector_type(PER)));
    vec* dst = reinterpret_cast<vec*>(out + base);
    for (int q = 0; q < SCAN_ITEMS / PER; ++q) {
      vec x;
      for (int j = 0; j < PER; ++j) x[j] = r[q * PER + j];
      dst[q] = x;
    }
  } else {
    for (int k = 0; k < SCAN_ITEMS; ++k) {
      if (base + k < n) out[base + k] = (OutT)ex;
      ex += v[k];
    }
  }
}

/* small inputs (one tile of SCAN_SMALL_THREADS lanes): the whole scan in one workgroup and one pass.
 * More tiles in one workgroup measured slower than the three launches over many workgroups. */
#define SCAN_SMALL_THREADS 1024u
#define SCAN_SMALL_MAX (SCAN_SMALL_THREADS * SCAN_ITEMS)
template <typename OutT>
__global__ void __launch_bounds__(SCAN_SMALL_THREADS) k_scan_small(const uint32_t* in, uint64_t n, OutT* out) {
  __shared__ uint64_t wave_sum[SCAN_SMALL_THREADS >> 6];
  const uint64_t base = (uint64_t)threadIdx.x * SCAN_ITEMS;
  uint32_t v[SCAN_ITEMS];
  uint64_t s = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) { v[k] = base + k < n ? in[base + k] : 0u; s += v[k]; }
  unsigned long long x = s; /* inclusive scan inside the wavefront, then over the wavefronts' sums */
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long y = __shfl_up(x, (unsigned)o);
    if ((int)lane_id() >= o) x += y;
  }
  const uint32_t w = threadIdx.x >> 6;
  if (lane_id() == 63) wave_sum[w] = x;
  __syncthreads();
  uint64_t before = 0, tot = 0;
  for (uint32_t k = 0; k < (SCAN_SMALL_THREADS >> 6); ++k) {
    const uint64_t t = wave_sum[k];
    if (k < w) before += t;
    tot += t;
  }
  uint64_t ex = before + x - s;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) { /* a lane reads and writes its own items only: in place is fine */
    if (base + k < n) out[base + k] = (OutT)ex;
    ex += v[k];
  }
}

uint64_t scan_tmp_elems(uint64_t n) { return (n + SCAN_TILE - 1) / SCAN_TILE + 2; }

hipError_t scan_u32_inplace(uint32_t* data, uint64_t n, uint64_t* tmp, hipStream_t st) {
  const uint64_t m = (n + SCAN_TILE - 1) / SCAN_TILE;
  if (m == 0) return hipSuccess;
  if (n <= SCAN_SMALL_MAX) {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_scan_small<uint32_t>), dim3(1), dim3(SCAN_SMALL_THREADS), 0, st, (const uint32_t*)data, n, data);
    return KTJ_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_scan_sums, dim3((unsigned)m), dim3(KTJ_BLOCK), 0, st, (const uint32_t*)data, n, tmp);
  hipLaunchKernelGGL(k_scan_of_sums, dim3(1), dim3(m > KTJ_BLOCK ? 1024 : KTJ_BLOCK), 0, st, tmp, m);
  /* every block reads its tile completely before writing it, and tiles do not overlap */
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_scan_final<uint32_t>), dim3((unsigned)m), dim3(KTJ_BLOCK), 0, st,
                     (const uint32_t*)data, n, (const uint64_t*)tmp, data);
  return KTJ_LAUNCH_CHECK();
}

/* ------------------------------------------------------------------------------------------ */
/* stage 1: decode, all record classes in one launch.  A workgroup pulls 256 packed records into   */
/* LDS with lane-consecutive 16-byte loads (fully coalesced), then each lane unpacks its own       */
/* record into the columns; the smallest and largest ids, from which the join tables are planned,  */
/* go to one of 64 copies of the ranges (atomics on a single address are carried out one after     */
/* the other, and an array of per-workgroup ranges takes another launch to reduce).                */
/* ------------------------------------------------------------------------------------------ */
template <typename Rec>
__device__ __forceinline__ const Rec* stage_records(const Rec* recs, uint64_t base, uint64_t n, uint4* stage, uint32_t* n_here) {
  constexpr uint32_t U = sizeof(Rec) / 16;
  const uint32_t cnt = (uint32_t)((n - base) < KTJ_BLOCK ? (n - base) : KTJ_BLOCK);
  const uint4* g = reinterpret_cast<const uint4*>(recs + base);
  const uint32_t last = cnt * U - 1u;
  uint4 x[U];
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) { const uint32_t i = threadIdx.x + k * KTJ_BLOCK; x[k] = g[i < last ? i : last]; }
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) { const uint32_t i = threadIdx.x + k * KTJ_BLOCK; stage[i < last ? i : last] = x[k]; }
  __syncthreads();
  *n_here = cnt;
  return reinterpret_cast<const Rec*>(stage);
}
/* Smallest and largest key of the workgroup's rows into the ranges of table `which`.  Must be reached by
 * every thread of the workgroup. */
__device__ __forceinline__ void block_key_range(bool has, uint64_t key, Scalars* sc, int which) {
  __shared__ unsigned long long s_lo[KTJ_BLOCK >> 6], s_hi[KTJ_BLOCK >> 6];
  unsigned long long lo = has ? key : ~0ULL, hi = has ? key : 0ULL;
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long l2 = __shfl_xor(lo, o), h2 = __shfl_xor(hi, o);
    lo = l2 < lo ? l2 : lo;
    hi = h2 > hi ? h2 : hi;
  }
  __syncthreads();
  if (lane_id() == 0) { s_lo[threadIdx.x >> 6] = lo; s_hi[threadIdx.x >> 6] = hi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t k = 1; k < (blockDim.x >> 6); ++k) { lo = s_lo[k] < lo ? s_lo[k] : lo; hi = s_hi[k] > hi ? s_hi[k] : hi; }
    unsigned long long* r = &sc->range_shard[blockIdx.x & (KTJ_COUNTER_SHARDS - 1u)][2 * which];
    if (lo <= hi) { atomicMin(&r[0], lo); atomicMax(&r[1], hi); }
  }
}
#define EXT_PER_BLOCK (KTJ_BLOCK * 8u)
__global__ void __launch_bounds__(KTJ_BLOCK) k_decode(DecodeJob J, Columns c, EmitCtx ctx, Scalars* sc) {
  __shared__ uint4 stage[KTJ_BLOCK * sizeof(ktj_runtime_rec) / 16];
  static_assert(sizeof(ktj_runtime_rec) >= sizeof(ktj_generic_rec) && sizeof(ktj_runtime_rec) >= sizeof(ktj_device_rec), "the largest record");
  if (blockIdx.x == 0 && threadIdx.x == 0 && J.whole_pass) stage_clock(sc, KTJ_CLOCK_DECODE);
  uint64_t b = blockIdx.x;
  uint32_t cnt;
  if (b < J.gb) {
    const ktj_generic_rec* l = stage_records(J.g, b * KTJ_BLOCK, J.ng, stage, &cnt);
    const bool has = threadIdx.x < cnt;
    if (J.whole_pass) block_key_range(has, has ? (uint64_t)(int64_t)l[threadIdx.x].id : 0, sc, KTJ_TBL_CPU);
    bool left = false;
    if (has) {
      const RowCols r = cols_generic(l[threadIdx.x], ctx);
      left = J.text && (r.meta & KTJ_M_VALID) && (weave::left_generic(l[threadIdx.x], r.dev, ctx, J.schemas_not_taken) || weave::far_apart(l[threadIdx.x].start_ns, l[0].start_ns));
      store_cols(c, J.first + b * KTJ_BLOCK + threadIdx.x, r, false);
    }
    /* rows that may need a Stream Sync row of their own are rare: the extra passes run only if any */
    block_add_two(sc, KTJ_CNT_SYNC_TYPED, has && l[threadIdx.x].type == KTJ_TYPE_CUDA_SYNC, KTJ_CNT_NOT_TEXT, left);
    return;
  }
  b -= J.gb;
  if (b < J.rb) {
    const ktj_runtime_rec* l = stage_records(J.r, b * KTJ_BLOCK, J.nr, stage, &cnt);
    const bool has = threadIdx.x < cnt;
    const uint64_t id = has ? l[threadIdx.x].id : 0;
    block_key_range(has, id, sc, KTJ_TBL_FULL);
    block_key_range(has, narrow_corr_key(id), sc, KTJ_TBL_NARROW);
    bool oor = false, left = false;
    if (has) {
      const RowCols r = cols_runtime(l[threadIdx.x], J.clk, J.win_start, J.win_end);
      oor = !(r.meta & KTJ_M_VALID);
      left = J.text && !oor && (weave::left_runtime(l[threadIdx.x], r.ts, r.dur, ctx, J.n_cids) || weave::far_apart(l[threadIdx.x].begin, l[0].begin));
      store_cols(c, J.ng + b * KTJ_BLOCK + threadIdx.x, r, false);
    }
    block_add_two(sc, KTJ_CNT_OUT_OF_RANGE, oor, KTJ_CNT_NOT_TEXT, left);
    return;
  }
  b -= J.rb;
  if (b < J.db) {
    const ktj_device_rec* l = stage_records(J.d, b * KTJ_BLOCK, J.nd, stage, &cnt);
    const bool has = threadIdx.x < cnt;
    block_key_range(has, has ? l[threadIdx.x].id : 0, sc, KTJ_TBL_FULL);
    bool oor = false, left = false;
    if (has) {
      const ktj_device_rec* d = &l[threadIdx.x];
      const uint64_t i = b * KTJ_BLOCK + threadIdx.x;
      const RowCols r = cols_device(*d, J.clk, J.win_start, J.win_end);
      oor = !(r.meta & KTJ_M_VALID);
      left = J.text && !oor && (weave::left_device(*d, r.ts, r.dur, r.res, ctx) || weave::far_apart(d->begin, l[0].begin));
      store_cols(c, J.ng + J.nr + i, r, true);
      J.queue[i] = d->queue;
    }
    block_add_two(sc, KTJ_CNT_OUT_OF_RANGE, oor, KTJ_CNT_NOT_TEXT, left);
    return;
  }
  b -= J.db; /* correlation ids of the external-correlation records */
  uint64_t lo = ~0ULL, hi = 0;
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k) {
    const uint64_t i = b * EXT_PER_BLOCK + k * KTJ_BLOCK + threadIdx.x;
    const uint64_t v = i < J.nx ? J.x[i].correlation : 0;
    if (i < J.nx) { lo = v < lo ? v : lo; hi = v > hi ? v : hi; }
  }
  block_key_range(lo <= hi, lo, sc, KTJ_TBL_NARROW);
  block_key_range(lo <= hi, hi, sc, KTJ_TBL_NARROW);
}
hipError_t decode(DecodeJob job, Columns c, EmitCtx ctx, Scalars* sc, hipStream_t st) {
  job.gb = grid_for(job.ng, KTJ_BLOCK); job.rb = grid_for(job.nr, KTJ_BLOCK); job.db = grid_for(job.nd, KTJ_BLOCK);
  const uint64_t blocks = (uint64_t)job.gb + job.rb + job.db + grid_for(job.nx, EXT_PER_BLOCK);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_decode, dim3((unsigned)blocks), dim3(KTJ_BLOCK), 0, st, job, c, ctx, sc);
  return KTJ_LAUNCH_CHECK();
}

/* ------------------------------------------------------------------------------------------ */
/* stage 2b: joins.  "Last writer wins" of the reference's sequential map updates becomes        */
/* atomicMax over the source row index; "first seen" becomes atomicMin over the arrival index.   */
/* What a device row takes over from "its" runtime row is then published into the table slot by  */
/* the winning row, so that a device row needs one slot of each table and no other row.          */
/* ------------------------------------------------------------------------------------------ */
/* The join tables' modes from the ranges of their keys, and what can be reached of them cleared (the
 * planned span in direct mode, the whole table otherwise).  Every workgroup reduces the 64 copies of the
 * ranges for itself; the first one leaves the plan for the kernels that follow. */
struct TableSpan { uint64_t n; bool direct; };
__device__ __forceinline__ void clear_keys(const Table& t, const TableSpan& s, uint64_t at, uint64_t step) {
  if (s.direct && !t.keyed_direct) return; /* keys are not used at all */
  for (uint64_t i = at; i < s.n; i += step) t.keys[i] = KTJ_EMPTY_KEY;
  if (at == 0) t.keys[t.mask + 1ull] = KTJ_EMPTY_KEY;
}
__global__ void __launch_bounds__(KTJ_BLOCK)
k_plan_clear(Scalars* sc, Table tf, FullCols fc, Table tn, NarrowCols nc, Table cpu, int force_hash, uint64_t n_rows, uint32_t* h_weave) {
  __shared__ TableCtl ctl[3];
  if (blockIdx.x == 0 && threadIdx.x == 0) stage_clock(sc, KTJ_CLOCK_JOIN);
  if (threadIdx.x < 64) {
    bool beyond_31_bits = false;
    static_assert(KTJ_TBL_FULL == 0 && KTJ_TBL_NARROW == 1, "the full table's range comes first");
    for (int k = 0; k < 3; ++k) {
      unsigned long long lo = sc->range_shard[threadIdx.x][2 * k], hi = sc->range_shard[threadIdx.x][2 * k + 1];
      for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long l2 = __shfl_xor(lo, o), h2 = __shfl_xor(hi, o);
        lo = l2 < lo ? l2 : lo;
        hi = h2 > hi ? h2 : hi;
      }
      const uint64_t cap = (uint64_t)(k == KTJ_TBL_FULL ? tf.mask : k == KTJ_TBL_NARROW ? tn.mask : cpu.mask) + 1u;
      TableCtl x;
      x.base = 0; x.span = 0; x.direct = 0; x.no_heads = 0;
      /* (KTJ_TBL_FULL, whose range has the ids of all runtime and device rows, comes first) */
      if (k == KTJ_TBL_FULL) beyond_31_bits = lo <= hi && hi >= 0x80000000ULL;
      if (k == KTJ_TBL_NARROW) x.no_heads = beyond_31_bits || !nc.head ? 1u : 0u;
      /* the reserved key never takes part in direct addressing (it has its own slot) */
      if (!force_hash && lo <= hi && hi - lo < cap) { x.base = lo; x.span = hi - lo; x.direct = 1; }
      if (threadIdx.x == 0) {
        ctl[k] = x;
        if (blockIdx.x == 0) { sc->plan.range[k].lo = lo; sc->plan.range[k].hi = hi; sc->plan.ctl[k] = x; }
      }
    }
    if (blockIdx.x == 0 && n_rows != 0) {
      uint32_t n = (uint32_t)sc->shard[threadIdx.x][KTJ_CNT_NOT_TEXT];
      for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
      if (threadIdx.x == 0) {
        const bool none = too_many_left(n, n_rows);
        sc->no_text = none ? 1u : 0u;
        __hip_atomic_store(h_weave, (uint32_t)(none ? KTJ_WEAVE_NONE : n ? KTJ_WEAVE_MOST : KTJ_WEAVE_ALL), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
  __syncthreads();
  const uint64_t at = (uint64_t)blockIdx.x * KTJ_BLOCK + threadIdx.x, step = (uint64_t)gridDim.x * KTJ_BLOCK;
  auto span = [&](int k, const Table& t) { TableSpan s; s.direct = ctl[k].direct != 0; s.n = s.direct ? ctl[k].span + 1ull : (uint64_t)t.runs * 16u; return s; };
  const TableSpan sf = span(KTJ_TBL_FULL, tf), sn = span(KTJ_TBL_NARROW, tn), scpu = span(KTJ_TBL_CPU, cpu);
  clear_keys(tf, sf, at, step);
  clear_keys(tn, sn, at, step);
  clear_keys(cpu, scpu, at, step);
  /* full table: the payload is not cleared: every runtime row writes all of its slot's payload, and a slot
   * without a runtime row (its bit in has_runtime is clear) is never read */
  for (uint64_t i = at; i <= sf.n; i += step) {
    const uint64_t k = i < sf.n ? i : tf.mask + 1ull; /* the last one is the reserved slot */
    fc.first[k] = 0xFFFFFFFFu; fc.stream_src[k] = 0;
  }
  const uint64_t words = (sf.n + 31) / 32; /* the bitmap: whole words up to the extent, and the word of the reserved slot */
  for (uint64_t i = at; i <= words; i += step) fc.has_runtime[i < words ? i : (tf.mask + 1ull) / 32] = 0;
  const bool no_heads = ctl[KTJ_TBL_NARROW].no_heads != 0;
  NarrowPay z;
  z.ext_val = 0; z.info = 0; z.pay[0] = z.pay[1] = z.pay[2] = 0;
  for (uint64_t i = at; i <= sn.n; i += step) {
    const uint64_t k = i < sn.n ? i : tn.mask + 1ull;
    nc.ext_src[k] = 0; nc.kern_src[k] = 0; nc.copy_src[k] = 0;
    if (no_heads) nc.pay[k] = z; else nc.head[k] = NarrowHead{0, 0};
  }
}
hipError_t plan_tables(Table tf, FullCols fc, Table tn, NarrowCols nc, Table cpu, bool force_hash, uint64_t n_rows, uint32_t* h_weave, Scalars* sc, hipStream_t st) {
  uint64_t most = (uint64_t)tf.mask + 1;
  if ((uint64_t)tn.mask + 1 > most) most = (uint64_t)tn.mask + 1;
  if ((uint64_t)cpu.mask + 1 > most) most = (uint64_t)cpu.mask + 1;
  const unsigned g = grid_stride_for(most, KTJ_BLOCK * 4);
  hipLaunchKernelGGL(k_plan_clear, dim3(g < 2048u ? g : 2048u), dim3(KTJ_BLOCK), 0, st, sc, tf, fc, tn, nc, cpu, force_hash ? 1 : 0, n_rows, h_weave);
  return KTJ_LAUNCH_CHECK();
}

/* What linkedActivity() (GenericActivityProfiler.cpp:397-408) finds for an external id: the slot's
 * "External id" value and link flags, or zeros when no CPU op has the id. */
__device__ __forceinline__ void resolved_external(uint64_t ext_id, const Table& cpu, const uint32_t* cpu_row, const ktj_generic_rec* g,
                                                  const EmitCtx& ctx, int32_t* ext_val, uint32_t* info) {
  *ext_val = 0;
  *info = 0;
  const uint32_t cs = slot_find(cpu, ext_id);
  if (cs == KTJ_NOSLOT) return;
  *ext_val = (int32_t)(int64_t)ext_id;
  *info = KTJ_NP_LINKED;
  if (cpu_row) { /* the linked op is the last record with that id (activityMap_, GenericActivityProfiler.cpp:262) */
    const uint32_t row = cpu_row[cs];
    if (row) *info |= collective_for_linked(g[row - 1], ctx) << KTJ_NP_COLL_SHIFT;
  }
}
__device__ __forceinline__ void leave_external(const TableView& tn, const NarrowCols& nc, uint32_t slot, int32_t ext_val, uint32_t info) {
  if (tn.no_heads) { nc.pay[slot].ext_val = ext_val; nc.pay[slot].info = info; }
  else nc.head[slot] = NarrowHead{ext_val, info};
}
/* cpuCorrelationMap_[correlation] = externalId: RocmActivityProfiler.cpp:135-148.  The last record of
 * a correlation id stays (atomicMax over the record index).  Every record resolves its external id
 * against the CPU-op ids at once and writes the result into the slot: that is final when no two
 * records share a correlation id, which the returning atomicMax tells; only otherwise
 * k_resolve_external lets the winners write again.  The CPU-op ids are in their table already, the
 * table was cleared, and the runtime rows come later. */
__global__ void k_build_extcorr(const ktj_extcorr_rec* e, uint64_t n, Table tn_planned, NarrowCols nc, Table cpu, const uint32_t* cpu_row,
                                const ktj_generic_rec* g, EmitCtx ctx, Scalars* sc) {
  const TableView tn = view(tn_planned);
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool repeats = false;
  if (i < n) {
    ktj_extcorr_rec rec;
    rec.correlation = load_once(&e[i].correlation);
    rec.external_id = load_once(&e[i].external_id);
    const uint32_t slot = slot_insert(tn, rec.correlation);
    if (slot == KTJ_NOSLOT) flag_error(sc, KTJ_DEVERR_TABLE_FULL);
    else {
      repeats = atomicMax(&nc.ext_src[slot], (uint32_t)i + 1u) != 0u;
      int32_t ext_val;
      uint32_t info;
      resolved_external(rec.external_id, cpu, cpu_row, g, ctx, &ext_val, &info);
      if (info != 0) leave_external(tn, nc, slot, ext_val, info);
    }
  }
  /* one store per workgroup at most: every lane storing the same flag would queue up in L2 */
  if (__syncthreads_or(repeats ? 1 : 0) && threadIdx.x == 0) sc->ext_ids_repeat = 1;
}
/* activityMap_[act->correlationId()] = act: GenericActivityProfiler.cpp:262 */
/* cpu_row (optional): per slot, 1 + index of the last record with that id, for the traces whose
 * CPU ops hand collective metadata to the kernels linked to them */
__global__ void k_build_cpu_ids(const ktj_generic_rec* g, uint64_t n, Table cpu_planned, uint32_t* cpu_row, Scalars* sc) {
  const TableView cpu = view(cpu_planned);
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t slot = slot_insert(cpu, (uint64_t)(int64_t)load_once(&g[i].id));
  if (slot == KTJ_NOSLOT) { flag_error(sc, KTJ_DEVERR_TABLE_FULL); return; }
  if (cpu_row) atomicMax(&cpu_row[slot], (uint32_t)i + 1u);
}
/* Only when external-correlation records share a correlation id: the record that won the slot
 * writes what it resolved again, zeros included, over whatever the other records of the id left. */
__global__ void k_resolve_external(const ktj_extcorr_rec* e, uint64_t n, Table tn, NarrowCols nc, Table cpu,
                                   const uint32_t* cpu_row, const ktj_generic_rec* g, EmitCtx ctx, const Scalars* sc) {
  if (sc->ext_ids_repeat == 0) return;
  const TableView table = view(tn);
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const ktj_extcorr_rec rec = e[i];
    const uint32_t slot = slot_find(table, rec.correlation);
    if (slot == KTJ_NOSLOT || nc.ext_src[slot] != (uint32_t)i + 1u) continue;
    int32_t ext_val;
    uint32_t info;
    resolved_external(rec.external_id, cpu, cpu_row, g, ctx, &ext_val, &info);
    leave_external(table, nc, slot, ext_val, info);
  }
}
/* One pass over the device rows with one slot of each table:
 *  - "External id" (output_json.cpp:871-874) from the narrow slot,
 *  - checkTimestampOrder (GenericActivityProfiler.cpp:363-395) against the first row of the id,
 *  - the stream of the correlation-matched runtime row (RocmStreamQueue.h:56-75, first pass),
 *  - the size or grid/block the launching row hands over (RocprofActivity_inl.h:161-180).
 * The first row of an id is its first runtime row wherever one exists (runtime rows arrive before
 * device rows), which a bitmap tells, and the slot's payload holds that row's timestamp, so the
 * array of first rows is only touched for ids that no runtime row has: in-window device rows take part in "first seen" there and are
 * checked afterwards by k_after_link.  Rows outside the window still take a stream from the
 * slot (slots with a stream come from runtime rows and exist already). */
__global__ void k_link_device(uint64_t n, Columns c, uint64_t first_device, Table tf_planned, FullCols fc, Table tn_planned, NarrowCols nc,
                              Links link, unsigned long long* orphans, Scalars* sc) {
  const TableView tf = view(tf_planned), tn = view(tn_planned);
  uint32_t n_linked = 0, n_bad = 0, n_unresolved = 0, n_orphans = 0;
  const bool have_stream_src = sc->have_stream_src != 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t a = first_device + i;
    /* all reads first (the row's columns, then one slot of each table), all writes after them:
     * the round trips overlap instead of queueing behind each other */
    const uint64_t id = load_once(&c.corr[a]);
    const uint32_t meta = load_once(&c.meta[a]);
    int64_t res = load_once(&c.res[a]);
    const int64_t t2 = load_once(&c.ts[a]);
    const uint32_t domain = (meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT;
    const bool valid = (meta & KTJ_M_VALID) != 0;
    const uint32_t sn = slot_find(tn, narrow_corr_key(id));
    const uint32_t sf = valid ? slot_insert(tf, id) : slot_find(tf, id);
    NarrowPay np;
    np.ext_val = 0; np.info = 0; np.pay[0] = np.pay[1] = np.pay[2] = 0;
    FullPay fp;
    fp.first_ts = 0; fp.stream = 0;
    uint32_t runtime_bits = 0;
    if (sn != KTJ_NOSLOT) np = nc.pay[sn];
    if (sf != KTJ_NOSLOT) {
      fp = fc.pay[sf];
      runtime_bits = fc.has_runtime[sf >> 5];
      if (!((runtime_bits >> (sf & 31u)) & 1u)) { fp.first_ts = 0; fp.stream = 0; } /* no runtime row wrote this slot in this pass */
    }
    if (sn != KTJ_NOSLOT && !tn.no_heads && !((runtime_bits >> (sf & 31u)) & 1u)) { /* nor that one */
      const NarrowHead head = nc.head[sn];
      np.ext_val = head.ext_val; np.info = head.info; np.pay[0] = np.pay[1] = np.pay[2] = 0;
    }
    uint32_t info = 0; /* for the joined row */
    if (sn != KTJ_NOSLOT) {
      if ((np.info & KTJ_NP_LINKED) && valid) ++n_linked;
      info = np.info & ~(KTJ_NP_LINKED | (domain != KTJ_DOM_MEMSET ? 0u : KTJ_NP_KIND_MASK));
    }
    bool orphan = false;
    store_once(&c.ext[a], np.ext_val);
    if (valid && sf == KTJ_NOSLOT) flag_error(sc, KTJ_DEVERR_TABLE_FULL);
    if (sf != KTJ_NOSLOT) {
      if (valid) {
        if ((runtime_bits >> (sf & 31u)) & 1u) { /* act1 = the first runtime row, act2 = this row */
          const int64_t t1 = fp.first_ts;
          if (t2 != 0 && t1 > t2) ++n_bad;
        } else {
          if (fc.first[sf] > (uint32_t)a) atomicMin(&fc.first[sf], (uint32_t)a);
          orphan = true;
          ++n_orphans;
        }
      }
      if (have_stream_src && is_async_op(domain) && res == 0 && fp.stream != 0) { res = (int64_t)fp.stream; c.res[a] = res; }
    }
    /* (whole lines or none: what a row does not have is not read) */
    store_once(&link.info[i], info);
    if (__any((info & KTJ_NP_KIND_MASK) != 0)) store_once(&link.p[0][i], np.pay[0]);
    if (__any((info & KTJ_DL_HAS_GRID) != 0)) { store_once(&link.p[1][i], np.pay[1]); store_once(&link.p[2][i], np.pay[2]); }
    if (is_async_op(domain) && res == 0) ++n_unresolved;
    /* a bit per row, for k_after_link: with the flag in the 32-byte link it read 352 MB to find the few of 11 M
     * rows (127 us, now 25); a wavefront's rows are 64 in a row */
    const unsigned long long some = __ballot(orphan);
    if (lane_id() == 0) orphans[i >> 6] = some;
  }
  block_add(sc, KTJ_CNT_LINKED, n_linked);
  block_add(sc, KTJ_CNT_OUT_OF_ORDER, n_bad);
  block_add_to(&sc->n_unresolved, n_unresolved);
  block_add_to(&sc->n_device_orphans, n_orphans);
}
/* What the device rows need once all of them are linked, both only where some row asks for it:
 *  - an in-window row whose id no runtime row has is checked against the first device row of its id
 *    (act1 = this row, act2 = the first one);
 *  - a row without a stream may take its queue's (RocmStreamQueue.h:42-136; the first pass of that, the
 *    stream of the correlation-matched runtime row, is part of k_link_device): which stream every queue
 *    shows, ambiguous when one queue shows two different ones. */
__global__ void k_after_link(uint64_t n, Columns c, uint64_t first_device, Table tf, FullCols fc, const unsigned long long* orphan_rows,
                             const uint64_t* queues, StreamTables t, Scalars* sc) {
  const bool orphans = sc->n_device_orphans != 0, by_queue = sc->have_stream_src != 0 && sc->n_unresolved != 0;
  uint32_t n_bad = 0;
  if (orphans || by_queue)
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
      const uint64_t a = first_device + i;
      if (orphans && (orphan_rows[i >> 6] >> (i & 63u) & 1ULL)) {
        const uint32_t sf = slot_find(tf, c.corr[a]);
        const uint64_t f = sf != KTJ_NOSLOT ? fc.first[sf] : a;
        if (f != a && f != 0xFFFFFFFFull) {
          const int64_t t1 = c.ts[a], t2 = c.ts[f];
          if (t2 != 0 && t1 > t2) ++n_bad;
        }
      }
      if (by_queue) {
        const uint64_t stream = (uint64_t)c.res[a], queue = queues[i];
        if (is_async_op(row_domain(c.meta[a])) && stream != 0 && queue != 0) {
          const uint32_t slot = table_insert_counted(t.q_keys, KTJ_QUEUE_CAP - 1u, queue, &sc->n_queues, KTJ_MAX_QUEUES);
          if (slot == KTJ_NOSLOT) flag_error(sc, KTJ_DEVERR_QUEUES);
          else {
            unsigned long long cur = t.q_stream[slot];
            if (cur == 0) cur = atomicCAS((unsigned long long*)&t.q_stream[slot], 0ULL, (unsigned long long)stream);
            if (cur != 0 && cur != stream) t.q_amb[slot] = 1u;
          }
        }
      }
    }
  block_add(sc, KTJ_CNT_OUT_OF_ORDER, n_bad);
}

/* Launches that find nothing to do in most passes: every workgroup looks that up, and 4096 of them take 4.6 us for it, 1024 three (where there
 * is something to do they take as long: ids that pairs of a million launches share, join 520 -> 410 us, rows without a launch 344 and 345). */
static unsigned grid_rarely(uint64_t n) { const unsigned g = grid_stride_for(n, KTJ_BLOCK); return g < 1024u ? g : 1024u; }
hipError_t build_cpu_ids(const ktj_generic_rec* g, uint64_t n, Table cpu, uint32_t* cpu_row, Scalars* sc, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_build_cpu_ids, dim3(grid_for(n, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, g, n, cpu, cpu_row, sc);
  return KTJ_LAUNCH_CHECK();
}
/* after build_cpu_ids: the external ids are resolved against that table as the records pass */
hipError_t build_extcorr(const ktj_extcorr_rec* e, uint64_t n, Table tn, NarrowCols nc, Table cpu, const uint32_t* cpu_row,
                         const ktj_generic_rec* g, EmitCtx ctx, Scalars* sc, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_build_extcorr, dim3(grid_for(n, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, e, n, tn, nc, cpu, cpu_row, g, ctx, sc);
  hipLaunchKernelGGL(k_resolve_external, dim3(grid_rarely(n)), dim3(KTJ_BLOCK), 0, st, e, n, tn, nc, cpu, cpu_row, g,
                     ctx, (const Scalars*)sc);
  return KTJ_LAUNCH_CHECK();
}
hipError_t link_device_rows(uint64_t n, Columns c, uint64_t first_device, Table tf, FullCols fc, Table tn, NarrowCols nc,
                            Links link, unsigned long long* orphans, Scalars* sc, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_link_device, dim3(grid_stride_for(n, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, n, c, first_device, tf, fc, tn,
                     nc, link, orphans, sc);
  return KTJ_LAUNCH_CHECK();
}

/* ---- GPU user annotations: GenericActivityProfiler.cpp:277-327, 423-433 ---- */
/* userCorrelationMap_[correlation] = externalId, the last record of an id stays */
__global__ void k_build_usercorr(const ktj_extcorr_rec* u, uint64_t n, SpanTables t, Scalars* sc) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t slot = table_insert(t.u_keys, t.u_mask, u[i].correlation);
  if (slot == KTJ_NOSLOT) { flag_error(sc, KTJ_DEVERR_TABLE_FULL); return; }
  atomicMax(&t.u_src[slot], (uint32_t)i + 1u);
}
__device__ __forceinline__ uint64_t span_hash(int64_t device, int64_t resource, uint64_t ext) {
  uint64_t h = hash64(ext ^ hash64((uint64_t)resource + 0x9E3779B97F4A7C15ULL) ^ hash64((uint64_t)device * 0xC2B2AE3D27D4EB4FULL + 1ULL));
  return h == KTJ_EMPTY_KEY ? 0x5bd1e995ULL : h;
}
/* the annotation a device row belongs to: its id and the slot of that id in the CPU-op table */
__device__ __forceinline__ bool span_of_row(const ktj_extcorr_rec* u, const SpanTables& t, const Table& cpu, uint64_t corr,
                                            uint64_t* ext, uint32_t* cpu_slot) {
  const uint32_t us = table_find(t.u_keys, t.u_mask, corr);
  if (us == KTJ_NOSLOT || t.u_src[us] == 0) return false;
  *ext = u[t.u_src[us] - 1u].external_id;
  *cpu_slot = slot_find(cpu, *ext);
  return *cpu_slot != KTJ_NOSLOT;
}
/* insertOrExtendEvent for every in-window device row: extent of the span, its first row */
__global__ void k_span_extend(const ktj_extcorr_rec* u, uint64_t n, Columns c, uint64_t first_device, Table cpu, SpanTables t,
                              Scalars* sc) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t a = first_device + i;
  if (!(c.meta[a] & KTJ_M_VALID)) return;
  uint64_t ext; uint32_t cs;
  if (!span_of_row(u, t, cpu, c.corr[a], &ext, &cs)) return;
  const uint32_t slot = table_insert(t.hash, t.mask, span_hash(c.dev[a], c.res[a], ext));
  if (slot == KTJ_NOSLOT) { flag_error(sc, KTJ_DEVERR_TABLE_FULL); return; }
  const int64_t ts = c.ts[a];
  atomicMin(&t.first[slot], (uint32_t)i);
  atomicMin((unsigned long long*)&t.lo[slot], (unsigned long long)((uint64_t)ts ^ 0x8000000000000000ULL));
  atomicMax((unsigned long long*)&t.hi[slot], (unsigned long long)((uint64_t)(ts + c.dur[a]) ^ 0x8000000000000000ULL));
  if (ts == 0) t.zero[slot] = 1u;
}
/* createUserGpuSpan: the first row of a span names it (single writer per slot) */
__global__ void k_span_owner(const ktj_extcorr_rec* u, const ktj_generic_rec* g, uint64_t n, Columns c, uint64_t first_device,
                             Table cpu, const uint32_t* cpu_row, SpanTables t) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t a = first_device + i;
  if (!(c.meta[a] & KTJ_M_VALID)) return;
  uint64_t ext; uint32_t cs;
  if (!span_of_row(u, t, cpu, c.corr[a], &ext, &cs)) return;
  const uint32_t slot = table_find(t.hash, t.mask, span_hash(c.dev[a], c.res[a], ext));
  if (slot == KTJ_NOSLOT || t.first[slot] != (uint32_t)i) return;
  t.dev[slot] = (int32_t)c.dev[a]; t.res[slot] = c.res[a]; t.ext[slot] = ext;
  const uint32_t row = cpu_row[cs]; /* the annotation is the last record with that id */
  t.name[slot] = row ? g[row - 1u].name_id : KTJ_NONE;
}
__global__ void k_span_compact(SpanTables t, SpanOut* out, uint32_t* n_out) {
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s > (uint64_t)t.mask + 1u || t.hash[s] == KTJ_EMPTY_KEY || t.first[s] == 0xFFFFFFFFu) return;
  SpanOut o;
  o.res = t.res[s]; o.ext = t.ext[s];
  o.start = (int64_t)(t.lo[s] ^ 0x8000000000000000ULL); o.end = (int64_t)(t.hi[s] ^ 0x8000000000000000ULL);
  o.dev = t.dev[s]; o.name = t.name[s]; o.first = t.first[s]; o.zero = t.zero[s] ? (uint32_t)s + 1u : 0u;
  out[atomicAdd(n_out, 1u)] = o;
}
/* rows of the spans whose start needs the sequential rule (a row at time 0), for the host */
__global__ void k_span_members(const ktj_extcorr_rec* u, uint64_t n, Columns c, uint64_t first_device, Table cpu,
                               SpanTables t, SpanMember* out, uint32_t cap_out, uint32_t* n_out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t a = first_device + i;
  if (!(c.meta[a] & KTJ_M_VALID)) return;
  uint64_t ext; uint32_t cs;
  if (!span_of_row(u, t, cpu, c.corr[a], &ext, &cs)) return;
  const uint32_t slot = table_find(t.hash, t.mask, span_hash(c.dev[a], c.res[a], ext));
  if (slot == KTJ_NOSLOT || t.zero[slot] == 0) return;
  const uint32_t k = atomicAdd(n_out, 1u);
  if (k < cap_out) { SpanMember m; m.slot = slot + 1u; m.row = (uint32_t)i; m.ts = c.ts[a]; out[k] = m; }
}
hipError_t build_usercorr(const ktj_extcorr_rec* u, uint64_t n, SpanTables t, Scalars* sc, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_build_usercorr, dim3(grid_for(n, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, u, n, t, sc);
  return KTJ_LAUNCH_CHECK();
}
hipError_t group_spans(const ktj_extcorr_rec* u, const ktj_generic_rec* g, uint64_t n_device, Columns c, uint64_t first_device,
                       Table cpu, const uint32_t* cpu_row, SpanTables t, SpanOut* out, uint32_t* n_out, Scalars* sc,
                       hipStream_t st) {
  hipError_t e = fill_u32(n_out, 0, 1, st);
  if (e != hipSuccess || n_device == 0) return e;
  const dim3 grid(grid_for(n_device, KTJ_BLOCK)), block(KTJ_BLOCK);
  hipLaunchKernelGGL(k_span_extend, grid, block, 0, st, u, n_device, c, first_device, cpu, t, sc);
  hipLaunchKernelGGL(k_span_owner, grid, block, 0, st, u, g, n_device, c, first_device, cpu, cpu_row, t);
  hipLaunchKernelGGL(k_span_compact, dim3(grid_for((uint64_t)t.mask + 2u, KTJ_BLOCK)), block, 0, st, t, out, n_out);
  return KTJ_LAUNCH_CHECK();
}
hipError_t span_members(const ktj_extcorr_rec* u, uint64_t n_device, Columns c, uint64_t first_device, Table cpu,
                        SpanTables t, SpanMember* out, uint32_t cap_out, uint32_t* n_out, hipStream_t st) {
  hipError_t e = fill_u32(n_out, 0, 1, st);
  if (e != hipSuccess || n_device == 0) return e;
  hipLaunchKernelGGL(k_span_members, dim3(grid_for(n_device, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, u, n_device, c, first_device,
                     cpu, t, out, cap_out, n_out);
  return KTJ_LAUNCH_CHECK();
}

/* This wavefront's stores and atomics have been carried out.  A barrier of the workgroup does not say that, and a
 * fence waits for those of the wavefront it is in only: where one thread speaks for the workgroup afterwards, every
 * wavefront has to come by here before the barrier. */
__device__ __forceinline__ void wave_stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
/* Every workgroup of a launch reports here when its results are in memory; true in all threads of the one
 * that reports last.  What that one reads of the others must have been written with atomics or agent_store()
 * and be read with agent_load(): these pass the caches of one XCD by.  (A fence for ordinary stores writes
 * the XCD's L2 back each time: with one per wavefront k_collect_distinct took 75 instead of 30 us on 733 000
 * rows.)  Must be reached by every thread of the workgroup. */
template <typename T> __device__ __forceinline__ void agent_store(T* p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T> __device__ __forceinline__ T agent_load(const T* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ bool last_workgroup(unsigned int* done) {
  __shared__ int last;
  wave_stores_done();
  __syncthreads();
  if (threadIdx.x == 0) last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1u ? 1 : 0;
  __syncthreads();
  return last != 0;
}
/* table_insert that also tells whether the key is new */
__device__ uint32_t table_insert_fresh(uint64_t* keys, uint32_t mask, uint64_t key, bool* fresh) {
  *fresh = false;
  if (key == KTJ_EMPTY_KEY) {
    *fresh = atomicExch((unsigned long long*)&keys[mask + 1u], 0ULL) != 0ULL;
    return mask + 1u;
  }
  uint32_t slot = (uint32_t)hash64(key) & mask;
  for (uint32_t probe = 0; probe <= mask && probe < KTJ_TABLE_PROBES; ++probe) {
    uint64_t cur = keys[slot];
    if (cur == key) return slot;
    if (cur == KTJ_EMPTY_KEY) {
      const unsigned long long prev = atomicCAS((unsigned long long*)&keys[slot], (unsigned long long)KTJ_EMPTY_KEY, (unsigned long long)key);
      if (prev == KTJ_EMPTY_KEY) { *fresh = true; return slot; }
      if (prev == key) return slot;
    }
    slot = (slot + 1u) & mask;
  }
  return KTJ_NOSLOT;
}

/* ---- stream back-fill: libkineto/src/RocmStreamQueue.h:42-136 ---- */
__device__ __forceinline__ uint64_t dense_hash(int32_t device, uint64_t key) {
  uint64_t h = hash64(key ^ hash64((uint64_t)(int64_t)device + 0x9E3779B97F4A7C15ULL));
  return h == KTJ_EMPTY_KEY ? 0x5bd1e995ULL : h;
}
/* Rows still without a stream take their queue's; then the first arrival index per (device, stream key).
 * Millions of rows share a few hundred pairs, so each workgroup first reduces its rows in an LDS table
 * and touches the global table once per pair.  The workgroup that ends last gives every pair its number:
 * 1 + number of pairs of the same device seen earlier. */
#define DENSE_LOCAL_SLOTS 1024u
/* (every workgroup enters each pair that it has: a million device rows 32 us with 489 workgroups of 256 threads, 21 with 245 of 1024; ten million 58 and 55
 * with 1002 and 251) */
#define DENSE_THREADS 1024u
#define DENSE_ROWS 4u
#define KTJ_DENSE_MAX KTJ_MAX_STREAM_PAIRS
__device__ __forceinline__ void dense_enter(StreamTables& t, uint64_t h, uint32_t first, int32_t dev, uint64_t key, Scalars* sc) {
  bool fresh;
  const uint32_t g = table_insert_fresh(t.d_hash, KTJ_DENSE_CAP - 1u, h, &fresh);
  if (g == KTJ_NOSLOT) { flag_error(sc, KTJ_DEVERR_STREAMS); return; }
  if (t.d_first[g] > first) atomicMin(&t.d_first[g], first); /* (an old value that is still in a cache is larger) */
  if (fresh) { /* two pairs with one hash are told apart when the rows read the table back */
    agent_store(&t.d_dev[g], dev);
    t.d_key[g] = key;
    const uint32_t k = atomicAdd(&sc->n_dense, 1u);
    if (k < KTJ_DENSE_MAX) agent_store(&t.d_list[k], g); else flag_error(sc, KTJ_DEVERR_STREAMS);
  }
}
__global__ void __launch_bounds__(DENSE_THREADS)
k_dense_first(const uint64_t* queues, uint64_t n, uint64_t per, Columns c, uint64_t first_device, StreamTables t, Scalars* sc) {
  __shared__ unsigned long long l_key[DENSE_LOCAL_SLOTS];
  __shared__ unsigned long long l_pair_key[DENSE_LOCAL_SLOTS];
  __shared__ int32_t l_pair_dev[DENSE_LOCAL_SLOTS];
  __shared__ uint32_t l_min[DENSE_LOCAL_SLOTS];
  if (sc->have_stream_src == 0) return;
  const bool fill = sc->n_unresolved != 0;
  for (uint32_t k = threadIdx.x; k < DENSE_LOCAL_SLOTS; k += blockDim.x) { l_key[k] = KTJ_EMPTY_KEY; l_min[k] = 0xFFFFFFFFu; }
  __syncthreads();
  const uint64_t lo = blockIdx.x * per, hi = n < lo + per ? n : lo + per;
  for (uint64_t i0 = lo + threadIdx.x; i0 < hi; i0 += DENSE_THREADS * DENSE_ROWS) {
    uint32_t row_meta[DENSE_ROWS];
    int64_t row_dev[DENSE_ROWS];
    uint64_t row_stream[DENSE_ROWS], row_queue[DENSE_ROWS];
#pragma unroll
    for (uint32_t r = 0; r < DENSE_ROWS; ++r) { /* all loads of the group in flight together */
      const uint64_t i = i0 + r * DENSE_THREADS, a = first_device + (i < hi ? i : hi - 1);
      row_meta[r] = c.meta[a]; row_dev[r] = c.dev[a]; row_stream[r] = (uint64_t)c.res[a];
    }
#pragma unroll
    for (uint32_t r = 0; r < DENSE_ROWS; ++r) {
      const uint64_t i = i0 + r * DENSE_THREADS;
      row_queue[r] = i < hi && row_stream[r] == 0 ? queues[i] : 0;
    }
#pragma unroll
    for (uint32_t r = 0; r < DENSE_ROWS; ++r) {
      const uint64_t i = i0 + r * DENSE_THREADS;
      if (i >= hi) break;
      uint64_t key, stream = row_stream[r];
      const uint32_t domain = row_domain(row_meta[r]);
      const int32_t device = (int32_t)row_dev[r];
      if (fill && stream == 0 && is_async_op(domain)) {
        const uint32_t slot = table_find(t.q_keys, KTJ_QUEUE_CAP - 1u, row_queue[r]);
        if (slot != KTJ_NOSLOT && t.q_amb[slot] == 0 && t.q_stream[slot] != 0) { stream = t.q_stream[slot]; c.res[first_device + i] = (int64_t)stream; }
      }
      if (!dense_key(domain, stream, row_queue[r], &key)) continue;
      const uint64_t h = dense_hash(device, key);
      uint32_t slot = (uint32_t)(h >> 20) & (DENSE_LOCAL_SLOTS - 1u);
      bool placed = false;
      for (uint32_t probe = 0; probe < 16 && !placed; ++probe) {
        unsigned long long cur = l_key[slot];
        if (cur == KTJ_EMPTY_KEY) {
          cur = atomicCAS(&l_key[slot], (unsigned long long)KTJ_EMPTY_KEY, (unsigned long long)h);
          /* the pair itself, for the table entry: every row of the pair would write the same two values */
          if (cur == KTJ_EMPTY_KEY) { l_pair_dev[slot] = device; l_pair_key[slot] = key; }
        }
        if (cur == KTJ_EMPTY_KEY || cur == h) { if (l_min[slot] > (uint32_t)i) atomicMin(&l_min[slot], (uint32_t)i); placed = true; }
        else slot = (slot + 1u) & (DENSE_LOCAL_SLOTS - 1u);
      }
      if (!placed) dense_enter(t, h, (uint32_t)i, device, key, sc); /* local table crowded: straight to the global one */
    }
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < DENSE_LOCAL_SLOTS; k += blockDim.x)
    if (l_key[k] != KTJ_EMPTY_KEY) dense_enter(t, l_key[k], l_min[k], l_pair_dev[k], l_pair_key[k], sc);
  if (!last_workgroup(&sc->done[KTJ_DONE_DENSE])) return;
  const uint32_t n_pairs = agent_load(&sc->n_dense), m = n_pairs < KTJ_DENSE_MAX ? n_pairs : KTJ_DENSE_MAX;
  unsigned long long* l_pair = l_key; /* device and first row of a chunk of the pairs */
  for (uint32_t p0 = 0; p0 < m; p0 += DENSE_THREADS) { /* every thread one pair of this round, against all of them */
    const uint32_t p = p0 + threadIdx.x;
    const uint32_t s = p < m ? agent_load(&t.d_list[p]) : 0u;
    const uint32_t dev = p < m ? (uint32_t)agent_load(&t.d_dev[s]) : 0u, first = p < m ? agent_load(&t.d_first[s]) : 0u;
    uint32_t rank = 1;
    for (uint32_t q0 = 0; q0 < m; q0 += DENSE_LOCAL_SLOTS) {
      const uint32_t here = m - q0 < DENSE_LOCAL_SLOTS ? m - q0 : DENSE_LOCAL_SLOTS;
      __syncthreads();
      for (uint32_t q = threadIdx.x; q < here; q += DENSE_THREADS) {
        const uint32_t o = agent_load(&t.d_list[q0 + q]);
        l_pair[q] = ((unsigned long long)(uint32_t)agent_load(&t.d_dev[o]) << 32) | agent_load(&t.d_first[o]);
      }
      __syncthreads();
      for (uint32_t q = 0; q < here; ++q) rank += (uint32_t)(l_pair[q] >> 32) == dev && (uint32_t)l_pair[q] < first ? 1u : 0u;
    }
    if (p < m) t.d_rank[s] = rank;
  }
}
/* pass 3c: resourceId() = stream != 0 ? stream : queue (RocprofActivity.h:100-102).  Part of k_collect_distinct, which reads the same
 * columns, but where the spans of user annotations ask for it before. */
__device__ __forceinline__ uint32_t dense_number(const StreamTables& t, int32_t device, uint64_t key, Scalars* sc) {
  const uint32_t slot = table_find(t.d_hash, KTJ_DENSE_CAP - 1u, dense_hash(device, key));
  if (slot == KTJ_NOSLOT || t.d_dev[slot] != device || t.d_key[slot] != key) { flag_error(sc, KTJ_DEVERR_HASH_COLLISION); return 0; }
  return t.d_rank[slot];
}
__global__ void k_dense_assign(const uint64_t* queues, uint64_t n, Columns c, uint64_t first_device, StreamTables t,
                               Scalars* sc) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t a = first_device + i;
  const uint32_t domain = row_domain(c.meta[a]);
  if (!is_async_op(domain)) return;
  uint64_t stream = (uint64_t)c.res[a], key;
  const uint64_t queue = stream == 0 ? queues[i] : 0;
  if (sc->have_stream_src != 0 && dense_key(domain, stream, queue, &key)) stream = dense_number(t, (int32_t)c.dev[a], key, sc);
  c.res[a] = (int64_t)(stream != 0 ? stream : queue);
}

hipError_t backfill_streams(const uint64_t* queue, uint64_t n, bool assign, Columns c, uint64_t first_device, Table tf, FullCols fc, const unsigned long long* orphans,
                            StreamTables t, Scalars* sc, hipStream_t st) {
  if (n == 0) return hipSuccess;
  const dim3 g(grid_for(n, KTJ_BLOCK)), b(KTJ_BLOCK);
  hipLaunchKernelGGL(k_after_link, dim3(grid_rarely(n)), b, 0, st, n, c, first_device, tf, fc, orphans, queue, t, sc);
  /* Every workgroup pays for its local table and for each pair it has seen: 2048 rows each, and from 524 288 rows on, where that would be more than a
   * workgroup per CU, as many as make 256 of them.  A workgroup's rows lie together, as buffers of a stream mostly do: it sees few of the pairs then
   * (measured with up to 1024 workgroups of 256 threads; rows a grid apart: 22 million records 85 us instead of 65, 3 million 37 instead of 32; 58 and 33 with
   * columns of 20 bytes a row instead of 24). */
  const unsigned few = grid_stride_for(n, DENSE_THREADS * 2), gd = few < 256u ? few : 256u;
  const uint64_t per = ((n + gd - 1) / gd + DENSE_THREADS - 1) / DENSE_THREADS * DENSE_THREADS;
  hipLaunchKernelGGL(k_dense_first, dim3((unsigned)((n + per - 1) / per)), dim3(DENSE_THREADS), 0, st, queue, n, per, c, first_device, t, sc);
  if (assign) hipLaunchKernelGGL(k_dense_assign, g, b, 0, st, queue, n, c, first_device, t, sc);
  return KTJ_LAUNCH_CHECK();
}

/* ------------------------------------------------------------------------------------------ */
/* stage 3: canonical order = stable sort by (deviceId, resourceId, timestamp), signed            */
/* ------------------------------------------------------------------------------------------ */
/* Workgroup-local set in LDS in front of the global set: a value reaches the global table once
 * per workgroup instead of once per row.  (All rows share a handful of device/resource ids, and
 * millions of probes of the same few global slots serialise in L2.)  Returns true when the
 * caller is the first in its workgroup to see the key, or when the local set is full. */
#define LOCAL_SET_SLOTS 1024u
__device__ __forceinline__ bool local_set_first(unsigned long long* lds /* LOCAL_SET_SLOTS + 1 */, uint64_t key) {
  if (key == KTJ_EMPTY_KEY) return lds[LOCAL_SET_SLOTS] != 0 && atomicExch(&lds[LOCAL_SET_SLOTS], 0ULL) != 0;
  const uint32_t h = ((uint32_t)key ^ ((uint32_t)(key >> 32) * 0x9E3779B1u)) * 0x85EBCA6Bu;
  uint32_t slot = h >> 22; /* 10 bits */
  for (uint32_t probe = 0; probe < 16; ++probe) {
    const unsigned long long cur = lds[slot];
    if (cur == key) return false;
    if (cur == KTJ_EMPTY_KEY) {
      const unsigned long long prev = atomicCAS(&lds[slot], (unsigned long long)KTJ_EMPTY_KEY, (unsigned long long)key);
      if (prev == KTJ_EMPTY_KEY) return true;
      if (prev == key) return false;
    }
    slot = (slot + 1u) & (LOCAL_SET_SLOTS - 1u);
  }
  return true;
}
#define COLLECT_ROWS 4
/* (of 256 threads, twice as many enter their values: 733 000 records 3 us longer, 3 million 8, 5 million 9; of 1024: the same, and 30 000
 * records 2 us longer) */
#define COLLECT_THREADS 512u
#define SORTP_BITS 8 /* of a digit of the one-word sort */
__device__ __forceinline__ void set_enter(uint64_t* keys, uint32_t* list, unsigned int* count, uint64_t v, Scalars* sc, unsigned too_many) {
  bool fresh;
  const uint32_t g = table_insert_fresh(keys, KTJ_SET_CAP - 1u, v, &fresh);
  if (g == KTJ_NOSLOT) { flag_error(sc, too_many); return; }
  if (fresh) {
    const uint32_t k = atomicAdd(count, 1u);
    if (k < KTJ_SET_MAX) agent_store(&list[k], g); else flag_error(sc, too_many);
  }
}
/* by one workgroup: rank of each distinct value = number of smaller values (signed) */
__device__ void rank_values(const uint64_t* keys, const uint32_t* list, uint32_t* rank, uint32_t m, int64_t* lds /* LOCAL_SET_SLOTS */) {
  auto value = [&](uint32_t slot) { return slot < KTJ_SET_CAP ? (int64_t)agent_load(&keys[slot]) : (int64_t)-1; };
  for (uint32_t p0 = 0; p0 < m; p0 += COLLECT_THREADS) {
    const uint32_t p = p0 + threadIdx.x;
    const uint32_t s = p < m ? agent_load(&list[p]) : 0u;
    const int64_t v = p < m ? value(s) : 0;
    uint32_t r = 0;
    for (uint32_t q0 = 0; q0 < m; q0 += LOCAL_SET_SLOTS) {
      const uint32_t here = m - q0 < LOCAL_SET_SLOTS ? m - q0 : LOCAL_SET_SLOTS;
      __syncthreads();
      for (uint32_t q = threadIdx.x; q < here; q += COLLECT_THREADS) lds[q] = value(agent_load(&list[q0 + q]));
      __syncthreads();
      for (uint32_t q = 0; q < here; ++q) r += lds[q] < v ? 1u : 0u;
    }
    if (p < m) rank[s] = r;
  }
}
/* The schemas' texts for the weaver, by one workgroup: a lane lays out each schema, sixteen move its descriptors behind the others',
 * a lane writes the characters of each field.  (One lane for all of it, in a launch of its own: 13 us for four schemas, 20 for
 * five.) */
struct SchemaLds {
  uint4 key[KTJ_WEAVE_FIELDS * (KTJ_WEAVE_KEY / 16u)];
  uint32_t text[weave::SCHEMA_TEXT * 4], desc[weave::MAX_SCHEMAS][weave::SCHEMA_DESC];
  ktj_field field[KTJ_WEAVE_FIELDS];
  uint32_t key_len[KTJ_WEAVE_FIELDS], place[KTJ_WEAVE_FIELDS];
  weave::SchemaPlan plan[weave::MAX_SCHEMAS];
  uint32_t size[weave::MAX_SCHEMAS], upto[weave::MAX_SCHEMAS]; /* descriptors | units of text << 16; the sum up to here, or none where it is not taken */
};
__device__ void lay_out_schemas(const EmitCtx& c, weave::SchemaBook* out, SchemaLds* l) {
  const uint32_t n = c.n_schemas < weave::MAX_SCHEMAS ? c.n_schemas : weave::MAX_SCHEMAS, k = threadIdx.x;
  static_assert(KTJ_BLOCK >= KTJ_WEAVE_FIELDS && KTJ_BLOCK == weave::MAX_SCHEMAS * 16u, "a lane per field, sixteen per schema");
  for (uint32_t j = k; j < weave::SCHEMA_TEXT * 4u; j += KTJ_BLOCK) l->text[j] = 0;
  if (k < KTJ_WEAVE_FIELDS) l->place[k] = ~0u;
  /* which schema the lane's field is of, and which fields the lane's schema has */
  uint32_t of = ~0u, of_field = 0, first = 0, n_fields = 0;
  for (uint32_t j = 0, at = 0; j < n; ++j) {
    const ktj_schema_desc d = c.schemas[j];
    if (k >= at && k - at < d.n_fields && k < KTJ_WEAVE_FIELDS) { of = j; of_field = d.first_field + (k - at); }
    if (j == k) { first = at; n_fields = d.n_fields; }
    at = d.n_fields < KTJ_WEAVE_FIELDS - at ? at + d.n_fields : KTJ_WEAVE_FIELDS;
  }
  if (of != ~0u) {
    const ktj_field fd = c.fields[of_field];
    uint32_t len = 0;
    if (fd.key_id != KTJ_NONE && fd.key_id < c.dict.n) {
      const DictEntry e = c.dict.entries[fd.key_id];
      const uint4* src = reinterpret_cast<const uint4*>(c.dict.arg_blob + e.arg_off);
      len = e.arg_len;
      if (len <= KTJ_WEAVE_KEY) for (uint32_t j = 0; j * 16u < len; ++j) l->key[k * (KTJ_WEAVE_KEY / 16u) + j] = src[j];
    }
    l->field[k] = fd;
    l->key_len[k] = len;
  }
  __syncthreads();
  if (k < 64u) {
    weave::SchemaPlan* const plan = &l->plan[k < weave::MAX_SCHEMAS ? k : 0u];
    weave::SchemaSize size{0, 0};
    if (k < weave::MAX_SCHEMAS) plan->what = 0;
    if (k < n && first + n_fields <= KTJ_WEAVE_FIELDS) size = weave::lay_out_schema(l->field + first, l->key_len + first, n_fields, plan, l->desc[k], l->place + first);
    const uint32_t mine = size.desc | (size.units << 16);
    uint32_t upto = mine;
    for (int o = 1; o < (int)weave::MAX_SCHEMAS; o <<= 1) { const uint32_t x = __shfl_up(upto, o); if ((int)k >= o) upto += x; }
    if (k < weave::MAX_SCHEMAS) {
      const uint32_t before = upto - mine;
      const bool taken = plan->what != 0 && (upto & 0xFFFFu) <= weave::SCHEMA_DESC && (upto >> 16) <= weave::SCHEMA_TEXT; /* (otherwise its rows are format_activity's) */
      l->size[k] = mine;
      l->upto[k] = taken ? upto : 0u;
      weave::SchemaPlan p = *plan;
      if (!taken) p.what = 0;
      p.args = KTJ_WREF_MOVED(p.args, before & 0xFFFFu);
      p.args2 = KTJ_WREF_MOVED(p.args2, KTJ_WREF_COUNT(p.args2) ? before & 0xFFFFu : 0u);
      out->plan[k] = p;
    }
  }
  __syncthreads();
  {
    const uint32_t schema = (k >> 4) & (weave::MAX_SCHEMAS - 1u), size = l->size[schema], upto = k < KTJ_BLOCK ? l->upto[schema] : 0u;
    if (upto) {
      const uint32_t before = upto - size;
      for (uint32_t j = k & 15u; j < (size & 0xFFFFu); j += 16u) out->desc[(before & 0xFFFFu) + j] = KTJ_WD_MOVED(l->desc[schema][j], before >> 16);
    }
  }
  if (of != ~0u && l->upto[of] != 0 && l->place[k] != ~0u)
    weave::put_field_text(l->field[k], reinterpret_cast<const char*>(l->key + k * (KTJ_WEAVE_KEY / 16u)), l->key_len[k],
                          KTJ_PLACE_MOVED(l->place[k], (l->upto[of] - l->size[of]) >> 16), reinterpret_cast<char*>(l->text));
  __syncthreads();
  for (uint32_t j = k; j < weave::SCHEMA_TEXT * 4u; j += KTJ_BLOCK) out->text[j] = l->text[j];
}
/* What a workgroup of k_collect_distinct has looked up of the pairs' numbers; a pair whose places are taken is looked up each time.  A
 * number is stored behind the pair it belongs to (PAIR_CLAIMED: not yet). */
#define PAIR_SLOTS 1024u
#define PAIR_CLAIMED 0xFFFFFFFFu
struct PairCache { unsigned long long key[PAIR_SLOTS]; int32_t dev[PAIR_SLOTS]; uint32_t number[PAIR_SLOTS]; };
__device__ __forceinline__ uint32_t pair_number(PairCache& l, const StreamTables& t, int32_t device, uint64_t key, Scalars* sc) {
  const uint32_t h = ((uint32_t)key ^ ((uint32_t)(key >> 32) * 0x9E3779B1u) ^ ((uint32_t)device * 0xC2B2AE35u)) * 0x85EBCA6Bu;
  uint32_t slot = h >> 22, free = PAIR_SLOTS; /* 10 bits */
  for (uint32_t probe = 0; probe < 4u; ++probe) {
    const uint32_t x = __hip_atomic_load(&l.number[slot], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (x == 0) { free = slot; break; }
    if (x != PAIR_CLAIMED && l.key[slot] == key && l.dev[slot] == device) return x;
    slot = (slot + 1u) & (PAIR_SLOTS - 1u);
  }
  const uint32_t number = dense_number(t, device, key, sc);
  if (free != PAIR_SLOTS && number != 0 && atomicCAS(&l.number[free], 0u, PAIR_CLAIMED) == 0u) {
    l.key[free] = key; l.dev[free] = device;
    __hip_atomic_store(&l.number[free], number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  return number;
}
/* Distinct deviceId and resourceId values, the range of the timestamps and the number of rows that are
 * printed.  The workgroup that ends last ranks the values and plans the sort's keys.  With a book the first
 * workgroup lays out the schemas instead of taking rows: this is the longest launch before the size pass that
 * small passes have, too.
 * Device rows take the number of their (device, stream) pair on the way, as their columns are read here anyway: a pass of its own
 * read 24 bytes a row, of them 16 that were made for it only (11 million records 3655 -> 3603 us, 22 million 7850 -> 7806, 30 000
 * 174 -> 171; 3 million 1169 -> 1161). */
__global__ void __launch_bounds__(COLLECT_THREADS) k_collect_distinct(Columns c, uint64_t n, uint64_t per, uint64_t n_device, Backfill fill, SortSets s, Scalars* sc, int straight, EmitCtx ctx, weave::SchemaBook* book) {
  __shared__ uint64_t red_min[COLLECT_THREADS >> 6], red_max[COLLECT_THREADS >> 6];
  __shared__ unsigned long long seen[2][LOCAL_SET_SLOTS + 1]; /* deviceId, resourceId values */
  __shared__ PairCache pairs;
  static_assert(sizeof(SchemaLds) <= sizeof(seen), "laid out where the values would be");
  const uint32_t books = book ? 1u : 0u;
  const bool lays_out = blockIdx.x < books;
  if (blockIdx.x == 0 && threadIdx.x == 0) stage_clock(sc, KTJ_CLOCK_SORT);
  if (lays_out) {
    if (sc->no_text == 0) lay_out_schemas(ctx, book, reinterpret_cast<SchemaLds*>(seen));
  } else for (uint32_t k = threadIdx.x; k <= LOCAL_SET_SLOTS; k += blockDim.x) { seen[0][k] = KTJ_EMPTY_KEY; seen[1][k] = KTJ_EMPTY_KEY; }
  for (uint32_t k = threadIdx.x; k < PAIR_SLOTS; k += blockDim.x) pairs.number[k] = 0;
  __syncthreads();
  uint64_t mn = ~0ULL, mx = 0ULL;
  uint64_t last_dev = 0, last_res = 0; /* of the thread's rows so far: most rows repeat them */
  const bool numbered = sc->have_stream_src != 0;
  uint64_t pair_key = 0; /* the thread's last pair; 0 is no key */
  int32_t pair_dev = 0;
  uint32_t pair_is = 0;
  bool any = false;
  uint32_t n_valid = 0;
  const uint64_t first = lays_out ? n : (blockIdx.x - books) * per, end = n < first + per ? n : first + per;
  for (uint64_t a0 = first + threadIdx.x; a0 < end; a0 += COLLECT_THREADS * COLLECT_ROWS) {
    uint32_t meta[COLLECT_ROWS];
    uint64_t dev[COLLECT_ROWS], res[COLLECT_ROWS], ts[COLLECT_ROWS];
#pragma unroll
    for (int r = 0; r < COLLECT_ROWS; ++r) { /* all loads of the group in flight together */
      const uint64_t at = a0 + (uint64_t)r * COLLECT_THREADS, a = at < end ? at : end - 1;
      meta[r] = c.meta[a];
      dev[r] = (uint64_t)c.dev[a];
      res[r] = (uint64_t)c.res[a];
      ts[r] = (uint64_t)c.ts[a];
    }
#pragma unroll
    for (int r = 0; r < COLLECT_ROWS; ++r) meta[r] = a0 + (uint64_t)r * COLLECT_THREADS < end ? meta[r] : 0u; /* (not a row) */
    uint32_t ask = 0; /* device rows that take their pair's number: the key stands in res meanwhile */
    uint64_t queue[COLLECT_ROWS];
#pragma unroll
    for (int r = 0; r < COLLECT_ROWS; ++r) {
      const uint64_t a = a0 + (uint64_t)r * COLLECT_THREADS, i = a - fill.first_device; /* (wraps around in front of them) */
      const bool device = a < end && a >= fill.first_device && i < fill.n && is_async_op(row_domain(meta[r]));
      ask |= (device ? 1u : 0u) << r;
      queue[r] = device && res[r] == 0 ? fill.queue[i] : 0;
    }
#pragma unroll
    for (int r = 0; r < COLLECT_ROWS; ++r) {
      if (!(ask >> r & 1u)) continue;
      uint64_t key;
      if (numbered && dense_key(row_domain(meta[r]), res[r], queue[r], &key)) res[r] = key;
      else {
        ask &= ~(1u << r);
        if (res[r] == 0 && queue[r] != 0) { res[r] = queue[r]; c.res[a0 + (uint64_t)r * COLLECT_THREADS] = (int64_t)queue[r]; }
      }
    }
    while (ask) {
      const uint32_t at = (uint32_t)__builtin_ctz(ask);
      ask &= ask - 1u;
      uint64_t key = res[0], device = dev[0];
#pragma unroll
      for (uint32_t r = 1; r < COLLECT_ROWS; ++r) { key = at == r ? res[r] : key; device = at == r ? dev[r] : device; }
      if (key != pair_key || (int32_t)device != pair_dev) {
        pair_key = key; pair_dev = (int32_t)device;
        pair_is = pair_number(pairs, fill.t, pair_dev, key, sc);
      }
#pragma unroll
      for (uint32_t r = 0; r < COLLECT_ROWS; ++r) res[r] = at == r ? (uint64_t)pair_is : res[r];
      c.res[a0 + (uint64_t)at * COLLECT_THREADS] = (int64_t)pair_is;
    }
    uint32_t todo = 0;
#pragma unroll
    for (int r = 0; r < COLLECT_ROWS; ++r) {
      if (!(meta[r] & KTJ_M_VALID)) continue;
      todo |= (!any || dev[r] != last_dev ? 1u : 0u) << r | (!any || res[r] != last_res ? 1u : 0u) << (COLLECT_ROWS + r);
      last_dev = dev[r]; last_res = res[r];
      any = true;
      const uint64_t tb = ts[r] ^ 0x8000000000000000ULL;
      mn = tb < mn ? tb : mn;
      mx = tb > mx ? tb : mx;
      ++n_valid;
    }
    while (todo) { /* one copy of the probing for all rows and both sets (unrolled it spilled 358 scalar registers) */
      const uint32_t at = (uint32_t)__builtin_ctz(todo), is_res = at / COLLECT_ROWS;
      todo &= todo - 1u;
      uint64_t v = dev[0];
#pragma unroll
      for (uint32_t r = 1; r < 2 * COLLECT_ROWS; ++r) v = at == r ? (r < COLLECT_ROWS ? dev[r] : res[r - COLLECT_ROWS]) : v;
      if (!local_set_first(seen[is_res], v)) continue;
      set_enter(is_res ? s.res_keys : s.dev_keys, is_res ? s.res_list : s.dev_list, is_res ? &sc->n_res_ranks : &sc->n_dev_ranks, v, sc,
                is_res ? KTJ_DEVERR_DISTINCT_RESOURCES : KTJ_DEVERR_DISTINCT_DEVICES);
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t on = __shfl_xor((unsigned long long)mn, o), ox = __shfl_xor((unsigned long long)mx, o);
    mn = on < mn ? on : mn;
    mx = ox > mx ? ox : mx;
  }
  if (lane_id() == 0) { red_min[threadIdx.x >> 6] = mn; red_max[threadIdx.x >> 6] = mx; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t k = 1; k < (blockDim.x >> 6); ++k) {
      mn = red_min[k] < mn ? red_min[k] : mn;
      mx = red_max[k] > mx ? red_max[k] : mx;
    }
    /* into one of 64 copies, as the other ranges: seven hundred workgroups and more queue up at a single one
     * (733 000 records 39 -> 30 us, 3 M 53 -> 41 us).  (Reading the current range first, to skip the atomics,
     * costs more than they do.) */
    if (mn <= mx) {
      unsigned long long* r = &sc->range_shard[blockIdx.x & (KTJ_COUNTER_SHARDS - 1u)][2 * KTJ_RANGE_TS];
      atomicMin(&r[0], (unsigned long long)mn);
      atomicMax(&r[1], (unsigned long long)mx);
    }
  }
  block_add(sc, KTJ_CNT_VALID, n_valid);
  if (!last_workgroup(&sc->done[KTJ_DONE_COLLECT])) return;
  const uint32_t nd = agent_load(&sc->n_dev_ranks), nr = agent_load(&sc->n_res_ranks);
  const uint32_t md = nd < KTJ_SET_MAX ? nd : KTJ_SET_MAX, mr = nr < KTJ_SET_MAX ? nr : KTJ_SET_MAX;
  rank_values(s.dev_keys, s.dev_list, s.dev_rank, md, reinterpret_cast<int64_t*>(seen[0]));
  rank_values(s.res_keys, s.res_list, s.res_rank, mr, reinterpret_cast<int64_t*>(seen[0]));
  if (threadIdx.x >= 64) return;
  static_assert(KTJ_COUNTER_SHARDS == 64, "a lane per copy");
  uint64_t lo = agent_load(&sc->range_shard[threadIdx.x][2 * KTJ_RANGE_TS]), hi = agent_load(&sc->range_shard[threadIdx.x][2 * KTJ_RANGE_TS + 1]);
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t on = __shfl_xor((unsigned long long)lo, o), ox = __shfl_xor((unsigned long long)hi, o);
    lo = on < lo ? on : lo;
    hi = ox > hi ? ox : hi;
  }
  const uint64_t sync_typed = __ballot(sc->shard[threadIdx.x][KTJ_CNT_SYNC_TYPED] != 0); /* the order decides which of them announces its row */
  unsigned long long valid = agent_load(&sc->shard[threadIdx.x][KTJ_CNT_VALID]);
  for (int o = 32; o > 0; o >>= 1) valid += __shfl_xor(valid, o);
  if (threadIdx.x == 0) {
    sc->ts_min_biased = lo;
    sc->ts_max_biased = hi;
    const uint64_t span = lo <= hi ? hi - lo : 0;
    auto bits = [](uint64_t v) -> uint32_t { return v ? 64u - (uint32_t)__builtin_clzll(v) : 0u; }; /* to hold 0..v */
    SortPlan p;
    p.ts_bits = bits(span);
    p.res_bits = bits(mr ? mr - 1u : 0u);
    p.n_dev = md;
    p.key_bits = p.ts_bits + p.res_bits + bits(valid < n ? md : md ? md - 1u : 0u); /* rows that are dropped: a device behind the others */
    /* The lowest bits that need no pass (k_sortp_finish): in 2^low ns, 65 us at most, a track has thirty-two rows or fewer (sixteen where the
     * trace takes all times of its bits, twice as many where it takes little more than half of them), were they
     * spread evenly over the trace and over the streams and threads; and no more bits than the passes that remain leave over.  (15
     * bits instead of 7 for 22 million, groups of 67 rows: a pass less, 135 us, but 220 us more behind the passes.) */
    const uint32_t pairs = sc->n_dense, threads = mr > pairs ? mr - pairs : 1u;
    const float of_thread = (float)(n - n_device) / (float)threads;
    const float of_stream = (float)n_device / (pairs ? (float)pairs : 0.5f * (float)threads); /* (no pairs: the streams are among the others) */
    const float rows = of_stream > of_thread ? of_stream : of_thread, times = p.ts_bits < 60u ? 16.0f * (float)(1ull << p.ts_bits) : 1e30f;
    uint32_t low = 0;
    while (low < 16u && rows * (float)(2u << low) <= times) ++low;
    const uint32_t passes = (p.key_bits > low ? p.key_bits - low + SORTP_BITS - 1u : SORTP_BITS) / SORTP_BITS;
    p.low_bits = p.key_bits > passes * SORTP_BITS && p.key_bits + bits(n - 1u) <= 64u ? p.key_bits - passes * SORTP_BITS : 0u;
    sc->sort = p;
    if (straight && sync_typed) flag_error(sc, KTJ_DEVERR_CAREFUL);
  }
}
/* Rank of a value through its set.  The rows of a wavefront mostly share one value: then a single
 * lookup with a wavefront-uniform key (which the compiler can keep on the scalar unit) serves all
 * lanes. */
__device__ __forceinline__ uint64_t set_rank(const uint64_t* keys, const uint32_t* rank, uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  const uint64_t first = ((uint64_t)hi << 32) | lo;
  if (__ballot(v != first) == 0) {
    const uint32_t slot = table_find(keys, KTJ_SET_CAP - 1u, first);
    return slot != KTJ_NOSLOT ? rank[slot] : 0;
  }
  const uint32_t slot = table_find(keys, KTJ_SET_CAP - 1u, v);
  return slot != KTJ_NOSLOT ? rank[slot] : 0;
}
/* The same for a thread that looks up one row after the other: rows that follow each other in a
 * record buffer mostly belong to one stream or thread, so the last wavefront-wide value and its rank
 * are kept, and a lookup (two dependent loads at least) is only made when the value changes.  A
 * lane's memo is a (value, rank) pair that it took part in looking up, or nothing. */
struct RankMemo { uint64_t key; uint32_t rank; bool have; };
__device__ __forceinline__ uint64_t set_rank_memo(const uint64_t* keys, const uint32_t* rank, uint64_t v, RankMemo& m) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  const uint64_t first = ((uint64_t)hi << 32) | lo;
  if (__ballot(v != first) == 0) {
    if (m.have && m.key == first) return m.rank;
    const uint32_t slot = table_find(keys, KTJ_SET_CAP - 1u, first);
    m.key = first; m.rank = slot != KTJ_NOSLOT ? rank[slot] : 0; m.have = true;
    return m.rank;
  }
  const uint32_t slot = table_find(keys, KTJ_SET_CAP - 1u, v);
  return slot != KTJ_NOSLOT ? rank[slot] : 0;
}
__global__ void k_make_keys(Columns c, uint64_t n, SortSets s, const Scalars* sc, uint32_t ts_bits, uint32_t res_bits,
                            uint32_t key_bits, uint64_t* keys, uint32_t* vals) {
  const uint64_t a = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= n) return;
  uint64_t key = key_bits >= 64 ? ~0ULL : (1ULL << key_bits); /* dropped rows sort behind everything */
  if (c.meta[a] & KTJ_M_VALID) {
    const uint64_t rd = set_rank(s.dev_keys, s.dev_rank, (uint64_t)c.dev[a]);
    const uint64_t rr = set_rank(s.res_keys, s.res_rank, (uint64_t)c.res[a]);
    const uint64_t rel = ((uint64_t)c.ts[a] ^ 0x8000000000000000ULL) - sc->ts_min_biased;
    uint64_t hi = (rd << res_bits) | rr;
    key = ts_bits >= 64 ? rel : ((hi << ts_bits) | rel);
  }
  keys[a] = key;
  vals[a] = (uint32_t)a;
}

/* Wide timestamp spans (a row at time 0 next to rows at wall-clock time) do not fit one 64-bit
 * composite key.  The order is then built in two stable sorts: by timestamp, then by the
 * (device, resource) ranks of the rows in that order. */
__global__ void k_make_ts_keys(Columns c, uint64_t n, const Scalars* sc, uint64_t* keys, uint32_t* vals) {
  const uint64_t a = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= n) return;
  keys[a] = (c.meta[a] & KTJ_M_VALID) ? (((uint64_t)c.ts[a] ^ 0x8000000000000000ULL) - sc->ts_min_biased) : 0;
  vals[a] = (uint32_t)a;
}
__global__ void k_make_rank_keys(Columns c, const uint32_t* order, uint64_t n, SortSets s, uint32_t res_bits,
                                 uint32_t rank_bits, uint64_t* keys, uint32_t* vals) {
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t a = order[p];
  uint64_t key = 1ULL << rank_bits; /* dropped rows sort behind everything */
  if (c.meta[a] & KTJ_M_VALID) {
    const uint64_t rd = set_rank(s.dev_keys, s.dev_rank, (uint64_t)c.dev[a]);
    const uint64_t rr = set_rank(s.res_keys, s.res_rank, (uint64_t)c.res[a]);
    key = (rd << res_bits) | rr;
  }
  keys[p] = key;
  vals[p] = a;
}
/* Traces with more distinct deviceId or resourceId values than the rank sets hold are ordered by
 * the raw values: one more stable sort per column (sign-biased 64-bit keys), and a last one that
 * moves the dropped rows behind the kept ones. */
__global__ void k_make_column_keys(const int64_t* column, const uint32_t* meta, const uint32_t* order, uint64_t n, int validity,
                                   uint64_t* keys, uint32_t* vals) {
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t a = order[p];
  const bool valid = (meta[a] & KTJ_M_VALID) != 0;
  keys[p] = validity ? (valid ? 0ull : 1ull) : (valid ? ((uint64_t)column[a] ^ 0x8000000000000000ULL) : 0ull);
  vals[p] = a;
}
hipError_t make_column_keys(const int64_t* column, const uint32_t* meta, const uint32_t* order, uint64_t n, int validity,
                            uint64_t* keys, uint32_t* vals, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_make_column_keys, dim3(grid_for(n, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, column, meta, order, n, validity,
                     keys, vals);
  return KTJ_LAUNCH_CHECK();
}
__global__ void k_clear_error_bits(Scalars* sc, unsigned int bits) { sc->error &= ~bits; }
hipError_t clear_error_bits(Scalars* sc, unsigned int bits, hipStream_t st) {
  hipLaunchKernelGGL(k_clear_error_bits, dim3(1), dim3(1), 0, st, sc, bits);
  return KTJ_LAUNCH_CHECK();
}
hipError_t make_ts_keys(Columns c, uint64_t n, const Scalars* sc, uint64_t* keys, uint32_t* vals, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_make_ts_keys, dim3(grid_for(n, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, c, n, sc, keys, vals);
  return KTJ_LAUNCH_CHECK();
}
hipError_t make_rank_keys(Columns c, const uint32_t* order, uint64_t n, SortSets s, uint32_t res_bits, uint32_t rank_bits,
                          uint64_t* keys, uint32_t* vals, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_make_rank_keys, dim3(grid_for(n, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, c, order, n, s, res_bits,
                     rank_bits, keys, vals);
  return KTJ_LAUNCH_CHECK();
}

hipError_t collect_distinct(Columns c, uint64_t n, uint64_t n_device, const Backfill& fill, SortSets s, Scalars* sc, bool straight, const EmitCtx& ctx, weave::SchemaBook* book, hipStream_t st) {
  if (n == 0) return hipSuccess;
  /* Few, fat workgroups: every one pays for its local sets and its atomics at the end once.  Up to a million rows four rows a
   * thread, then sixteen and, from 4.2 million on, more: at most 512 workgroups, two per CU, keep enough loads in flight (of 256 threads, when the numbers of
   * streams were another launch's: 4096 of them 230 us for 22 million rows, 1024 170). */
  unsigned g = grid_stride_for(n, n < (1u << 20) ? COLLECT_THREADS * COLLECT_ROWS : COLLECT_THREADS * 16);
  if (g > 1024u * 256u / COLLECT_THREADS) g = 1024u * 256u / COLLECT_THREADS;
  /* (a workgroup's rows lie together and have few values, as above: 733 000 records 34 -> 28 us, 22 million 151 -> 141; 32 and 168 since
   * device rows take their numbers here, 66 in a launch of its own for 22 million) */
  const uint64_t per = ((n + g - 1) / g + COLLECT_THREADS - 1) / COLLECT_THREADS * COLLECT_THREADS;
  hipLaunchKernelGGL(k_collect_distinct, dim3((unsigned)((n + per - 1) / per) + (book ? 1u : 0u)), dim3(COLLECT_THREADS), 0, st, c, n, per, n_device, fill, s, sc, straight ? 1 : 0, ctx, book);
  return KTJ_LAUNCH_CHECK();
}
hipError_t make_keys(Columns c, uint64_t n, SortSets s, const Scalars* sc, uint32_t ts_bits, uint32_t res_bits,
                     uint32_t key_bits, uint64_t* keys, uint32_t* vals, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_make_keys, dim3(grid_for(n, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, c, n, s, sc, ts_bits,
                     res_bits, key_bits, keys, vals);
  return KTJ_LAUNCH_CHECK();
}

/* ---- stable LSD radix sort, 8 bits per pass ----
 * A workgroup owns a tile of 4096 consecutive keys, one quarter per wavefront.  Ranks within the
 * tile come from wavefront match (ballots) plus per-wavefront running counts; the tile is then
 * laid out in LDS in digit order and written from there, so that neighbouring lanes store
 * neighbouring elements of a digit's run (whole lines instead of single 8-byte stores). */
#define RADIX_ITEMS 16
#define RADIX_TILE (KTJ_BLOCK * RADIX_ITEMS)
#define RADIX_WAVES (KTJ_BLOCK >> 6)
#define RADIX_WAVE_KEYS (64 * RADIX_ITEMS)

__global__ void __launch_bounds__(KTJ_BLOCK)
k_radix_hist(const uint64_t* keys, uint64_t n, uint32_t shift, uint32_t* hist, uint32_t n_blocks) {
  __shared__ uint32_t h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * RADIX_TILE;
  for (int r = 0; r < RADIX_ITEMS; ++r) {
    const uint64_t i = base + (uint64_t)r * KTJ_BLOCK + threadIdx.x;
    if (i < n) atomicAdd(&h[(uint32_t)(keys[i] >> shift) & 0xFFu], 1u);
  }
  __syncthreads();
  hist[(uint64_t)threadIdx.x * n_blocks + blockIdx.x] = h[threadIdx.x]; /* digit-major */
}
__global__ void __launch_bounds__(KTJ_BLOCK)
k_radix_scatter(const uint64_t* keys_in, const uint32_t* vals_in, uint64_t* keys_out, uint32_t* vals_out, uint64_t n,
                uint32_t shift, const uint32_t* hist_scanned, uint32_t n_blocks) {
  __shared__ uint64_t s_key[RADIX_TILE];
  __shared__ uint32_t s_val[RADIX_TILE];
  __shared__ uint32_t wave_run[RADIX_WAVES][256]; /* count per (wavefront, digit), then its start inside the digit's run */
  __shared__ uint32_t digit_start[256];           /* start of the digit's run inside the tile     */
  __shared__ uint32_t base_of[256];               /* global offset of this tile's run per digit   */
  __shared__ uint32_t wave_tot[RADIX_WAVES];
  base_of[threadIdx.x] = hist_scanned[(uint64_t)threadIdx.x * n_blocks + blockIdx.x];
  for (int k = 0; k < RADIX_WAVES; ++k) wave_run[k][threadIdx.x] = 0;
  __syncthreads();
  const uint32_t w = threadIdx.x >> 6, lane = lane_id();
  const uint64_t lt = lanemask_lt();
  const uint64_t tile_base = (uint64_t)blockIdx.x * RADIX_TILE;
  const uint64_t chunk = tile_base + (uint64_t)w * RADIX_WAVE_KEYS;
  /* my_run: this wavefront's running counts; accessed as LDS (a plain pointer to the row would
   * turn into flat accesses), re-read every round because other lanes of the wavefront update it */
  typedef volatile __attribute__((address_space(3))) uint32_t* lds_counts;
  lds_counts my_run = (lds_counts)&wave_run[w][0];
  uint64_t key[RADIX_ITEMS];
  uint32_t val[RADIX_ITEMS], rank[RADIX_ITEMS];
#pragma unroll
  for (int r = 0; r < RADIX_ITEMS; ++r) {
    const uint64_t i = chunk + (uint64_t)r * 64u + lane;
    const bool valid = i < n;
    key[r] = valid ? keys_in[i] : ~0ULL;
    val[r] = valid ? vals_in[i] : 0u;
  }
#pragma unroll
  for (int r = 0; r < RADIX_ITEMS; ++r) {
    const bool valid = chunk + (uint64_t)r * 64u + lane < n;
    const uint32_t digit = (uint32_t)(key[r] >> shift) & 0xFFu;
    /* lanes of this wavefront holding the same digit */
    uint64_t peers = __ballot(valid ? 1 : 0);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint64_t bal = __ballot((digit >> b) & 1u);
      peers &= ((digit >> b) & 1u) ? bal : ~bal;
    }
    const uint32_t rank_in_wave = (uint32_t)__popcll(peers & lt);
    const uint32_t before = my_run[digit];   /* same digit in earlier rounds of this wavefront */
    rank[r] = before + rank_in_wave;
    if (valid && rank_in_wave == 0) my_run[digit] = before + (uint32_t)__popcll(peers);
  }
  __syncthreads();
  {
    /* per digit: wavefront counts -> starts inside the digit's run; digit totals -> exclusive scan */
    uint32_t tot = 0;
    for (int k = 0; k < RADIX_WAVES; ++k) { const uint32_t cnt = wave_run[k][threadIdx.x]; wave_run[k][threadIdx.x] = tot; tot += cnt; }
    uint32_t inc = tot;
    for (int o = 1; o < 64; o <<= 1) { const uint32_t t = __shfl_up(inc, o); if (lane >= (uint32_t)o) inc += t; }
    if (lane == 63) wave_tot[w] = inc;
    __syncthreads();
    uint32_t add = 0;
    for (uint32_t k = 0; k < w; ++k) add += wave_tot[k];
    digit_start[threadIdx.x] = add + inc - tot;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RADIX_ITEMS; ++r) {
    if (chunk + (uint64_t)r * 64u + lane < n) {
      const uint32_t digit = (uint32_t)(key[r] >> shift) & 0xFFu;
      const uint32_t p = digit_start[digit] + wave_run[w][digit] + rank[r];
      s_key[p] = key[r];
      s_val[p] = val[r];
    }
  }
  __syncthreads();
  const uint32_t cnt = (uint32_t)(n - tile_base < RADIX_TILE ? n - tile_base : RADIX_TILE);
  for (uint32_t p = threadIdx.x; p < cnt; p += KTJ_BLOCK) {
    const uint64_t k = s_key[p];
    const uint32_t digit = (uint32_t)(k >> shift) & 0xFFu;
    const uint64_t dst = (uint64_t)base_of[digit] + (p - digit_start[digit]);
    keys_out[dst] = k;
    vals_out[dst] = s_val[p];
  }
}

#define SORTP_STREAM_N (1ull << 24)
/* Keys per thread of the packed sort's tiles, 256 threads to each: as few as leave no CU without a tile, as many as keep the counts, a
 * launch of 256 workgroups per pass to add up, short.  2 / 4 / 8 / 16, passes in us: 240 000 keys 219 / 221 / 228 / 243, 396 000 287 / 286 / 289 / 304,
 * 600 000 321 / 317 / 321 / 332, 733 000 386 / 380 / 383 / 394, 900 000 406 / 398 / 399 / 408, 1.5 million 591 / 564 / 560 / 574, 3 million 1039 / 986 / 965 / 962,
 * 4.4 million 1622 / 1519 / 1470 / 1472. */
static const uint64_t sort_items_end[] = {3ull << 17, 1ull << 20, 1ull << 21};
static uint32_t sort_items(uint64_t n) {
  uint32_t items = 2;
  for (const uint64_t end : sort_items_end) items *= n >= end ? 2u : 1u;
  return items;
}
/* counts per (digit, tile) plus the digits' totals, of up to n keys: fewer may have more tiles */
uint64_t radix_tmp_elems(uint64_t n) {
  uint64_t tiles = (n + RADIX_TILE - 1) / RADIX_TILE;
  for (const uint64_t end : sort_items_end) {
    const uint64_t m = n < end ? n : end - 1u, tile = 256ull * sort_items(m), t = (m + tile - 1) / tile;
    tiles = t > tiles ? t : tiles;
  }
  return 256ull * tiles + 256;
}

hipError_t radix_sort(uint64_t* keys_a, uint32_t* vals_a, uint64_t* keys_b, uint32_t* vals_b, uint64_t n,
                      uint32_t bits, uint32_t* hist, uint64_t* scan_tmp, uint64_t** res_keys, uint32_t** res_vals,
                      hipStream_t st) {
  *res_keys = keys_a;
  *res_vals = vals_a;
  if (n == 0) return hipSuccess;
  const uint32_t n_blocks = (uint32_t)((n + RADIX_TILE - 1) / RADIX_TILE);
  uint64_t* ki = keys_a; uint32_t* vi = vals_a; uint64_t* ko = keys_b; uint32_t* vo = vals_b;
  for (uint32_t shift = 0; shift < bits; shift += 8) {
    hipLaunchKernelGGL(k_radix_hist, dim3(n_blocks), dim3(KTJ_BLOCK), 0, st, (const uint64_t*)ki, n, shift, hist, n_blocks);
    hipError_t e = scan_u32_inplace(hist, 256ull * n_blocks, scan_tmp, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_radix_scatter, dim3(n_blocks), dim3(KTJ_BLOCK), 0, st, (const uint64_t*)ki, (const uint32_t*)vi,
                       ko, vo, n, shift, (const uint32_t*)hist, n_blocks);
    uint64_t* tk = ki; ki = ko; ko = tk;
    uint32_t* tv = vi; vi = vo; vo = tv;
  }
  *res_keys = ki;
  *res_vals = vi;
  return KTJ_LAUNCH_CHECK();
}

/* ---- the same sort on single 64-bit words ----
 * When the composite key and the arrival index fit one word, the sort moves 8 bytes per row and
 * pass instead of 12 and needs no separate index array.  The first pass reads the full keys
 * (arrival index = position) and consumes their lowest digit, so the words it writes hold only
 * the remaining key bits above the index: word = (key >> BITS) << idx_bits | index.  Later passes
 * take their digit from the word; the last one writes the bare indices.  The per-tile digit
 * counts of the first pass come from the kernel that builds the keys. */
/* How many passes there are is the plan that k_collect_distinct leaves on the device: the host launches as
 * many as it expects, those beyond the plan end at once, and a plan beyond them (or one that does not fit
 * a word) is flagged for the host to take the pass again, looking at the plan (KTJ_DEVERR_CAREFUL). */
/* Where the word has room for the whole key (low != 0) the passes leave the lowest bits out, and k_sortp_finish puts the rows
 * that differ in these only into their order; otherwise the first pass's digit leaves the word. */
struct SortRun { uint32_t low, passes; };
__device__ __forceinline__ SortRun sort_run(const Scalars* sc, int finish) {
  SortRun r;
  r.low = finish ? sc->sort.low_bits : 0u;
  const uint32_t bits = sc->sort.key_bits - r.low;
  r.passes = bits ? (bits + SORTP_BITS - 1u) / SORTP_BITS : 1u;
  return r;
}
__device__ __forceinline__ bool sort_pass_idle(const Scalars* sc, const SortRun& r, uint32_t pass) { return sc->error != 0 || pass >= r.passes; }
__device__ __forceinline__ uint32_t sort_shift(const SortRun& r, uint32_t pass, uint32_t idx_bits) { return idx_bits + r.low + (r.low ? pass : pass - 1u) * SORTP_BITS; }
__device__ __forceinline__ bool sort_words_suffice(const Scalars* sc, const SortRun& r, uint32_t key_bits, uint32_t idx_bits, uint32_t passes_launched) {
  return sc->error == 0 && key_bits <= 62u && (r.low ? key_bits : key_bits > SORTP_BITS ? key_bits - SORTP_BITS : 0u) + idx_bits <= 64u &&
         r.passes <= passes_launched;
}
__device__ __forceinline__ uint64_t sort_key(const SortPlan& p, uint64_t rank_dev, uint64_t rank_res, uint64_t rel) {
  return (((rank_dev << p.res_bits) | rank_res) << p.ts_bits) | rel;
}
__device__ __forceinline__ uint64_t sort_key_dropped(const SortPlan& p) { return (uint64_t)p.n_dev << (p.res_bits + p.ts_bits); } /* behind everything */
template <int BITS, int THREADS, int ITEMS_> struct SortP {
  static constexpr int NB = 1 << BITS;
  static constexpr int WAVES = THREADS / 64;
  static constexpr int ITEMS = ITEMS_; /* keys per thread (sort_items) */
  static constexpr int TILE = THREADS * ITEMS;
  static constexpr int WAVE_KEYS = 64 * ITEMS;
  static_assert(NB % THREADS == 0 || THREADS % NB == 0, "digits and threads must divide");
};

/* CHAIN: for k_sortp_chain, whose counts are tile by tile (hist[(pass * n_blocks + tile) * 256 + digit]) and, behind
 * the first pass's, start from zero. */
template <int BITS, int THREADS, int ITEMS, bool CHAIN>
__global__ void __launch_bounds__(THREADS)
k_sortp_make_keys(Columns c, uint64_t n, SortSets s, Scalars* sc, uint32_t idx_bits, uint32_t passes_launched, int finish, uint64_t* keys, uint32_t* hist,
                  uint32_t n_blocks) {
  using P = SortP<BITS, THREADS, ITEMS>;
  const SortPlan plan = sc->sort;
  const SortRun run = sort_run(sc, finish);
  if (!sort_words_suffice(sc, run, plan.key_bits, idx_bits, passes_launched)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) flag_error(sc, KTJ_DEVERR_CAREFUL);
    return;
  }
  __shared__ uint32_t h[P::NB];
  for (int d = threadIdx.x; d < P::NB; d += THREADS) h[d] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * P::TILE;
  const uint64_t ts_min = sc->ts_min_biased;
  constexpr int G = ITEMS < 4 ? ITEMS : 4; /* rows per thread whose loads are in flight together */
  RankMemo memo_dev{0, 0, false}, memo_res{0, 0, false};
  for (int r0 = 0; r0 < P::ITEMS; r0 += G) {
    uint32_t meta[G];
    uint64_t dev[G], res[G], ts[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const uint64_t at = base + (uint64_t)(r0 + g) * THREADS + threadIdx.x, a = at < n ? at : n - 1; /* (what is behind the last does not count) */
      meta[g] = c.meta[a];
      dev[g] = (uint64_t)c.dev[a];
      res[g] = (uint64_t)c.res[a];
      ts[g] = (uint64_t)c.ts[a];
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const uint64_t a = base + (uint64_t)(r0 + g) * THREADS + threadIdx.x;
      if (a >= n) continue;
      uint64_t key = sort_key_dropped(plan);
      if (meta[g] & KTJ_M_VALID) {
        const uint64_t rd = set_rank_memo(s.dev_keys, s.dev_rank, dev[g], memo_dev);
        const uint64_t rr = set_rank_memo(s.res_keys, s.res_rank, res[g], memo_res);
        key = sort_key(plan, rd, rr, (ts[g] ^ 0x8000000000000000ULL) - ts_min);
      }
      keys[a] = key;
      atomicAdd(&h[(uint32_t)(key >> run.low) & (P::NB - 1u)], 1u);
    }
  }
  __syncthreads();
  if (CHAIN) {
    for (uint32_t k = threadIdx.x; k < run.passes * P::NB; k += THREADS)
      hist[((uint64_t)(k / P::NB) * n_blocks + blockIdx.x) * P::NB + k % P::NB] = k < P::NB ? h[k] : 0u;
  } else if (hist != nullptr)
    for (int d = threadIdx.x; d < P::NB; d += THREADS) hist[(uint64_t)d * n_blocks + blockIdx.x] = h[d]; /* digit-major */
}
template <int BITS, int THREADS, int ITEMS>
__global__ void __launch_bounds__(THREADS)
k_sortp_hist(const uint64_t* words, uint64_t n, uint32_t pass, uint32_t idx_bits, int finish, const Scalars* sc, uint32_t* hist, uint32_t n_blocks) {
  using P = SortP<BITS, THREADS, ITEMS>;
  const SortRun run = sort_run(sc, finish);
  if (sort_pass_idle(sc, run, pass)) return;
  const uint32_t shift = sort_shift(run, pass, idx_bits);
  __shared__ uint32_t h[P::NB];
  for (int d = threadIdx.x; d < P::NB; d += THREADS) h[d] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * P::TILE;
  uint64_t word[P::ITEMS]; /* (all asked for before any is counted: under a condition each is waited for before the next; 733 000 keys 6.6 us, now 4.8) */
#pragma unroll
  for (int r = 0; r < P::ITEMS; ++r) { const uint64_t i = base + (uint64_t)r * THREADS + threadIdx.x; word[r] = words[i < n ? i : n - 1]; }
#pragma unroll
  for (int r = 0; r < P::ITEMS; ++r)
    if (base + (uint64_t)r * THREADS + threadIdx.x < n) atomicAdd(&h[(uint32_t)(word[r] >> shift) & (P::NB - 1u)], 1u);
  __syncthreads();
  for (int d = threadIdx.x; d < P::NB; d += THREADS) hist[(uint64_t)d * n_blocks + blockIdx.x] = h[d];
}
/* The per-tile digit counts (digit-major: hist[d * n_blocks + tile]) become, for every digit, the
 * running count over the tiles before each tile, and the digit's total goes to totals[d]: workgroup
 * d scans row d, every thread a contiguous piece of it.  One launch; the digits' own offsets (a scan
 * over 256 totals) are left to every scatter workgroup. */
template <int THREADS>
__global__ void __launch_bounds__(THREADS)
k_sortp_scan_digits(uint32_t* hist, uint32_t n_blocks, uint32_t* totals, uint32_t pass, int finish, const Scalars* sc) {
  if (sort_pass_idle(sc, sort_run(sc, finish), pass)) return;
  __shared__ uint32_t wave_tot[THREADS / 64];
  uint32_t* row = hist + (uint64_t)blockIdx.x * n_blocks;
  const uint32_t per = (n_blocks + THREADS - 1) / THREADS;
  const uint32_t lo = threadIdx.x * per < n_blocks ? threadIdx.x * per : n_blocks;
  const uint32_t hi = lo + per < n_blocks ? lo + per : n_blocks;
  /* eight at a time (one at a time, each waited for: 13.1 us for the 5372 tiles of 22 million keys, now 11.7) */
  uint32_t sum = 0;
  for (uint32_t t0 = lo; t0 < hi; t0 += 8u) {
    uint32_t c[8];
#pragma unroll
    for (uint32_t j = 0; j < 8u; ++j) c[j] = row[t0 + j < hi ? t0 + j : t0];
#pragma unroll
    for (uint32_t j = 0; j < 8u; ++j) sum += t0 + j < hi ? c[j] : 0u;
  }
  uint32_t inc = sum;
  const uint32_t lane = lane_id(), w = threadIdx.x >> 6;
  for (int o = 1; o < 64; o <<= 1) { const uint32_t v = __shfl_up(inc, o); if (lane >= (uint32_t)o) inc += v; }
  if (lane == 63) wave_tot[w] = inc;
  __syncthreads();
  uint32_t run = inc - sum;
  uint32_t all = 0;
  for (uint32_t k = 0; k < THREADS / 64; ++k) { if (k < w) run += wave_tot[k]; all += wave_tot[k]; }
  for (uint32_t t0 = lo; t0 < hi; t0 += 8u) {
    uint32_t c[8];
#pragma unroll
    for (uint32_t j = 0; j < 8u; ++j) c[j] = row[t0 + j < hi ? t0 + j : t0];
#pragma unroll
    for (uint32_t j = 0; j < 8u; ++j) if (t0 + j < hi) { row[t0 + j] = run; run += c[j]; }
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = all;
}

template <int BITS, int THREADS, int ITEMS, bool FROM_KEYS>
__global__ void __launch_bounds__(THREADS)
k_sortp_scatter(const uint64_t* in, uint64_t* words_out, uint32_t* perm_out, uint64_t n, uint32_t pass, uint32_t idx_bits, int finish, const Scalars* sc,
                const uint32_t* hist_scanned, const uint32_t* totals, uint32_t n_blocks) {
  using P = SortP<BITS, THREADS, ITEMS>;
  const SortRun run = sort_run(sc, finish);
  if (sort_pass_idle(sc, run, pass)) return;
  const bool TO_PERM = pass + 1u == run.passes && run.low == 0;
  const uint32_t shift = FROM_KEYS ? run.low : sort_shift(run, pass, idx_bits);
  const uint32_t gone = run.low ? 0u : (uint32_t)BITS; /* of the key, from the word */
  __shared__ uint64_t s_word[P::TILE];
  __shared__ uint16_t s_digit[FROM_KEYS ? P::TILE : 1]; /* the first pass's digit is no longer part of the word */
  __shared__ uint32_t wave_run[P::WAVES][P::NB]; /* count per (wavefront, digit), then its start inside the digit's run */
  __shared__ uint32_t digit_start[P::NB];        /* start of the digit's run inside the tile     */
  __shared__ uint32_t base_of[P::NB];            /* global offset of this tile's run per digit   */
  __shared__ uint32_t wave_tot[P::WAVES];
  const uint32_t w = threadIdx.x >> 6, lane = lane_id();
  const uint64_t tile_base = (uint64_t)blockIdx.x * P::TILE;
  const uint64_t chunk = tile_base + (uint64_t)w * P::WAVE_KEYS;
  /* The words and the digits' counts are asked for at once, in front of everything (one after the other: the first pass of 22 million
   * keys 104 us, now 94, of 733 000 13.1 and 11.2).  Those behind the
   * last are its copies and not counted. */
  uint64_t word[P::ITEMS];
  uint32_t rank[P::ITEMS];
  uint16_t dig[P::ITEMS];
  uint32_t total_of = 0, tiles_before = 0;
  static_assert(P::NB <= THREADS, "a thread scans one digit's total");
  if (hist_scanned != nullptr) {
    const uint32_t d = (int)threadIdx.x < P::NB ? threadIdx.x : 0u;
    total_of = totals[d];
    tiles_before = hist_scanned[(uint64_t)d * n_blocks + blockIdx.x];
  }
  /* this pass is the last to read the words: where they are more than the last-level cache keeps
   * between the count and the scatter anyway, they are loaded past the L2's usual replacement
   * (config 3, 22 M words: 1.20 -> 1.11 ms for the sort; at 11 M words the hint costs 2 %) */
  if (n > SORTP_STREAM_N) {
#pragma unroll
    for (int r = 0; r < P::ITEMS; ++r) { const uint64_t i = chunk + (uint64_t)r * 64u + lane; word[r] = load_once(&in[i < n ? i : n - 1]); }
  } else {
#pragma unroll
    for (int r = 0; r < P::ITEMS; ++r) { const uint64_t i = chunk + (uint64_t)r * 64u + lane; word[r] = in[i < n ? i : n - 1]; }
  }
  {
    /* where a digit's run begins in the output: the totals of the digits before it, scanned here by
     * every workgroup (256 values), plus the count of that digit in the tiles before this one */
    const uint32_t tot = (int)threadIdx.x < P::NB ? total_of : 0u;
    uint32_t inc = tot;
    for (int o = 1; o < 64; o <<= 1) { const uint32_t v = __shfl_up(inc, o); if (lane >= (uint32_t)o) inc += v; }
    if (lane == 63) wave_tot[w] = inc;
    __syncthreads();
    uint32_t digit_base = inc - tot;
    for (uint32_t k = 0; k < w; ++k) digit_base += wave_tot[k];
    if ((int)threadIdx.x < P::NB) {
      const int d = (int)threadIdx.x;
      base_of[d] = hist_scanned != nullptr ? digit_base + tiles_before : 0u;
      for (int k = 0; k < P::WAVES; ++k) wave_run[k][d] = 0;
    }
  }
  __syncthreads();
  const uint64_t lt = lanemask_lt();
  /* my_run: this wavefront's running counts; accessed as LDS (a plain pointer to the row would
   * turn into flat accesses), re-read every round because other lanes of the wavefront update it */
  typedef volatile __attribute__((address_space(3))) uint32_t* lds_counts;
  lds_counts my_run = (lds_counts)&wave_run[w][0];
#pragma unroll
  for (int r = 0; r < P::ITEMS; ++r) {
    const uint64_t i = chunk + (uint64_t)r * 64u + lane;
    const bool valid = i < n;
    uint32_t digit;
    digit = (uint32_t)(word[r] >> shift) & (P::NB - 1u);
    if (FROM_KEYS) word[r] = ((word[r] >> gone) << idx_bits) | i;
    dig[r] = (uint16_t)digit;
    /* lanes of this wavefront holding the same digit */
    uint64_t peers = __ballot(valid ? 1 : 0);
#pragma unroll
    for (int b = 0; b < BITS; ++b) {
      const uint64_t bal = __ballot((digit >> b) & 1u);
      peers &= ((digit >> b) & 1u) ? bal : ~bal;
    }
    const uint32_t rank_in_wave = (uint32_t)__popcll(peers & lt);
    const uint32_t before = my_run[digit];   /* same digit in earlier rounds of this wavefront */
    rank[r] = before + rank_in_wave;
    if (valid && rank_in_wave == 0) my_run[digit] = before + (uint32_t)__popcll(peers);
  }
  __syncthreads();
  {
    /* per digit: wavefront counts -> starts inside the digit's run; digit totals -> exclusive scan.
     * A thread owns K consecutive digits (or none, where there are more threads than digits). */
    constexpr int K = P::NB >= THREADS ? P::NB / THREADS : 1;
    const bool owner = (int)threadIdx.x * K < P::NB;
    uint32_t tot[K], sum = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      uint32_t t = 0;
      if (owner) {
        const int d = (int)threadIdx.x * K + j;
        for (int k = 0; k < P::WAVES; ++k) { const uint32_t cnt = wave_run[k][d]; wave_run[k][d] = t; t += cnt; }
      }
      tot[j] = t;
      sum += t;
    }
    uint32_t inc = sum;
    for (int o = 1; o < 64; o <<= 1) { const uint32_t t = __shfl_up(inc, o); if (lane >= (uint32_t)o) inc += t; }
    if (lane == 63) wave_tot[w] = inc;
    __syncthreads();
    uint32_t start = inc - sum;
    for (uint32_t k = 0; k < w; ++k) start += wave_tot[k];
    if (owner) {
#pragma unroll
      for (int j = 0; j < K; ++j) { digit_start[(int)threadIdx.x * K + j] = start; start += tot[j]; }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < P::ITEMS; ++r) {
    if (chunk + (uint64_t)r * 64u + lane < n) {
      const uint32_t digit = dig[r];
      const uint32_t p = digit_start[digit] + wave_run[w][digit] + rank[r];
      s_word[p] = word[r];
      if (FROM_KEYS) s_digit[p] = dig[r];
    }
  }
  __syncthreads();
  const uint32_t cnt = (uint32_t)(n - tile_base < (uint64_t)P::TILE ? n - tile_base : (uint64_t)P::TILE);
  const uint64_t idx_mask = idx_bits >= 64 ? ~0ULL : ((1ULL << idx_bits) - 1ULL);
  for (uint32_t p = threadIdx.x; p < cnt; p += THREADS) {
    const uint64_t v = s_word[p];
    const uint32_t digit = FROM_KEYS ? (uint32_t)s_digit[p] : ((uint32_t)(v >> shift) & (P::NB - 1u));
    /* a single tile (no counts given): the tile's order is the output's */
    const uint64_t dst = hist_scanned != nullptr ? (uint64_t)base_of[digit] + (p - digit_start[digit]) : (uint64_t)p;
    if (TO_PERM) perm_out[dst] = (uint32_t)(v & idx_mask);
    else words_out[dst] = v;
  }
}

/* A trace of one tile: keys, every pass and the permutation in one launch of one workgroup (six
 * launches of a few microseconds each otherwise).  Keys and arrival indices stay in registers and
 * LDS between the passes; a pass ranks the keys as k_sortp_scatter does (ballots among the lanes of
 * a wavefront, running counts per wavefront and digit) and puts them in LDS in the new order, from
 * where every thread takes the keys of its positions for the next pass.  Bound by the rounds of a wavefront,
 * one key per lane each: sixteen wavefronts with four rounds a pass instead of four with sixteen, 4001 keys
 * 56 -> 29 us. */
template <int BITS, int THREADS, int ITEMS>
__global__ void __launch_bounds__(THREADS)
k_sortp_single(Columns c, uint32_t n, SortSets s, Scalars* sc, uint32_t* perm_out) {
  using P = SortP<BITS, THREADS, ITEMS>;
  const SortPlan plan = sc->sort;
  const uint32_t key_bits = plan.key_bits;
  if (!sort_words_suffice(sc, sort_run(sc, 0), key_bits, 0u, 64u)) { /* key and index are kept apart here */
    if (threadIdx.x == 0) flag_error(sc, KTJ_DEVERR_CAREFUL);
    return;
  }
  __shared__ uint64_t s_key[P::TILE];
  __shared__ uint16_t s_idx[P::TILE];
  __shared__ uint32_t wave_run[P::WAVES][P::NB];
  __shared__ uint32_t digit_start[P::NB];
  __shared__ uint32_t wave_tot[P::WAVES];
  static_assert(P::TILE <= 65536, "arrival indices are kept as 16 bits");
  static_assert(P::NB <= THREADS, "a thread owns one digit");
  const uint32_t w = threadIdx.x >> 6, lane = lane_id();
  const uint64_t lt = lanemask_lt();
  const uint32_t chunk = w * P::WAVE_KEYS;
  typedef volatile __attribute__((address_space(3))) uint32_t* lds_counts;
  lds_counts my_run = (lds_counts)&wave_run[w][0];
  uint64_t key[P::ITEMS];
  uint16_t idx[P::ITEMS];
  uint32_t rank[P::ITEMS];
  uint16_t dig[P::ITEMS];
  const uint64_t ts_min = sc->ts_min_biased;
#pragma unroll
  for (int r = 0; r < P::ITEMS; ++r) {
    const uint32_t a = chunk + (uint32_t)r * 64u + lane;
    uint64_t k = sort_key_dropped(plan);
    if (a < n && (c.meta[a] & KTJ_M_VALID)) {
      const uint64_t rd = set_rank(s.dev_keys, s.dev_rank, (uint64_t)c.dev[a]);
      const uint64_t rr = set_rank(s.res_keys, s.res_rank, (uint64_t)c.res[a]);
      k = sort_key(plan, rd, rr, ((uint64_t)c.ts[a] ^ 0x8000000000000000ULL) - ts_min);
    }
    key[r] = k;
    idx[r] = (uint16_t)a;
  }
  const uint32_t passes = key_bits ? (key_bits + BITS - 1u) / BITS : 1u;
  for (uint32_t pass = 0; pass < passes; ++pass) {
    const uint32_t shift = pass * BITS;
#pragma unroll
    for (int k = 0; k < P::WAVES * P::NB / THREADS; ++k) (&wave_run[0][0])[k * THREADS + (int)threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < P::ITEMS; ++r) {
      const bool valid = chunk + (uint32_t)r * 64u + lane < n;
      const uint32_t digit = (uint32_t)(key[r] >> shift) & (P::NB - 1u);
      dig[r] = (uint16_t)digit;
      uint64_t peers = __ballot(valid ? 1 : 0);
#pragma unroll
      for (int b = 0; b < BITS; ++b) {
        const uint64_t bal = __ballot((digit >> b) & 1u);
        peers &= ((digit >> b) & 1u) ? bal : ~bal;
      }
      const uint32_t rank_in_wave = (uint32_t)__popcll(peers & lt);
      const uint32_t before = my_run[digit];
      rank[r] = before + rank_in_wave;
      if (valid && rank_in_wave == 0) my_run[digit] = before + (uint32_t)__popcll(peers);
    }
    __syncthreads();
    {
      /* thread d: the wavefronts' counts of digit d become their starts inside the digit's run, the
       * digit's total goes into the scan that gives the run's start inside the tile */
      const int d = (int)threadIdx.x;
      uint32_t t = 0, inc = 0;
      if (d < P::NB) {
#pragma unroll
        for (int k = 0; k < P::WAVES; ++k) { const uint32_t cnt = wave_run[k][d]; wave_run[k][d] = t; t += cnt; }
        inc = t;
        for (int o = 1; o < 64; o <<= 1) { const uint32_t v = __shfl_up(inc, o); if (lane >= (uint32_t)o) inc += v; }
        if (lane == 63) wave_tot[w] = inc;
      }
      __syncthreads();
      if (d < P::NB) {
        uint32_t start = inc - t;
        for (uint32_t k = 0; k < w; ++k) start += wave_tot[k];
        digit_start[d] = start;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < P::ITEMS; ++r) {
      if (chunk + (uint32_t)r * 64u + lane < n) {
        const uint32_t digit = dig[r];
        const uint32_t p = digit_start[digit] + wave_run[w][digit] + rank[r];
        s_key[p] = key[r];
        s_idx[p] = idx[r];
      }
    }
    __syncthreads();
    if (pass + 1 == passes) break;
#pragma unroll
    for (int r = 0; r < P::ITEMS; ++r) {
      const uint32_t a = chunk + (uint32_t)r * 64u + lane;
      if (a < n) { key[r] = s_key[a]; idx[r] = s_idx[a]; }
    }
    __syncthreads();
  }
  for (uint32_t p = threadIdx.x; p < n; p += THREADS) perm_out[p] = s_idx[p];
}

/* The words are in order but for their lowest bits (of the key; the index below them makes every word another).  Rows that differ
 * in these only are neighbours, rows of a track within 65 us at most: a group.  They are in order of arrival, mostly that of their
 * times; a row moves up by the rows in front of it that are larger and down by those behind it that are smaller.  A row is
 * compared as 32 bits, the number of its group in the workgroup's rows and the lowest bits, so that rows of other groups need no
 * look of their own.  Groups of more than FINISH_MOST rows must be in order already, or the whole order is made again with passes over all
 * bits (KTJ_DEVERR_UNSORTED).  How long a group is, every workgroup that has a row of it sees alike: it loads that many rows in front
 * of and behind its own.
 *
 * Takes the place of one or two of five passes (a count, a scan, a scatter each: 135 us for 22 million rows). */
#define FINISH_MOST 256u
#define CHAIN_MAX_N 98304ull /* of sort_packed_chain */
template <int THREADS, int ITEMS> struct FinishLds {
  static constexpr uint32_t ROWS = ITEMS + 2, SPAN = THREADS * ROWS, CHUNKS = SPAN / 64u; /* the tile's rows, a turn in front of and one behind them */
  static_assert(THREADS == FINISH_MOST && CHUNKS <= 128u && SPAN < 0x10000u, "chunks of a wavefront's lanes, numbers of groups");
  uint64_t edge[CHUNKS], start[CHUNKS]; /* a chunk's last word; a bit per row: first of its group */
  uint32_t val[SPAN];
};
/* own_bits: those of Scalars::error that the launch sets */
template <int THREADS, int ITEMS>
__device__ __forceinline__ void finish_tile(const uint64_t* buf_a, const uint64_t* buf_b, uint32_t* perm, uint64_t n, uint32_t idx_bits, Scalars* sc,
                                            unsigned int own_bits, uint64_t tile, FinishLds<THREADS, ITEMS>& lds) {
  constexpr uint32_t ROWS = FinishLds<THREADS, ITEMS>::ROWS, SPAN = FinishLds<THREADS, ITEMS>::SPAN, CHUNKS = FinishLds<THREADS, ITEMS>::CHUNKS;
  uint32_t* const s_val = lds.val;
  uint64_t* const s_edge = lds.edge;
  uint64_t* const s_start = lds.start;
  const SortRun run = sort_run(sc, 1);
  /* (low of 0: the last pass has written the permutation.)  All wavefronts of a workgroup must see the same here, as they number
   * groups and compare rows for each other: what this launch sets does not count. */
  if ((sc->error & ~own_bits) != 0 || run.low == 0) return;
  const uint64_t* in = run.passes & 1u ? buf_b : buf_a;
  const uint32_t group_shift = idx_bits + run.low, lane = lane_id(), wave = threadIdx.x >> 6;
  const uint64_t idx_mask = (1ULL << idx_bits) - 1ULL;
  const uint64_t from = tile * (THREADS * ITEMS) - FINISH_MOST; /* (below 0: not loaded) */
  uint64_t word[ROWS];
  /* All loads in flight together.  Many words go past the caches, as in the scatter: left there they push out what k_gather_len reads behind
   * the joined rows (22 million rows: 94 us there instead of 84, 61 and 60 here.  11 million and less: the same). */
  if (ITEMS >= 16 && n > SORTP_STREAM_N) {
#pragma unroll
    for (uint32_t r = 0; r < ROWS; ++r) {
      const uint64_t i = from + r * THREADS + threadIdx.x; /* row, or wrapped around */
      word[r] = i < n ? load_once(&in[i]) : 0;
    }
  } else {
#pragma unroll
    for (uint32_t r = 0; r < ROWS; ++r) {
      const uint64_t i = from + r * THREADS + threadIdx.x;
      word[r] = i < n ? in[i] : 0;
    }
  }
#pragma unroll
  for (uint32_t r = 0; r < ROWS; ++r) if (lane == 63u) s_edge[r * (THREADS / 64u) + wave] = word[r];
  __syncthreads();
  uint32_t turns = 0; /* a bit per row: smaller than the one in front of it, of the same group */
#pragma unroll
  for (uint32_t r = 0; r < ROWS; ++r) {
    const uint64_t i = from + r * THREADS + threadIdx.x;
    const uint32_t c = r * (THREADS / 64u) + wave;
    uint64_t before = (uint64_t)__shfl_up((unsigned long long)word[r], 1);
    if (lane == 0u) before = s_edge[c ? c - 1u : 0u];
    /* (the first of the span begins a group whatever is in front of it: with a row of this tile that is one of too many) */
    const bool same = (c != 0u || lane != 0u) && i < n && i != 0 && ((word[r] ^ before) >> group_shift) == 0;
    const uint64_t starts = __ballot(!same);
    if (lane == 0u) s_start[c] = starts;
    turns |= (same && word[r] < before ? 1u : 0u) << r;
  }
  if (!__syncthreads_or((int)turns)) {
#pragma unroll
    for (uint32_t r = 1; r <= ITEMS; ++r) {
      const uint64_t i = from + r * THREADS + threadIdx.x;
      if (i < n) perm[i] = (uint32_t)(word[r] & idx_mask);
    }
    return;
  }
  /* Groups that are too long have three chunks without a start, and more.  One that is not in order: nothing needs this order.  (To
   * compare with 256 rows on either side before that is known took 220 us for 2 million rows in groups of 400.) */
  uint32_t stay = 0; /* a bit per row: of such a group */
  bool none = false;
  for (uint32_t c = lane; c + 2u < CHUNKS; c += 64u) none = none || (s_start[c] | s_start[c + 1u] | s_start[c + 2u]) == 0;
  if (__any(none)) { /* (the same for all wavefronts) */
#pragma unroll 1
    for (uint32_t r = 1; r <= ITEMS; ++r) {
      const uint32_t c = r * (THREADS / 64u) + wave;
      uint32_t first = 0, next = SPAN; /* of the rows of its group, as far as four chunks on either side show it */
#pragma unroll 1
      for (uint32_t q = 0; q <= 4u; ++q) {
        const uint64_t w = s_start[c - q] & (q ? ~0ULL : ~0ULL >> (63u - lane));
        if (w) { first = (c - q) * 64u + 63u - (uint32_t)__builtin_clzll(w); break; }
      }
#pragma unroll 1
      for (uint32_t q = 0; q <= 4u; ++q) {
        const uint64_t w = s_start[c + q] & (q ? ~0ULL : ~1ULL << lane);
        if (w) { next = (c + q) * 64u + (uint32_t)__builtin_ctzll(w); break; }
      }
      stay |= (next - first > FINISH_MOST ? 1u : 0u) << r;
    }
    if (__syncthreads_or((int)(stay & turns))) {
      if (threadIdx.x == 0) flag_error(sc, KTJ_DEVERR_UNSORTED);
      return;
    }
  }
  uint32_t upto0 = (uint32_t)__popcll(s_start[lane < CHUNKS ? lane : 0u]), upto1 = CHUNKS > 64u ? (uint32_t)__popcll(s_start[lane + 64u < CHUNKS ? lane + 64u : 0u]) : 0u;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t x = __shfl_up(upto0, o), y = __shfl_up(upto1, o);
    if (lane >= (uint32_t)o) { upto0 += x; upto1 += y; }
  }
  uint32_t val[ROWS];
  const uint32_t low_mask = (1u << run.low) - 1u, all0 = __builtin_amdgcn_readlane(upto0, 63);
#pragma unroll
  for (uint32_t r = 0; r < ROWS; ++r) {
    const uint32_t c = __builtin_amdgcn_readfirstlane(r * (THREADS / 64u) + wave);
    const uint32_t groups = c == 0u ? 0u : c <= 64u ? __builtin_amdgcn_readlane(upto0, (c - 1u) & 63u) : all0 + __builtin_amdgcn_readlane(upto1, (c - 65u) & 63u);
    const uint64_t starts = s_start[c] & (~0ULL >> (63u - lane));
    val[r] = ((groups + (uint32_t)__popcll(starts)) << 16) | ((uint32_t)(word[r] >> idx_bits) & low_mask);
    s_val[r * THREADS + threadIdx.x] = val[r];
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 1; r <= ITEMS; ++r) {
    const uint64_t i = from + r * THREADS + threadIdx.x;
    const uint32_t k = r * THREADS + threadIdx.x, v = val[r];
    const bool moving = !(stay >> r & 1u);
    uint32_t moves = 0;
    for (uint32_t d = 1; d < FINISH_MOST; d += 2u) { /* as far as any lane's group reaches */
      const uint32_t x0 = s_val[k + d], y0 = s_val[k - d], x1 = s_val[k + d + 1u], y1 = s_val[k - d - 1u];
      moves += x0 < v ? 1u : 0u;
      moves += x1 < v ? 1u : 0u;
      moves -= y0 > v ? 1u : 0u;
      moves -= y1 > v ? 1u : 0u;
      const uint32_t x = x1 ^ v, y = y1 ^ v;
      if (!__any(moving && (x < y ? x : y) < 0x10000u)) break;
    }
    if (!moving) moves = 0;
    if (i < n) perm[i + (uint64_t)(int64_t)(int32_t)moves] = (uint32_t)(word[r] & idx_mask);
  }
}
template <int THREADS, int ITEMS>
__global__ void __launch_bounds__(THREADS)
k_sortp_finish(const uint64_t* buf_a, const uint64_t* buf_b, uint32_t* perm, uint64_t n, uint32_t idx_bits, Scalars* sc) {
  __shared__ FinishLds<THREADS, ITEMS> lds;
  finish_tile<THREADS, ITEMS>(buf_a, buf_b, perm, n, idx_bits, sc, KTJ_DEVERR_UNSORTED, blockIdx.x, lds);
}
static bool finish_and_rows(const uint64_t* buf_a, const uint64_t* buf_b, uint32_t* perm, uint64_t n, uint32_t idx_bits, uint64_t tile, Scalars* sc,
                            RowsJob* job, hipStream_t st);
static hipError_t sort_finish(const uint64_t* buf_a, const uint64_t* buf_b, uint32_t* perm, uint64_t n, uint32_t idx_bits, Scalars* sc, RowsJob* job, hipStream_t st) {
  /* tiles that leave no CU without one; large ones where there are enough, as the rows around a tile are loaded twice */
  auto launch = [&](auto kernel, uint64_t tile) {
    if (finish_and_rows(buf_a, buf_b, perm, n, idx_bits, tile, sc, job, st)) return;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((n + tile - 1) / tile)), dim3(256), 0, st, buf_a, buf_b, perm, n, idx_bits, sc);
  };
  if (n <= CHAIN_MAX_N) launch(k_sortp_finish<256, 1>, 256);
  else if (n < 1ull << 20) launch(k_sortp_finish<256, 4>, 1024);
  else launch(k_sortp_finish<256, 16>, 4096);
  return KTJ_LAUNCH_CHECK();
}

template <int BITS, int THREADS, int ITEMS>
static hipError_t sort_packed_t(Columns c, uint64_t n, SortSets s, Scalars* sc, uint32_t passes, int finish, uint32_t idx_bits, uint64_t* buf_a, uint64_t* buf_b,
                                uint32_t* perm, uint32_t* hist, RowsJob* job, hipStream_t st) {
  using P = SortP<BITS, THREADS, ITEMS>;
  const uint32_t n_blocks = (uint32_t)((n + P::TILE - 1) / P::TILE);
  const dim3 g(n_blocks), b(THREADS);
  /* one tile: a pass needs no counts from other tiles, so no count and scan launches */
  const bool single = n_blocks == 1;
  uint32_t* counts = single ? nullptr : hist;
  /* the digits' totals live behind the counts (radix_tmp_elems leaves 256 spare entries) */
  uint32_t* totals = hist + (uint64_t)P::NB * n_blocks;
  static_assert(P::NB <= 256, "room for the totals behind the counts");
  hipLaunchKernelGGL((k_sortp_make_keys<BITS, THREADS, ITEMS, false>), g, b, 0, st, c, n, s, sc, idx_bits, passes, finish, buf_a, counts, n_blocks);
  if (!single) hipLaunchKernelGGL((k_sortp_scan_digits<THREADS>), dim3(P::NB), b, 0, st, hist, n_blocks, totals, 0u, finish, (const Scalars*)sc);
  hipLaunchKernelGGL((k_sortp_scatter<BITS, THREADS, ITEMS, true>), g, b, 0, st, (const uint64_t*)buf_a, buf_b, perm, n, 0u, idx_bits, finish,
                     (const Scalars*)sc, (const uint32_t*)counts, (const uint32_t*)totals, n_blocks);
  uint64_t* in = buf_b; uint64_t* out = buf_a;
  for (uint32_t p = 1; p < passes; ++p) {
    if (!single) {
      hipLaunchKernelGGL((k_sortp_hist<BITS, THREADS, ITEMS>), g, b, 0, st, (const uint64_t*)in, n, p, idx_bits, finish, (const Scalars*)sc, hist, n_blocks);
      hipLaunchKernelGGL((k_sortp_scan_digits<THREADS>), dim3(P::NB), b, 0, st, hist, n_blocks, totals, p, finish, (const Scalars*)sc);
    }
    hipLaunchKernelGGL((k_sortp_scatter<BITS, THREADS, ITEMS, false>), g, b, 0, st, (const uint64_t*)in, out, perm, n, p, idx_bits, finish,
                       (const Scalars*)sc, (const uint32_t*)counts, (const uint32_t*)totals, n_blocks);
    uint64_t* t = in; in = out; out = t;
  }
  if (finish) return sort_finish(buf_a, buf_b, perm, n, idx_bits, sc, job, st);
  return KTJ_LAUNCH_CHECK();
}

/* Up to CHAIN_MAX_N keys a pass is one launch instead of three (count, scan, scatter: with five passes that was
 * half the launches of a trace of 30 000 records, each some 3 us for hardly a microsecond of work):
 *   - a workgroup adds the digit counts of the tiles before its own, and of all, up by itself: a few dozen
 *     loads per thread, all in flight together;
 *   - while it puts its keys to their places it counts the next pass's digits per tile of the output, in LDS
 *     (16 bits each: a tile holds 1024 keys), and adds what it has to the next pass's counts.
 * Bound by the chain of its short phases, some 5 us whatever the tile holds: one key per thread is the
 * shortest of them (a first form that put a tile in order before it was written out took 17 us more for 30 000
 * records with tiles of 2048 keys, and 26 us more with 4096).  Three launches a pass against this, whole pass:
 * 4500 records 203 -> 177 us, 30 000 219 -> 202, 60 000 224 -> 216, 90 000 228 both, 120 000 229 -> 234; counts to
 * add up and cells to hand on grow with the tiles (at 733 000 keys a pass took 30 us instead of 25). */
#define CHAIN_THREADS 1024
template <int BITS, bool FROM_KEYS>
__global__ void __launch_bounds__(CHAIN_THREADS)
k_sortp_chain(const uint64_t* in, uint64_t* words_out, uint32_t* perm_out, uint32_t n, uint32_t pass, uint32_t idx_bits, int finish, const Scalars* sc,
              uint32_t* hist, uint32_t n_blocks) {
  using P = SortP<BITS, CHAIN_THREADS, 1>;
  constexpr uint32_t NB = P::NB, GROUPS = CHAIN_THREADS / NB;
  const SortRun run = sort_run(sc, finish);
  if (sort_pass_idle(sc, run, pass)) return;
  const bool LAST = pass + 1u == run.passes, TO_PERM = LAST && run.low == 0;
  const uint32_t shift = FROM_KEYS ? run.low : sort_shift(run, pass, idx_bits);
  const uint32_t next_shift = sort_shift(run, pass + 1u, idx_bits);
  __shared__ uint32_t next[CHAIN_MAX_N / P::TILE * (NB / 2u)]; /* two cells a word */
  __shared__ uint32_t wave_run[P::WAVES][NB];
  __shared__ uint32_t part[2][GROUPS][NB]; /* counts before this tile, of all tiles */
  __shared__ uint32_t base_of[NB];
  __shared__ uint32_t wave_tot[NB / 64];
  const uint32_t w = threadIdx.x >> 6, lane = lane_id();
  const uint32_t tile_base = blockIdx.x * P::TILE, i = tile_base + threadIdx.x;
  const bool valid = i < n;
  uint64_t word = in[valid ? i : n - 1u];
  {
    const uint32_t d = threadIdx.x & (NB - 1u), group = threadIdx.x / NB;
    const uint32_t* row = hist + (uint64_t)pass * n_blocks * NB + d;
    uint32_t before = 0, all = 0;
#pragma unroll 8
    for (uint32_t t = group; t < n_blocks; t += GROUPS) {
      const uint32_t c = row[t * NB];
      all += c;
      before += t < blockIdx.x ? c : 0u;
    }
    part[0][group][d] = before;
    part[1][group][d] = all;
  }
  for (uint32_t k = threadIdx.x; k < P::WAVES * NB; k += CHAIN_THREADS) (&wave_run[0][0])[k] = 0;
  if (!LAST)
    for (uint32_t k = threadIdx.x; k < n_blocks * (NB / 2u); k += CHAIN_THREADS) next[k] = 0;
  __syncthreads();
  const uint32_t digit = (uint32_t)(word >> shift) & (NB - 1u);
  if (FROM_KEYS) word = ((word >> (run.low ? 0u : (uint32_t)BITS)) << idx_bits) | i;
  uint64_t peers = __ballot(valid ? 1 : 0);
#pragma unroll
  for (int b = 0; b < BITS; ++b) {
    const uint64_t bal = __ballot((digit >> b) & 1u);
    peers &= ((digit >> b) & 1u) ? bal : ~bal;
  }
  const uint32_t rank = (uint32_t)__popcll(peers & lanemask_lt());
  if (valid && rank == 0) wave_run[w][digit] = (uint32_t)__popcll(peers);
  __syncthreads();
  /* thread d: where each wavefront's keys with digit d begin among the tile's, and where the tile's go */
  uint32_t before = 0, in_all = 0, inc = 0;
  const uint32_t d = threadIdx.x;
  if (d < NB) {
    uint32_t run = 0;
#pragma unroll
    for (int k = 0; k < P::WAVES; ++k) { const uint32_t cnt = wave_run[k][d]; wave_run[k][d] = run; run += cnt; }
#pragma unroll
    for (uint32_t g = 0; g < GROUPS; ++g) { before += part[0][g][d]; in_all += part[1][g][d]; }
    inc = in_all;
    for (int o = 1; o < 64; o <<= 1) { const uint32_t t = __shfl_up(inc, o); if (lane >= (uint32_t)o) inc += t; }
    if (lane == 63) wave_tot[w] = inc;
  }
  __syncthreads();
  if (d < NB) {
    uint32_t base = inc - in_all + before;
    for (uint32_t k = 0; k < w; ++k) base += wave_tot[k];
    base_of[d] = base;
  }
  __syncthreads();
  if (valid) { /* (a digit's keys of a tile lie together: hardly more lines than if the tile were put in order first) */
    const uint32_t dst = base_of[digit] + wave_run[w][digit] + rank;
    if (TO_PERM) perm_out[dst] = (uint32_t)(word & ((1ULL << idx_bits) - 1ULL));
    else {
      words_out[dst] = word;
      if (LAST) return;
      const uint32_t cell = (dst / (uint32_t)P::TILE) * NB + ((uint32_t)(word >> next_shift) & (NB - 1u));
      atomicAdd(&next[cell >> 1], cell & 1u ? 0x10000u : 1u);
    }
  }
  if (LAST) return;
  __syncthreads();
  uint32_t* next_hist = hist + (uint64_t)(pass + 1u) * n_blocks * NB;
  for (uint32_t k = threadIdx.x; k < n_blocks * (NB / 2u); k += CHAIN_THREADS) {
    const uint32_t c = next[k];
    if (c & 0xFFFFu) atomicAdd(&next_hist[2u * k], c & 0xFFFFu);
    if (c >> 16) atomicAdd(&next_hist[2u * k + 1u], c >> 16);
  }
}
template <int BITS>
static hipError_t sort_packed_chain(Columns c, uint64_t n, SortSets s, Scalars* sc, uint32_t passes, int finish, uint32_t idx_bits, uint64_t* buf_a,
                                    uint64_t* buf_b, uint32_t* perm, uint32_t* hist, RowsJob* job, hipStream_t st) {
  using P = SortP<BITS, CHAIN_THREADS, 1>;
  const uint32_t n_blocks = (uint32_t)((n + P::TILE - 1) / P::TILE);
  const dim3 g(n_blocks), b(CHAIN_THREADS);
  hipLaunchKernelGGL((k_sortp_make_keys<BITS, CHAIN_THREADS, 1, true>), g, b, 0, st, c, n, s, sc, idx_bits, passes, finish, buf_a, hist, n_blocks);
  hipLaunchKernelGGL((k_sortp_chain<BITS, true>), g, b, 0, st, (const uint64_t*)buf_a, buf_b, perm, (uint32_t)n, 0u, idx_bits, finish,
                     (const Scalars*)sc, hist, n_blocks);
  uint64_t* in = buf_b; uint64_t* out = buf_a;
  for (uint32_t p = 1; p < passes; ++p) {
    hipLaunchKernelGGL((k_sortp_chain<BITS, false>), g, b, 0, st, (const uint64_t*)in, out, perm, (uint32_t)n, p, idx_bits, finish,
                       (const Scalars*)sc, hist, n_blocks);
    uint64_t* t = in; in = out; out = t;
  }
  if (finish) return sort_finish(buf_a, buf_b, perm, n, idx_bits, sc, job, st);
  return KTJ_LAUNCH_CHECK();
}
#define SORTP_THREADS 256
/* tests: the one-launch sort of a single tile switched off, so that such a trace takes the passes of a large one */
static bool g_sortp_no_single = false;
void sort_packed_force_passes(bool on) { g_sortp_no_single = on; }
bool sort_packed_passes_forced() { return g_sortp_no_single; }
bool sort_packed_in_one_launch(uint64_t n) { return n <= (uint64_t)SORTP_THREADS * 16u && !g_sortp_no_single; }
static uint32_t sort_idx_bits(uint64_t n) { return (uint32_t)(64 - __builtin_clzll(n > 1 ? n - 1 : 1)); }
bool sort_packed_fits(uint64_t n, const SortPlan& plan) {
  return plan.key_bits <= 62u && (plan.key_bits > SORTP_BITS ? plan.key_bits - SORTP_BITS : 0u) + sort_idx_bits(n) <= 64u;
}
uint32_t sort_packed_passes(const SortPlan& plan, bool finish) {
  const uint32_t bits = plan.key_bits - (finish ? plan.low_bits : 0u);
  return bits ? (bits + SORTP_BITS - 1u) / SORTP_BITS : 1u;
}
hipError_t sort_packed(Columns c, uint64_t n, SortSets s, Scalars* sc, uint32_t passes, bool finish, uint64_t* buf_a, uint64_t* buf_b, uint32_t* perm,
                       uint32_t* hist, uint32_t* chain_hist, RowsJob* job, hipStream_t st) {
  if (n == 0) return hipSuccess;
  const uint32_t idx_bits = sort_idx_bits(n);
  if (sort_packed_in_one_launch(n)) {
    hipLaunchKernelGGL((k_sortp_single<SORTP_BITS, 1024, 4>), dim3(1), dim3(1024), 0, st, c, (uint32_t)n, s, sc, perm);
    return KTJ_LAUNCH_CHECK();
  }
  /* a few thousand keys are one tile; then one launch a pass, where the counts of all passes (1 KiB per pass and
   * tile) fit the 8 bytes per row of chain_hist: eight passes of an odd few thousand keys do not.  Behind that tiles by sort_items */
  if (n > (uint64_t)SORTP_THREADS * 16u && n <= CHAIN_MAX_N && 256ull * passes * ((n + CHAIN_THREADS - 1) / CHAIN_THREADS) <= 2 * (n + 1))
    return sort_packed_chain<SORTP_BITS>(c, n, s, sc, passes, finish, idx_bits, buf_a, buf_b, perm, chain_hist, job, st);
  const uint32_t items = n > (uint64_t)SORTP_THREADS * 16u ? sort_items(n) : 16u;
  const auto tiles = [&](auto sort) { return sort(c, n, s, sc, passes, finish, idx_bits, buf_a, buf_b, perm, hist, job, st); };
  return items == 2u ? tiles(sort_packed_t<SORTP_BITS, SORTP_THREADS, 2>) : items == 4u ? tiles(sort_packed_t<SORTP_BITS, SORTP_THREADS, 4>)
       : items == 8u ? tiles(sort_packed_t<SORTP_BITS, SORTP_THREADS, 8>) : tiles(sort_packed_t<SORTP_BITS, SORTP_THREADS, 16>);
}

/* ------------------------------------------------------------------------------------------ */
/* stage 4a: joined rows and exact byte lengths, arrival order                                  */
/* ------------------------------------------------------------------------------------------ */
__device__ __forceinline__ void store_row(MatRow* dst, const MatRow& m) {
  const uint4* s = reinterpret_cast<const uint4*>(&m);
  uint4* d = reinterpret_cast<uint4*>(dst);
  for (int k = 0; k < (int)(sizeof(MatRow) / 16); ++k) d[k] = s[k];
}
/* Packed rows between global memory and LDS: a lane that loads or stores its own 64- or 96-byte
 * row touches a cache line (or two) of its own with every 16-byte access, 64 lines per
 * instruction; moved by the workgroup with lane-consecutive 16-byte accesses the same bytes are
 * whole lines.  `rows` is the workgroup's first row, `cnt` its number of rows; the callers put
 * the barriers (workgroups of KTJ_BLOCK).  Records are read once and joined rows written once: both go past the L2's usual
 * replacement (config 3: join stage 2.51 -> 2.26 ms).
 * All loads of a group are asked for before any is waited for, those behind the last row again for its last block: in a loop of a
 * length that the compiler does not know each was waited for and stored before the next, six trips to memory one after the other for the
 * largest records (22 million records: rows 697 -> 600 us, join 1970 -> 1880, decode 486 -> 466; 5 million operators: rows 462 -> 397). */
template <typename T>
__device__ __forceinline__ void rows_global_to_lds(const T* rows, uint32_t cnt, uint4* lds) {
  typedef unsigned int v4u __attribute__((ext_vector_type(4)));
  const v4u* g = reinterpret_cast<const v4u*>(rows);
  v4u* l = reinterpret_cast<v4u*>(lds);
  constexpr uint32_t U = sizeof(T) / 16;
  const uint32_t last = cnt * U - 1u;
  v4u x[U];
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) { const uint32_t i = threadIdx.x + k * KTJ_BLOCK; x[k] = load_once(&g[i < last ? i : last]); }
#pragma unroll
  for (uint32_t k = 0; k < U; ++k) { const uint32_t i = threadIdx.x + k * KTJ_BLOCK; l[i < last ? i : last] = x[k]; }
}
template <typename T>
__device__ __forceinline__ void rows_lds_to_global(T* rows, uint32_t cnt, const uint4* lds) {
  typedef unsigned int v4u __attribute__((ext_vector_type(4)));
  v4u* g = reinterpret_cast<v4u*>(rows);
  const v4u* l = reinterpret_cast<const v4u*>(lds);
#pragma unroll
  for (uint32_t u = 0; u < (uint32_t)(sizeof(T) / 16); ++u) { const uint32_t k = threadIdx.x + u * KTJ_BLOCK; if (k < cnt * (uint32_t)(sizeof(T) / 16)) store_once(&g[k], l[k]); }
}
/* rows that are a line of eight blocks, block b of row r at b ^ (r & 7): neighbouring lanes write theirs to other banks */
template <>
__device__ __forceinline__ void rows_lds_to_global(weave::TextRow* rows, uint32_t cnt, const uint4* lds) {
  typedef unsigned int v4u __attribute__((ext_vector_type(4)));
  v4u* g = reinterpret_cast<v4u*>(rows);
  const v4u* l = reinterpret_cast<const v4u*>(lds);
#pragma unroll
  for (uint32_t u = 0; u < 8u; ++u) { const uint32_t k = threadIdx.x + u * KTJ_BLOCK; if (k < cnt * 8u) store_once(&g[k], l[k ^ ((k >> 3) & 7u)]); }
}
template <typename T>
__device__ __forceinline__ T row_from_lds(const uint4* lds) {
  T r;
  uint4* d = reinterpret_cast<uint4*>(&r);
#pragma unroll
  for (int k = 0; k < (int)(sizeof(T) / 16); ++k) d[k] = lds[threadIdx.x * (sizeof(T) / 16) + k];
  return r;
}
template <typename T>
__device__ __forceinline__ void row_to_lds(const T& r, uint4* lds) {
  const uint4* s = reinterpret_cast<const uint4*>(&r);
#pragma unroll
  for (int k = 0; k < (int)(sizeof(T) / 16); ++k) lds[threadIdx.x * (sizeof(T) / 16) + k] = s[k];
}
struct RowStats { uint32_t n_flow = 0, n_blank = 0; };
__device__ __forceinline__ void count_row_stats(const MatRow& m, const EmitCtx& ctx, RowStats* rs) {
  if (!(m.meta & KTJ_M_VALID)) return;
  if (m.meta & KTJ_M_FLOW) ++rs->n_flow;
  if (!(m.meta & KTJ_M_NAME_BUILTIN) && m.name_id < ctx.dict.n && (dict_flags(ctx.dict, m.name_id) & KTJ_SF_NAME_UNKNOWN))
    ++rs->n_blank;
}
__device__ __forceinline__ void flush_row_stats(const RowStats& rs, Scalars* sc) {
  block_add(sc, KTJ_CNT_FLOW, rs.n_flow);
  block_add(sc, KTJ_CNT_BLANK_NAMES, rs.n_blank);
}

/* Stream Sync rows (output_json.cpp:913-943): which activity is the first of its (device, row) key
 * in emission order.  Pass a: smallest sorted position per key; pass b: the activity at that
 * position is marked.  Both run over the sorted positions of generic rows only when the stream
 * holds CUDA_SYNC activities at all. */
__device__ __forceinline__ bool is_stream_sync(const ktj_generic_rec& g, const DictViews& d) {
  return g.type == KTJ_TYPE_CUDA_SYNC && g.name_id < d.n && (dict_flags(d, g.name_id) & KTJ_SF_STREAM_SYNC);
}
__global__ void k_sync_first_a(const uint32_t* perm, uint64_t n_sorted, const ktj_generic_rec* g, uint64_t n_generic,
                               const int64_t* dev, DictViews d, uint64_t* keys, uint32_t* first_pos, Scalars* sc) {
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n_sorted) return;
  const uint64_t a = perm[p];
  if (a >= n_generic || !is_stream_sync(g[a], d)) return;
  const uint32_t slot = table_insert_counted(keys, KTJ_SYNC_CAP - 1u, stream_sync_key(dev[a], g[a].resource), &sc->n_sync_rows,
                                             KTJ_MAX_SYNC_ROWS);
  if (slot == KTJ_NOSLOT) { flag_error(sc, KTJ_DEVERR_SYNC_ROWS); return; }
  atomicMin(&first_pos[slot], (uint32_t)p);
}
__global__ void k_sync_first_b(const uint32_t* perm, uint64_t n_sorted, const ktj_generic_rec* g, uint64_t n_generic,
                               const int64_t* dev, DictViews d, const uint64_t* keys, const uint32_t* first_pos, uint32_t* is_first) {
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n_sorted) return;
  const uint64_t a = perm[p];
  if (a >= n_generic) return;
  uint32_t first = 0;
  if (is_stream_sync(g[a], d)) {
    const uint32_t slot = table_find(keys, KTJ_SYNC_CAP - 1u, stream_sync_key(dev[a], g[a].resource));
    first = slot != KTJ_NOSLOT && first_pos[slot] == (uint32_t)p;
  }
  is_first[a] = first;
}
hipError_t stream_sync_first(const uint32_t* perm, uint64_t n_sorted, const ktj_generic_rec* g, uint64_t n_generic,
                             const int64_t* dev, DictViews d, uint64_t* keys, uint32_t* first_pos, uint32_t* is_first, Scalars* sc,
                             hipStream_t st) {
  if (n_sorted == 0 || n_generic == 0) return hipSuccess;
  hipError_t e = fill_u64(keys, KTJ_EMPTY_KEY, KTJ_SYNC_CAP + 1ull, st);
  if (e != hipSuccess) return e;
  e = fill_u32(first_pos, 0xFFFFFFFFu, KTJ_SYNC_CAP + 1ull, st);
  if (e != hipSuccess) return e;
  e = fill_u32(is_first, 0u, n_generic, st);
  if (e != hipSuccess) return e;
  const dim3 grid(grid_for(n_sorted, KTJ_BLOCK)), b(KTJ_BLOCK);
  hipLaunchKernelGGL(k_sync_first_a, grid, b, 0, st, perm, n_sorted, g, n_generic, dev, d, keys, first_pos, sc);
  hipLaunchKernelGGL(k_sync_first_b, grid, b, 0, st, perm, n_sorted, g, n_generic, dev, d, (const uint64_t*)keys,
                     (const uint32_t*)first_pos, is_first);
  return KTJ_LAUNCH_CHECK();
}

/* A joined row and its length are done: the row goes to the staging area as the emit kernels want it, and this is what is
 * stored of its length. */
template <bool TEXT> struct RowOf { typedef MatRow T; };
template <> struct RowOf<true> { typedef weave::TextRow T; };
template <bool TEXT>
__device__ __forceinline__ uint32_t stage_row(const MatRow& m, const EmitCtx& ctx, const Rows& rows, uint32_t wide_at, Scalars* sc, uint4* stage) {
  if (!TEXT) { row_to_lds(m, stage); return row_length(m, ctx, sc); }
  weave::TextRow* const t = reinterpret_cast<weave::TextRow*>(stage) + threadIdx.x;
  uint32_t n = 0, tail;
  if (m.meta & KTJ_M_VALID) {
    const bool text = sc->no_text == 0;
    if (text && weave::text_row(m, ctx, rows.schemas->plan, t, threadIdx.x & 7u, rows.wide, wide_at, &n, &tail)) return n | (tail << 30);
    n = row_length(m, ctx, sc) | (text ? KTJ_KIND_LEFT << 30 : 0u); /* (all are left: no list is made, they are printed in order) */
  }
  static_assert(sizeof(MatRow) == 96, "six blocks");
  auto block = [&](uint32_t k) { __builtin_memcpy(t->w[k ^ (threadIdx.x & 7u)], reinterpret_cast<const char*>(&m) + 16u * k, 16); };
  block(0); block(1); block(2); block(3); block(4); block(5); /* (a loop would keep m in memory) */
  t->w[7u ^ (threadIdx.x & 7u)][3] = KTJ_ROW_LEFT << 24;
  return n;
}

template <bool TEXT>
__device__ __forceinline__ void mat_generic_block(const ktj_generic_rec* g, uint64_t n, uint64_t first, const EmitCtx& ctx, const uint32_t* sync_first,
                                                  Rows rows, uint32_t* len, Scalars* sc, uint64_t block, uint64_t blocks, uint4* stage) {
  RowStats rs;
  for (uint64_t base = block * KTJ_BLOCK; base < n; base += blocks * KTJ_BLOCK) {
    const uint32_t cnt = (uint32_t)(n - base < KTJ_BLOCK ? n - base : KTJ_BLOCK);
    __syncthreads(); /* the previous round's rows have left the staging area */
    rows_global_to_lds(g + base, cnt, stage);
    __syncthreads();
    const uint64_t i = base + threadIdx.x;
    const bool active = threadIdx.x < cnt;
    MatRow m;
    if (active) {
      const ktj_generic_rec rec = row_from_lds<ktj_generic_rec>(stage);
      m = mat_generic(rec, generic_device(rec, ctx.args, ctx.n_args));
      if (!generic_record_prints(rec, ctx)) m.meta &= ~KTJ_M_VALID;
      attach_own_collective(m, rec, ctx);
      mark_stream_sync(m, ctx, sync_first != nullptr && sync_first[i] != 0);
      count_row_stats(m, ctx, &rs);
    }
    __syncthreads(); /* every lane has taken its record */
    if (active) len[first + i] = stage_row<TEXT>(m, ctx, rows, (uint32_t)i, sc, stage);
    __syncthreads();
    rows_lds_to_global(static_cast<typename RowOf<TEXT>::T*>(rows.p) + first + base, cnt, stage);
  }
  flush_row_stats(rs, sc);
}
/* The pass over the runtime rows.
 * full table : correlation id → stream_src = last runtime row that carries a stream
 *              (RocmStreamQueue.h:47-54), first = first arrival index seen, for checkTimestampOrder
 *              (GenericActivityProfiler.cpp:363-395)
 * narrow table: int-narrowed id → kern_src = last in-window kernel row, copy_src = last in-window
 *              copy/malloc row (thread_local correlationToGrid/Block/Size,
 *              RocprofActivity_inl.h:28-30, 221-223, 245, 267)
 * Every row writes what device rows take over from it (timestamp, stream, grid/block or size)
 * into the payload of its slots straight away.  That is final when no two runtime rows share a
 * slot, which the returning atomicMin on `first` tells; only otherwise k_runtime_winners finds
 * the winning row of each slot field and k_republish_runtime lets the winners write again.  The
 * "External id" was resolved before this pass, so the joined row and its length are produced here
 * too.  The slots are remembered per row for those two passes. */
__device__ __forceinline__ bool runtime_rows_share_slots(const Scalars* sc) {
  /* ids beyond 31 bits may coincide after narrowing without sharing a slot of the full table */
  const KeyRange r = sc->plan.range[KTJ_TBL_FULL];
  return sc->runtime_ids_repeat != 0 || (r.lo <= r.hi && r.hi >= 0x80000000ULL);
}
/* Sets the slot's bit in a bitmap and tells whether it was set before.  All lanes of the wavefront
 * call it (active = the lane has a slot).  Rows that arrive in id order put up to 32 neighbouring
 * lanes on one word, so the lanes are grouped by word (up to BITMAP_GROUPS groups, found with
 * ballots; 64 consecutive slots lie in two or three words) and the lowest lane of each group sets
 * all of its group's bits in one atomic; the groups' atomics leave in a single instruction.  Lanes
 * beyond the last group set their own bit.  Two lanes of the wavefront with the same slot are
 * reported as "set before" for every lane of their group (callers only ask whether any slot is
 * shared). */
#define BITMAP_GROUPS 4
__device__ __forceinline__ uint32_t wave_or_u32(uint32_t v) {
  for (int o = 32; o > 0; o >>= 1) v |= (uint32_t)__shfl_xor((int)v, o);
  return v;
}
__device__ __forceinline__ bool bitmap_test_and_set(uint32_t* bitmap, uint32_t slot, bool active) {
  const uint32_t word = slot >> 5, bit = active ? 1u << (slot & 31u) : 0u;
  uint64_t todo = __ballot(active);
  if (!todo) return false;
  int leader = (int)lane_id();   /* lanes outside every group lead themselves */
  uint32_t bits = bit;
  bool twice = false;
  for (int g = 0; g < BITMAP_GROUPS && todo; ++g) {
    const int l = __ffsll((unsigned long long)todo) - 1;
    const uint32_t w = (uint32_t)__shfl((int)word, l);
    const bool in = ((todo >> lane_id()) & 1ull) != 0 && word == w;
    const uint64_t m = __ballot(in);
    const uint32_t all = wave_or_u32(in ? bit : 0u);
    if (in) { leader = l; bits = all; twice = (uint32_t)__popc(all) != (uint32_t)__popcll(m); }
    todo &= ~m;
  }
  uint32_t old = 0;
  if (active && leader == (int)lane_id()) old = atomicOr(&bitmap[word], bits);
  old = (uint32_t)__shfl((int)old, leader);
  return active && (twice || (old & bit) != 0);
}
#define JOIN_ROWS 4u
#ifndef KX_JOIN_ATTR
#define KX_JOIN_ATTR
#endif
template <bool TEXT>
__global__ void KX_JOIN_ATTR k_join_runtime(const ktj_runtime_rec* r, uint64_t n, Columns c, uint64_t first_runtime, ApiTable api, Table tf_planned,
                               FullCols fc, Table tn_planned, NarrowCols nc, uint32_t* slot_f, uint32_t* slot_n, ClockDev clk, EmitCtx ctx, Rows rows,
                               uint32_t* len, Scalars* sc, int rounds) {
  const TableView tf = view(tf_planned), tn = view(tn_planned);
  RowStats rs;
  uint32_t n_linked = 0;
  bool any_carries_stream = false, any_repeats = false;
  /* a workgroup takes `rounds` consecutive groups of blockDim.x rows: the per-workgroup counters
   * at the end (one atomic each on a hot address) are paid once for all of them */
  static_assert(sizeof(MatRow) == sizeof(ktj_runtime_rec), "the staging area holds the records, then the joined rows");
  __shared__ uint4 stage[KTJ_BLOCK * sizeof(typename RowOf<TEXT>::T) / 16];
  for (int round = 0; round < rounds; ++round) {
    const uint64_t base = ((uint64_t)blockIdx.x * rounds + round) * blockDim.x;
    if (base >= n) break;
    const uint32_t cnt = (uint32_t)(n - base < blockDim.x ? n - base : blockDim.x);
    const uint64_t i = base + threadIdx.x;
    bool carries_stream = false;
    uint32_t sf = KTJ_NOSLOT;
    MatRow m;
    /* everything the row reads from its own record and columns is requested up front, so that the
     * table accesses below (each a round trip of its own) overlap with it */
    const uint64_t a = first_runtime + (i < n ? i : 0);
    const uint32_t meta_of = load_once(&c.meta[a]);
    const int64_t ts_of = load_once(&c.ts[a]);
    __syncthreads(); /* the previous round's rows have left the staging area */
    rows_global_to_lds(r + base, cnt, stage);
    __syncthreads();
    /* the lane's record stays in LDS and is read field by field; the joined row takes its place */
    uint4* my_slot = &stage[threadIdx.x * (sizeof(ktj_runtime_rec) / 16)];
    const ktj_runtime_rec& rec = *reinterpret_cast<const ktj_runtime_rec*>(my_slot);
    uint64_t id = 0;
    uint32_t meta = 0;
    int64_t ts = 0, dur = 0;
    if (i < n) {
      id = rec.id;
      meta = meta_of;
      ts = ts_of;
      sf = slot_insert(tf, id);
    }
    const uint32_t kind = (meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT;
    const bool valid = (meta & KTJ_M_VALID) != 0;
    const bool publishes = valid && kind != KTJ_RT_DEFAULT;
    /* every slot that carries an external id exists already (k_build_extcorr ran before) */
    uint32_t sn = KTJ_NOSLOT;
    if (i < n) sn = publishes ? slot_insert(tn, narrow_corr_key(id)) : slot_find(tn, narrow_corr_key(id));
    int32_t ext = 0;
    uint32_t np_info = 0;
    if (sn != KTJ_NOSLOT) {
      const NarrowHead head = tn.no_heads ? NarrowHead{nc.pay[sn].ext_val, nc.pay[sn].info} : nc.head[sn];
      ext = head.ext_val; np_info = head.info;
    }
    const bool repeats = bitmap_test_and_set(fc.has_runtime, sf, sf != KTJ_NOSLOT);
    if (i < n) {
      carries_stream = (meta & KTJ_M_HAS_STREAM) != 0;
      store_once(&slot_f[i], sf);
      if (sf == KTJ_NOSLOT) flag_error(sc, KTJ_DEVERR_TABLE_FULL);
      else {
        FullPay fp;
        fp.first_ts = ts;
        fp.stream = 0;
        if (carries_stream) fp.stream = rec.kind == KTJ_RT_KERNEL ? rec.u.kernel.stream : rec.u.copy.stream;
        fc.pay[sf] = fp;
      }
      if (publishes && sn == KTJ_NOSLOT) flag_error(sc, KTJ_DEVERR_TABLE_FULL);
      if (sn != KTJ_NOSLOT && (publishes || !tn.no_heads)) { /* (with heads there is nothing there that another row's would be) */
        NarrowPay np;
        np.ext_val = ext; np.info = np_info & ~KTJ_NP_KIND_MASK;
        np.pay[0] = np.pay[1] = np.pay[2] = 0;
        if (publishes) {
          if (kind == KTJ_RT_KERNEL) pack_grid(rec, np.pay);
          else np.pay[0] = rec.kind == KTJ_RT_COPY ? rec.u.copy.size : rec.u.malloc_.size;
          np.info |= kind == KTJ_RT_KERNEL ? KTJ_DL_HAS_GRID : KTJ_DL_HAS_SIZE;
        }
        typedef unsigned int v4u __attribute__((ext_vector_type(4)));
        v4u* const dst = reinterpret_cast<v4u*>(&nc.pay[sn]);
        dst[0] = reinterpret_cast<const v4u*>(&np)[0];
        dst[1] = reinterpret_cast<const v4u*>(&np)[1];
      }
      store_once(&slot_n[i], sn);
      if ((np_info & KTJ_NP_LINKED) && valid) ++n_linked;
      if (c.all) store_once(&c.ext[a], ext);
      dur = duration_from(clk, clk.runtime_mode, ts, rec.end);
      const bool known = rec.cid < api.n_cids;
      const uint32_t name = known ? api.cid_name_ids[rec.cid] : KTJ_NONE;
      const bool fstart = known && ((api.flow_start_bits[rec.cid >> 5] >> (rec.cid & 31u)) & 1u);
      if (TEXT) m = mat_runtime(rec, ts, dur, valid, ext, name, fstart, rec.cid == api.malloc_cid);
      else {
        MatRow* in_place = reinterpret_cast<MatRow*>(my_slot);
        *in_place = mat_runtime(rec, ts, dur, valid, ext, name, fstart, rec.cid == api.malloc_cid);
        store_once(&len[a], row_length(*in_place, ctx, sc));
        count_row_stats(*in_place, ctx, &rs);
      }
    }
    if (TEXT) { /* (its rows are longer than the records: every lane has taken its own before any is put down) */
      __syncthreads();
      if (i < n) {
        count_row_stats(m, ctx, &rs);
        store_once(&len[a], stage_row<true>(m, ctx, rows, 0, sc, stage));
      }
    }
    __syncthreads(); /* the joined rows go out the way the records came in */
    rows_lds_to_global(static_cast<typename RowOf<TEXT>::T*>(rows.p) + first_runtime + base, cnt, stage);
    any_carries_stream |= carries_stream;
    any_repeats |= repeats;
  }
  /* one store per workgroup at most: every lane storing the same flag would queue up in L2 */
  const int any_stream = __syncthreads_or(any_carries_stream ? 1 : 0);
  const int any_repeat = __syncthreads_or(any_repeats ? 1 : 0);
  if (threadIdx.x == 0) {
    if (any_stream) sc->have_stream_src = 1;
    if (any_repeat) sc->runtime_ids_repeat = 1;
  }
  flush_row_stats(rs, sc);
  block_add(sc, KTJ_CNT_LINKED, n_linked);
}
/* Only when runtime rows share slots: which row of a slot the device rows take each value from
 * (the last row that carries a stream; the last in-window kernel launch; the last in-window copy
 * or allocation), by atomicMax over row indices.  k_republish_runtime reads the winners. */
__global__ void k_runtime_winners(uint64_t n, Columns c, uint64_t first, FullCols fc, NarrowCols nc, const uint32_t* slot_f,
                                  const uint32_t* slot_n, const Scalars* sc) {
  if (!runtime_rows_share_slots(sc)) return;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t meta = c.meta[first + i];
    const uint32_t kind = (meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT;
    const uint32_t sf = slot_f[i], sn = slot_n[i];
    if (sf != KTJ_NOSLOT) {
      atomicMin(&fc.first[sf], (uint32_t)(first + i));
      if (meta & KTJ_M_HAS_STREAM) atomicMax(&fc.stream_src[sf], (uint32_t)i + 1u);
    }
    if (sn != KTJ_NOSLOT && (meta & KTJ_M_VALID) && kind != KTJ_RT_DEFAULT)
      atomicMax(kind == KTJ_RT_KERNEL ? &nc.kern_src[sn] : &nc.copy_src[sn], (uint32_t)i + 1u);
  }
}
/* Only when runtime rows share slots: the row that won a slot field writes the payload again, and
 * every row is checked against the first row of its id (checkTimestampOrder with the roles
 * swapped).  Where no two runtime rows share a slot each row is the first of its id and what it
 * wrote in k_join_runtime stands. */
__global__ void k_republish_runtime(const ktj_runtime_rec* r, uint64_t n, Columns c, uint64_t first, FullCols fc, NarrowCols nc,
                                    const uint32_t* slot_f, const uint32_t* slot_n, Scalars* sc) {
  if (!runtime_rows_share_slots(sc)) return;
  uint32_t n_bad = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t a = first + i;
    const ktj_runtime_rec rec = r[i];
    const int64_t ts = c.ts[a];
    const uint32_t sf = slot_f[i], sn = slot_n[i];
    if (sf != KTJ_NOSLOT) {
      const uint64_t f = fc.first[sf];
      if (f == a) fc.pay[sf].first_ts = ts;
      else if (f != 0xFFFFFFFFull) { /* an earlier runtime row has this id */
        const int64_t t1 = c.ts[f];
        if (ts != 0 && t1 > ts) ++n_bad;
      }
      const uint32_t stream_src = fc.stream_src[sf];
      if (stream_src == (uint32_t)i + 1u)
        fc.pay[sf].stream = rec.kind == KTJ_RT_KERNEL ? rec.u.kernel.stream : rec.u.copy.stream;
      else if (stream_src == 0) fc.pay[sf].stream = 0; /* no row of this id carries one */
    }
    if (sn != KTJ_NOSLOT) {
      NarrowPay* np = &nc.pay[sn];
      const uint32_t copy_src = nc.copy_src[sn]; /* final: the pass above has ended */
      if (copy_src == (uint32_t)i + 1u) {
        np->pay[0] = rec.kind == KTJ_RT_COPY ? rec.u.copy.size : rec.u.malloc_.size;
        np->info = (np->info & ~KTJ_NP_KIND_MASK) | KTJ_DL_HAS_SIZE;
      } else if (copy_src == 0 && nc.kern_src[sn] == (uint32_t)i + 1u) {
        pack_grid(rec, np->pay);
        np->info = (np->info & ~KTJ_NP_KIND_MASK) | KTJ_DL_HAS_GRID;
      }
    }
  }
  block_add(sc, KTJ_CNT_OUT_OF_ORDER, n_bad);
}
template <bool TEXT>
__device__ __forceinline__ void mat_device_block(const ktj_device_rec* d, uint64_t n, const Columns& c, uint64_t first, const Links& link,
                                                 const ClockDev& clk, const EmitCtx& ctx, Rows rows, uint32_t* len, Scalars* sc, uint64_t block,
                                                 uint64_t blocks, uint4* stage) {
  RowStats rs;
  /* which values of its link a row has is asked for a group ahead */
  const auto info_at = [&](uint64_t i) { return load_once(&link.info[i < n ? i : n - 1]); };
  uint32_t next_info = info_at(block * KTJ_BLOCK + threadIdx.x);
  for (uint64_t base = block * KTJ_BLOCK; base < n; base += blocks * KTJ_BLOCK) {
    const uint32_t cnt = (uint32_t)(n - base < KTJ_BLOCK ? n - base : KTJ_BLOCK);
    const uint32_t info = next_info;
    next_info = info_at(base + blocks * KTJ_BLOCK + threadIdx.x);
    const uint64_t i = base + (threadIdx.x < cnt ? threadIdx.x : 0u), a = first + i;
    const bool active = threadIdx.x < cnt;
    MatRow m;
    uint64_t p0 = 0, p1 = 0, p2 = 0; /* (the columns and the link are on their way with the records) */
    if (info & KTJ_NP_KIND_MASK) p0 = load_once(&link.p[0][i]);
    if (info & KTJ_DL_HAS_GRID) { p1 = load_once(&link.p[1][i]); p2 = load_once(&link.p[2][i]); }
    const int64_t ts = load_once(&c.ts[a]), res = load_once(&c.res[a]);
    const uint32_t meta = load_once(&c.meta[a]);
    const int32_t ext = load_once(&c.ext[a]);
    __syncthreads(); /* the previous round's rows have left the staging area */
    rows_global_to_lds(d + base, cnt, stage);
    __syncthreads();
    if (active) {
      const ktj_device_rec rec = row_from_lds<ktj_device_rec>(stage);
      m = mat_device_v(rec, ts, duration_from(clk, clk.device_mode, ts, rec.end), res,
                       (meta & KTJ_M_VALID) != 0, ext,
                       (info & KTJ_DL_HAS_GRID) != 0, p0, p1, p2, (info & KTJ_DL_HAS_SIZE) != 0, p0, info >> KTJ_NP_COLL_SHIFT);
      count_row_stats(m, ctx, &rs);
    }
    __syncthreads(); /* every lane has taken its record */
    if (active) store_once(&len[a], stage_row<TEXT>(m, ctx, rows, 0, sc, stage));
    __syncthreads();
    rows_lds_to_global(static_cast<typename RowOf<TEXT>::T*>(rows.p) + first + base, cnt, stage);
  }
  flush_row_stats(rs, sc);
}
/* joined rows and lengths of the generic records (first workgroups) and of the device records (the others);
 * the runtime rows' are made in k_join_runtime.  Where there are both classes one launch makes them, as neither fills the GPU to its
 * end (400 000 rows 34 us, two launches 47; a million 72 and 78; 2 million 140 and 150; 6 million 405 and 409; 12 million, of them 2 million
 * generic, 698 and 701; 11 million and 20 000 generic 620 and 627). */
template <bool GENERIC, bool DEVICE, bool TEXT>
__global__ void __launch_bounds__(KTJ_BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
k_mat_rows(const ktj_generic_rec* g, uint64_t ng, uint64_t first_generic, const uint32_t* sync_first, uint32_t generic_blocks, const ktj_device_rec* d,
           uint64_t nd, Columns c, uint64_t first_device, Links link, ClockDev clk, EmitCtx ctx, Rows rows, uint32_t* len, Scalars* sc, int clock) {
  static_assert(sizeof(MatRow) >= sizeof(ktj_generic_rec) && sizeof(MatRow) >= sizeof(ktj_device_rec), "the staging area holds the records, then the joined rows");
  __shared__ uint4 stage[KTJ_BLOCK * sizeof(typename RowOf<TEXT>::T) / 16];
  if (blockIdx.x == 0 && threadIdx.x == 0 && clock) stage_clock(sc, KTJ_CLOCK_SIZE);
  /* The pass ends, or the host takes another way from the sort on.  All wavefronts of a workgroup must see the same
   * here, as they move records for each other: the one bit that this launch sets does not count.  Nor does a sort that comes again:
   * rows lie in order of arrival, and are not made again. */
  if (sc->error & ~(KTJ_DEVERR_RECORD_TOO_LONG | KTJ_DEVERR_UNSORTED)) return;
  if (GENERIC && (!DEVICE || blockIdx.x < generic_blocks))
    mat_generic_block<TEXT>(g, ng, first_generic, ctx, sync_first, rows, len, sc, blockIdx.x, generic_blocks, stage);
  else if (DEVICE)
    mat_device_block<TEXT>(d, nd, c, first_device, link, clk, ctx, rows, len, sc, blockIdx.x - generic_blocks, gridDim.x - generic_blocks, stage);
}
/* The sort's last launch (first workgroups) and the rows of either class in one: neither needs anything of the other, and the former is a
 * chain of loads and LDS accesses that leaves the memory idle, with fewer workgroups than the GPU holds up to a few million rows.  Passes,
 * one after the other and now, us: 30 000 records 172 -> 168 (no more than runs differ), 180 000 220 -> 213, 733 000 413 -> 407, 3 million 985 -> 972; 11 and 22 million, where both are
 * at the memory's rate by themselves, 3153 and 3146, 6838 and 6841.  CPU ops or kernels alone: 20 000 records 140 -> 138, 150 000 220 -> 215, a million
 * 771 -> 766, 3 million 2058 -> 2048. */
template <int ITEMS>
__global__ void __launch_bounds__(KTJ_BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
k_finish_and_rows(const uint64_t* buf_a, const uint64_t* buf_b, uint32_t* perm, uint64_t n, uint32_t idx_bits, uint32_t finish_blocks, const ktj_generic_rec* g,
                  uint64_t ng, uint32_t generic_blocks, const ktj_device_rec* d, uint64_t nd, Columns c, uint64_t first_device, Links link, ClockDev clk,
                  EmitCtx ctx, Rows rows, uint32_t* len, Scalars* sc) {
  using Lds = FinishLds<KTJ_BLOCK, ITEMS>;
  __shared__ union { uint4 stage[KTJ_BLOCK * sizeof(typename RowOf<true>::T) / 16]; Lds finish; } lds;
  if (blockIdx.x == 0 && threadIdx.x == 0) stage_clock(sc, KTJ_CLOCK_SIZE);
  constexpr unsigned int own_bits = KTJ_DEVERR_RECORD_TOO_LONG | KTJ_DEVERR_UNSORTED;
  if (blockIdx.x < finish_blocks) {
    finish_tile<KTJ_BLOCK, ITEMS>(buf_a, buf_b, perm, n, idx_bits, sc, own_bits, blockIdx.x, lds.finish);
    return;
  }
  if (sc->error & ~own_bits) return; /* (as in k_mat_rows) */
  const uint32_t block = blockIdx.x - finish_blocks;
  if (block < generic_blocks) mat_generic_block<true>(g, ng, 0, ctx, nullptr, rows, len, sc, block, generic_blocks, lds.stage);
  else mat_device_block<true>(d, nd, c, first_device, link, clk, ctx, rows, len, sc, block - generic_blocks, gridDim.x - finish_blocks - generic_blocks, lds.stage);
}
/* Collective metadata: the first activity, in emission order, that prints each entry, per
 * backend (first[2k] nccl, first[2k + 1] hccl).  The host replays appendCollectiveMetadata's
 * bookkeeping (output_json.cpp:799-835) over these.  Runs only for traces that carry any. */
__global__ void k_collective_first(const MatRow* mat, const uint32_t* perm, uint64_t n_rows, uint32_t n_coll, uint32_t* first) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_rows) return;
  const MatRow* m = &mat[perm[i]];
  const uint32_t meta = m->meta;
  const uint32_t cls = (meta & KTJ_M_CLASS_MASK) >> KTJ_M_CLASS_SHIFT;
  uint32_t k = 0;
  if (cls == KTJ_CLASS_GENERIC) k = (uint32_t)m->p[1];
  else if (cls == KTJ_CLASS_DEVICE && (meta & KTJ_M_TYPE_MASK) == KTJ_TYPE_CONCURRENT_KERNEL) k = (uint32_t)m->p[4];
  if (k == 0 || k > n_coll) return;
  const uint32_t hccl = cls == KTJ_CLASS_GENERIC && (meta & KTJ_M_TYPE_MASK) == KTJ_TYPE_MTIA_CCP_EVENTS ? 1u : 0u;
  atomicMin(&first[2u * (k - 1u) + hccl], (uint32_t)i);
}
hipError_t collective_first(const MatRow* mat, const uint32_t* perm, uint64_t n_rows, uint32_t n_coll, uint32_t* first,
                            hipStream_t st) {
  hipError_t e = fill_u32(first, 0xFFFFFFFFu, 2ull * n_coll, st);
  if (e != hipSuccess || n_rows == 0) return e;
  hipLaunchKernelGGL(k_collective_first, dim3(grid_for(n_rows, KTJ_BLOCK)), dim3(KTJ_BLOCK), 0, st, mat, perm, n_rows, n_coll,
                     first);
  return KTJ_LAUNCH_CHECK();
}
/* lengths and tail kinds in emission order (the size pass leaves both in one word per arrival index), and
 * the lengths' sum per tile of 2048 for the scan that follows */
__global__ void __launch_bounds__(KTJ_BLOCK)
k_gather_len(const uint32_t* perm, const uint32_t* len, uint64_t n, uint32_t* len_sorted, uint8_t* kind_sorted, uint64_t* sums, uint32_t* left, Scalars* sc) {
  __shared__ uint64_t wave_tot[KTJ_BLOCK >> 6];
  __shared__ uint32_t n_left, left_at;
  if (blockIdx.x == 0 && threadIdx.x == 0) stage_clock(sc, KTJ_CLOCK_SCAN);
  if (sc->error != 0) return; /* there may be no order */
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + threadIdx.x;
  uint32_t v[SCAN_ITEMS] = {};
  if (n != 0) {
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) { const uint64_t i = base + (uint64_t)k * KTJ_BLOCK; v[k] = load_once(&perm[i < n ? i : n - 1]); }
    /* (each without a condition: under one it is waited for before the next; 3 million rows 41 us, now 31, 22 million 87 and 77) */
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) v[k] = len[v[k]];
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) v[k] = base + (uint64_t)k * KTJ_BLOCK < n ? v[k] : 0u;
  }
  uint32_t n_mine = 0;
  unsigned long long sum = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const uint64_t i = base + (uint64_t)k * KTJ_BLOCK;
    n_mine += (v[k] >> 30) == KTJ_KIND_LEFT ? 1u : 0u;
    if (i < n) { len_sorted[i] = v[k] & 0x3FFFFFFFu; kind_sorted[i] = (uint8_t)(v[k] >> 30); }
    sum += v[k] & 0x3FFFFFFFu;
  }
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
  if (lane_id() == 0) wave_tot[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t s = 0;
    for (uint32_t k = 0; k < (KTJ_BLOCK >> 6); ++k) s += wave_tot[k];
    sums[blockIdx.x] = s;
  }
  /* the places of the rows that are left to emit_direct, in no particular order: one atomic per tile that has any */
  if (!__syncthreads_or(n_mine != 0 ? 1 : 0)) return;
  if (threadIdx.x == 0) n_left = 0;
  __syncthreads();
  uint32_t at = n_mine ? atomicAdd(&n_left, n_mine) : 0u;
  __syncthreads();
  if (threadIdx.x == 0) left_at = atomicAdd(&sc->n_left, n_left);
  __syncthreads();
  at += left_at;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k)
    if ((v[k] >> 30) == KTJ_KIND_LEFT) left[at++] = (uint32_t)(base + (uint64_t)k * KTJ_BLOCK);
}

hipError_t mat_rows(const ktj_generic_rec* g, uint64_t ng, uint64_t first_generic, const uint32_t* sync_first, const ktj_device_rec* d, uint64_t nd,
                    Columns c, uint64_t first_device, Links link, const ClockDev& clk, EmitCtx ctx, Rows rows, uint32_t* len, Scalars* sc, hipStream_t st) {
  const unsigned gb = grid_stride_for(ng, KTJ_BLOCK), db = grid_stride_for(nd, KTJ_BLOCK);
  auto launch = [&](auto kernel, unsigned g_blocks, unsigned d_blocks, bool clock) {
    hipLaunchKernelGGL(kernel, dim3(g_blocks + d_blocks), dim3(KTJ_BLOCK), 0, st, g, ng, first_generic, sync_first, g_blocks, d, nd, c, first_device,
                       link, clk, ctx, rows, len, sc, clock ? 1 : 0);
  };
  const bool clock = first_generic == 0;
  if (gb && db) {
    if (rows.schemas) launch(k_mat_rows<true, true, true>, gb, db, clock); else launch(k_mat_rows<true, true, false>, gb, db, clock);
  } else {
    if (gb) { if (rows.schemas) launch(k_mat_rows<true, false, true>, gb, 0, clock); else launch(k_mat_rows<true, false, false>, gb, 0, clock); }
    if (db) { if (rows.schemas) launch(k_mat_rows<false, true, true>, 0, db, clock && !gb); else launch(k_mat_rows<false, true, false>, 0, db, clock && !gb); }
  }
  return KTJ_LAUNCH_CHECK();
}

static bool finish_and_rows(const uint64_t* buf_a, const uint64_t* buf_b, uint32_t* perm, uint64_t n, uint32_t idx_bits, uint64_t tile, Scalars* sc,
                            RowsJob* job, hipStream_t st) {
  if (!job || job->ng + job->nd == 0 || !job->rows.schemas) return false;
  const unsigned fb = (unsigned)((n + tile - 1) / tile), gb = job->ng ? grid_stride_for(job->ng, KTJ_BLOCK) : 0u, db = job->nd ? grid_stride_for(job->nd, KTJ_BLOCK) : 0u;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(fb + gb + db), dim3(KTJ_BLOCK), 0, st, buf_a, buf_b, perm, n, idx_bits, fb, job->g, job->ng, gb, job->d, job->nd, job->c,
                       job->first_device, job->link, job->clk, job->ctx, job->rows, job->len, sc);
  };
  if (tile == 1u * KTJ_BLOCK) launch(k_finish_and_rows<1>);
  else if (tile == 4u * KTJ_BLOCK) launch(k_finish_and_rows<4>);
  else launch(k_finish_and_rows<16>);
  job->made = true;
  return true;
}

hipError_t join_runtime_rows(const ktj_runtime_rec* r, uint64_t n, Columns c, uint64_t first, ApiTable api, Table tf, FullCols fc,
                             Table tn, NarrowCols nc, uint32_t* slot_f, uint32_t* slot_n, const ClockDev& clk, EmitCtx ctx, Rows rows,
                             uint32_t* len, Scalars* sc, hipStream_t st) {
  if (n == 0) return hipSuccess;
  /* As many groups per workgroup as let all workgroups run at a time (four per CU, by their registers and LDS), as far as JOIN_ROWS do:
   * with fewer the last ones run alone, with more CUs stand idle.  Behind that two, so that the last workgroups, which do not fill the
   * GPU, are short ones.  1 / 2 / 3 / 4 groups, us: 333 000 rows 54 / 48 / 56 / 65, 500 000 50 / 48 / 54 / 63, 600 000 74 / 84 / 75 / 79,
   * a million 103 / 106 / 120 / 107; 1.5 million 190 / 190 / 187 / 218, 2.5 million 302 / 301 / 324 / 332, 4 million 468 / 472 / 482 / 477,
   * 10 million 1169 / 1151 / 1138 / 1148. */
  const uint64_t groups = grid_for(n, KTJ_BLOCK), at_once = 1024u;
  const int rounds = groups > at_once * JOIN_ROWS ? 2 : (int)((groups + at_once - 1u) / at_once);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid_for(n, KTJ_BLOCK * rounds)), dim3(KTJ_BLOCK), 0, st, r, n, c, first, api, tf, fc, tn, nc,
                       slot_f, slot_n, clk, ctx, rows, len, sc, rounds);
  };
  if (rows.schemas) launch(k_join_runtime<true>); else launch(k_join_runtime<false>);
  return KTJ_LAUNCH_CHECK();
}
hipError_t republish_runtime_rows(const ktj_runtime_rec* r, uint64_t n, Columns c, uint64_t first, FullCols fc, NarrowCols nc,
                                  const uint32_t* slot_f, const uint32_t* slot_n, Scalars* sc, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_runtime_winners, dim3(grid_rarely(n)), dim3(KTJ_BLOCK), 0, st, n, c, first, fc, nc, slot_f,
                     slot_n, (const Scalars*)sc);
  hipLaunchKernelGGL(k_republish_runtime, dim3(grid_rarely(n)), dim3(KTJ_BLOCK), 0, st, r, n, c, first, fc, nc,
                     slot_f, slot_n, sc);
  return KTJ_LAUNCH_CHECK();
}
/* The activities' offsets from their lengths and the tiles' sums.  Few tiles: every workgroup adds up the
 * sums before its own (OFFS_DIRECT_TILES of them are 16 KB from the L2), many: k_scan_of_sums has run.
 * The workgroups behind the tiles' know the total: with a document to prepare (out != null) the first of them
 * puts the footer text behind the activities and hands the scalars to the host, and the others put the header,
 * 4 KiB each (all of that takes some microseconds over the host link, which the offsets need not wait for; 40 KB
 * of header by one workgroup took 20 us). */
#define PREFIX_PIECE 4096u
#define OFFS_DIRECT_TILES 2048u
__device__ void publish_scalars(Scalars* sc, Scalars* h_sc, bool document_fits);
__global__ void __launch_bounds__(KTJ_BLOCK)
k_offsets(const uint32_t* len, uint64_t n, const uint64_t* sums, uint32_t n_tiles, uint64_t* offs, Scalars* sc, DocText T) {
  __shared__ uint64_t lds_wave[SCAN_MAX_WAVES];
  __shared__ uint64_t s_before;
  const bool ok = sc->error == 0; /* otherwise there are no lengths: only the host is told */
  const uint32_t tile = blockIdx.x < n_tiles ? blockIdx.x : n_tiles; /* behind the tiles: all of them */
  uint64_t before = 0;
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
  uint32_t v[SCAN_ITEMS];
  if (ok && blockIdx.x < n_tiles) scan_load_items(len, n, base, v);
  if (n_tiles <= OFFS_DIRECT_TILES) {
    unsigned long long s = 0;
    if (ok && tile)
      for (uint32_t k0 = threadIdx.x; k0 < tile; k0 += 4u * KTJ_BLOCK) {
        uint64_t x[4];
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) { const uint32_t k = k0 + j * KTJ_BLOCK; x[j] = sums[k < tile ? k : tile - 1u]; }
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) s += k0 + j * KTJ_BLOCK < tile ? x[j] : 0u;
      }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane_id() == 0) lds_wave[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) { uint64_t b = 0; for (uint32_t k = 0; k < (KTJ_BLOCK >> 6); ++k) b += lds_wave[k]; s_before = b; }
    __syncthreads();
    before = s_before;
  } else before = ok ? sums[tile] : 0;
  if (blockIdx.x >= n_tiles) {
    /* no text where the document does not fit or there is none: the buffer stays as it was */
    const bool fits = ok && T.n_prefix + before + T.n_suffix + 64u <= T.out_cap;
    if (blockIdx.x > n_tiles) {
      const uint64_t at = (uint64_t)(blockIdx.x - n_tiles - 1u) * PREFIX_PIECE, left = T.n_prefix - at;
      if (fits) put_text_block(T.prefix + at, T.out + at, left < PREFIX_PIECE ? left : PREFIX_PIECE);
      return;
    }
    if (threadIdx.x == 0) offs[n] = before;
    if (!T.out) return;
    publish_scalars(sc, T.h_sc, fits);
    if (threadIdx.x == 0) *T.h_total = before;
    if (fits) put_text_block(T.suffix, T.out + T.n_prefix + before, T.n_suffix);
    return;
  }
  if (!ok) return;
  uint64_t s = 0;
  for (int k = 0; k < SCAN_ITEMS; ++k) s += v[k];
  uint64_t tot;
  uint64_t ex = block_exclusive_scan_u64(s, lds_wave, &tot) + before;
  if (base + SCAN_ITEMS <= n) { /* the lane's run as 16-byte stores (the offsets are a 16-byte aligned device buffer) */
    typedef unsigned long long v2u64 __attribute__((ext_vector_type(2)));
    v2u64* dst = reinterpret_cast<v2u64*>(offs + base);
#pragma unroll
    for (int q = 0; q < SCAN_ITEMS / 2; ++q) { v2u64 x; x.x = ex; ex += v[2 * q]; x.y = ex; ex += v[2 * q + 1]; dst[q] = x; }
  } else {
    for (int k = 0; k < SCAN_ITEMS; ++k) { if (base + k < n) offs[base + k] = ex; ex += v[k]; }
  }
}
uint64_t offsets_tmp_elems(uint64_t n) { return (n + SCAN_TILE - 1) / SCAN_TILE + 2; }
hipError_t gather_offsets(const uint32_t* perm, const uint32_t* len, uint64_t n, uint32_t* len_sorted, uint8_t* kind_sorted, uint64_t* sums,
                          uint64_t* offs, uint32_t* left, Scalars* sc, const DocText& text, hipStream_t st) {
  const uint64_t tiles = n ? (n + SCAN_TILE - 1) / SCAN_TILE : 1;
  hipLaunchKernelGGL(k_gather_len, dim3((unsigned)tiles), dim3(KTJ_BLOCK), 0, st, perm, len, n, len_sorted, kind_sorted, sums, left, sc);
  if (tiles > OFFS_DIRECT_TILES) hipLaunchKernelGGL(k_scan_of_sums, dim3(1), dim3(1024), 0, st, sums, tiles);
  const uint64_t prefix_blocks = text.out ? (text.n_prefix + PREFIX_PIECE - 1) / PREFIX_PIECE : 0;
  hipLaunchKernelGGL(k_offsets, dim3((unsigned)(tiles + 1u + prefix_blocks)), dim3(KTJ_BLOCK), 0, st, (const uint32_t*)len_sorted, n, (const uint64_t*)sums,
                     (uint32_t)tiles, offs, sc, text);
  return KTJ_LAUNCH_CHECK();
}

/* What the host needs during a pass goes straight into its pinned memory, and the text it made
 * (header, infos, footer) comes straight out of it: one small kernel each instead of one copy
 * engine transfer per value. */
__device__ void publish_scalars(Scalars* sc, Scalars* h_sc, bool document_fits) { /* by one workgroup */
  /* the sharded counters: their sums so far into the fields the host reads (written, not added: a pass
   * may publish twice) */
  static_assert(KTJ_COUNTER_SHARDS == 64, "a lane per copy");
  if (threadIdx.x < 64) {
    unsigned long long sum[KTJ_CNT_COUNT];
    for (int k = 0; k < KTJ_CNT_COUNT; ++k) sum[k] = sc->shard[threadIdx.x][k];
    for (int k = 0; k < KTJ_CNT_COUNT; ++k)
      for (int o = 32; o > 0; o >>= 1) sum[k] += __shfl_xor(sum[k], o);
    if (threadIdx.x == 0) {
      sc->out_of_range = sum[KTJ_CNT_OUT_OF_RANGE]; sc->out_of_order = sum[KTJ_CNT_OUT_OF_ORDER];
      sc->n_flow = sum[KTJ_CNT_FLOW]; sc->n_linked = sum[KTJ_CNT_LINKED]; sc->n_blank_names = sum[KTJ_CNT_BLANK_NAMES];
      sc->n_valid = sum[KTJ_CNT_VALID]; sc->n_sync_typed = sum[KTJ_CNT_SYNC_TYPED];
      sc->emit_rows = sc->error == 0 && document_fits ? sum[KTJ_CNT_VALID] : 0;
    }
  }
  if (threadIdx.x == 0) stage_clock(sc, KTJ_CLOCK_EMIT);
  __syncthreads();
  constexpr uint32_t head_words = (uint32_t)(offsetof(Scalars, shard) / 4);
  const uint32_t* src = reinterpret_cast<const uint32_t*>(sc);
  uint32_t* dst = reinterpret_cast<uint32_t*>(h_sc);
  for (uint32_t k = threadIdx.x; k < head_words; k += blockDim.x) dst[k] = src[k];
}
__global__ void k_publish(Scalars* sc, const uint64_t* total, const uint32_t* list, uint32_t n_list, Scalars* h_sc,
                          uint64_t* h_total, uint32_t* h_list) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  if (blockIdx.x == 0) publish_scalars(sc, h_sc, true);
  for (uint32_t k = t; k < n_list; k += stride) h_list[k] = list[k];
  if (t == 0 && total != nullptr) *h_total = *total;
  __threadfence_system();
}
hipError_t publish(Scalars* sc, const uint64_t* total, const uint32_t* list, uint32_t n_list, Scalars* h_sc,
                   uint64_t* h_total, uint32_t* h_list, hipStream_t st) {
  static_assert(KTJ_CNT_COUNT == 7, "publish_scalars names every sharded counter");
  hipLaunchKernelGGL(k_publish, dim3(n_list > 4096 ? 16 : 1), dim3(KTJ_BLOCK), 0, st, sc, total, list, n_list, h_sc, h_total, h_list);
  return KTJ_LAUNCH_CHECK();
}
/* two pieces of text, each to its place; source and destination of a piece agree modulo 16 */
__global__ void k_put_text(const char* src_a, char* dst_a, uint64_t n_a, const char* src_b, char* dst_b, uint64_t n_b) {
  const char* src = blockIdx.y ? src_b : src_a;
  char* dst = blockIdx.y ? dst_b : dst_a;
  const uint64_t n = blockIdx.y ? n_b : n_a;
  uint64_t head = (16u - (uint32_t)((uintptr_t)dst & 15u)) & 15u;
  if (head > n) head = n;
  const uint64_t body = (n - head) >> 4, tail = (n - head) & 15u;
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
  if (t < head) dst[t] = src[t];
  const uint4* sv = reinterpret_cast<const uint4*>(src + head);
  uint4* dv = reinterpret_cast<uint4*>(dst + head);
  for (uint64_t k = t; k < body; k += stride) dv[k] = sv[k];
  if (t < tail) dst[head + body * 16u + t] = src[head + body * 16u + t];
}
hipError_t put_text(const char* src_a, char* dst_a, uint64_t n_a, const char* src_b, char* dst_b, uint64_t n_b, hipStream_t st) {
  if ((((uintptr_t)src_a ^ (uintptr_t)dst_a) & 15u) || (((uintptr_t)src_b ^ (uintptr_t)dst_b) & 15u)) return hipErrorInvalidValue;
  const uint64_t most = n_a > n_b ? n_a : n_b;
  if (most == 0) return hipSuccess;
  hipLaunchKernelGGL(k_put_text, dim3(grid_stride_for((most >> 4) + 1, KTJ_BLOCK), 2), dim3(KTJ_BLOCK), 0, st, src_a, dst_a, n_a, src_b,
                     dst_b, n_b);
  return KTJ_LAUNCH_CHECK();
}

/* up to KTJ_MAX_PIECES pieces of page-locked host memory, each to its place in device memory (the
 * small submissions an engine has gathered); source and destination of a piece agree modulo 16 */
__global__ void k_put_pieces(PieceJobs jobs) {
  const char* src = jobs.src[blockIdx.y];
  char* dst = jobs.dst[blockIdx.y];
  const uint64_t n = jobs.n[blockIdx.y];
  uint64_t head = (16u - (uint32_t)((uintptr_t)dst & 15u)) & 15u;
  if (head > n) head = n;
  const uint64_t body = (n - head) >> 4, tail = (n - head) & 15u;
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
  if (t < head) dst[t] = src[t];
  const uint4* sv = reinterpret_cast<const uint4*>(src + head);
  uint4* dv = reinterpret_cast<uint4*>(dst + head);
  for (uint64_t k = t; k < body; k += stride) dv[k] = sv[k];
  if (t < tail) dst[head + body * 16u + t] = src[head + body * 16u + t];
}
hipError_t put_pieces(const PieceJobs& jobs, hipStream_t st) {
  if (jobs.count == 0) return hipSuccess;
  if (jobs.count > KTJ_MAX_PIECES) return hipErrorInvalidValue;
  uint64_t most = 0;
  for (uint32_t k = 0; k < jobs.count; ++k) {
    if (((uintptr_t)jobs.src[k] ^ (uintptr_t)jobs.dst[k]) & 15u) return hipErrorInvalidValue;
    if (jobs.n[k] > most) most = jobs.n[k];
  }
  hipLaunchKernelGGL(k_put_pieces, dim3(grid_stride_for((most >> 4) + 1, KTJ_BLOCK), jobs.count), dim3(KTJ_BLOCK), 0, st, jobs);
  return KTJ_LAUNCH_CHECK();
}

/* The document's way to the host: bound by the link (57 GB/s), which few workgroups fill; they take the
 * parts one after the other so that the host can copy a part on while the next ones cross.  One launch
 * for many parts: between copy engine transfers or launches of one part each, the event behind every
 * part costs 15 us or 6 us (12.6 MB in 1 MiB parts: 463 and 385 us). */
#define COPY_PARTS_GRID 64u
__global__ void __launch_bounds__(KTJ_BLOCK)
k_copy_parts(const uint4* src, uint64_t n16, uint64_t first, uint64_t last, uint64_t part16, uint32_t n_slots, uint4* slots,
             uint64_t* flag, uint64_t seq, unsigned int* done) {
  for (uint64_t c = first; c < last; ++c) {
    const uint64_t from = c * part16, len = n16 - from < part16 ? n16 - from : part16;
    const uint32_t slot = (uint32_t)(c % n_slots);
    const uint4* s = src + from;
    uint4* d = slots + (uint64_t)slot * part16;
    for (uint64_t k = (uint64_t)blockIdx.x * KTJ_BLOCK + threadIdx.x; k < len; k += (uint64_t)gridDim.x * KTJ_BLOCK) d[k] = s[k];
    wave_stores_done();
    __syncthreads();
    if (threadIdx.x == 0) {
      __threadfence_system(); /* this workgroup's share, all of it stored by now, is in host memory before it counts as done */
      if (atomicAdd(&done[slot], 1u) == gridDim.x - 1u) {
        done[slot] = 0;
        __threadfence_system();
        __hip_atomic_store(&flag[slot], seq + c, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
}
hipError_t copy_parts(const char* src, uint64_t n, uint64_t first, uint64_t last, uint64_t part_bytes, uint32_t n_slots, char* slots,
                      uint64_t* flag, uint64_t seq, unsigned int* done, hipStream_t st) {
  if (first >= last) return hipSuccess;
  if ((((uintptr_t)src | (uintptr_t)slots | part_bytes) & 15u) || n_slots == 0 || n_slots > KTJ_PART_SLOTS || last - first > n_slots ||
      (last - 1) * part_bytes >= n)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_copy_parts, dim3(COPY_PARTS_GRID), dim3(KTJ_BLOCK), 0, st, reinterpret_cast<const uint4*>(src), (n + 15) / 16,
                     first, last, part_bytes / 16, n_slots, reinterpret_cast<uint4*>(slots), flag, seq, done);
  return KTJ_LAUNCH_CHECK();
}

/* plain 16-byte-per-lane copy of known size: the yardstick for the HBM counters */
__global__ void k_copy_reference(const uint4* src, uint4* dst, uint64_t n16) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * blockDim.x) dst[i] = src[i];
}
hipError_t copy_reference(const void* src, void* dst, uint64_t bytes, hipStream_t st) {
  const uint64_t n16 = bytes / 16;
  if (n16 == 0) return hipSuccess;
  hipLaunchKernelGGL(k_copy_reference, dim3(grid_stride_for(n16, KTJ_BLOCK * 4)), dim3(KTJ_BLOCK), 0, st,
                     static_cast<const uint4*>(src), static_cast<uint4*>(dst), n16);
  return KTJ_LAUNCH_CHECK();
}

}  // namespace gpu
}  // namespace ktj
