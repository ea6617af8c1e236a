/*
 * small.hip — the whole pass for traces of up to SMALL_ROWS records, in three launches.
 *
 * A pass over a few hundred records is bound by the number of dependent steps, not by bytes: the forty
 * launches of a large trace, each one or two microseconds of work behind five of start, end and gap,
 * two read-backs, and a formatter that fetches fifty kilobytes of code cold (35 us for fifteen
 * activities) came to 260 us.  Here
 *   k_small_join   one workgroup decodes every record and makes all joins in tables in LDS (160 KB hold
 *                  tables for 2048 rows), barriers in place of launches; the other workgroups make the
 *                  dictionary views beside it
 *   k_small_rows   the first workgroup puts the rows in canonical order (keys in registers and LDS), the
 *                  others make the joined rows and their lengths beside it
 *   k_small_emit   every workgroup finds its activities' places (a sum over at most 2048 lengths), a
 *                  wavefront formats one activity at a time (SegWriter), header and footer text and the
 *                  scalars for the host go along
 * and the host waits once.  What the three do not handle (rows that need a Stream Sync row of their own,
 * a span of timestamps too wide for a sort key) they flag, and the host takes the launches of a large trace.
 */
#include "gpu_common.h"

namespace ktj {
namespace gpu {

#define SMALL_SLOTS (2u * SMALL_ROWS)
#define SMALL_JOIN_THREADS 1024u
#define SMALL_PER ((SMALL_ROWS + SMALL_JOIN_THREADS - 1u) / SMALL_JOIN_THREADS) /* rows of a class per thread */
#define SMALL_DICT_PER_BLOCK (SMALL_JOIN_THREADS / 64u)

/* ------------------------------------------------------------------------------------------ */
/* first launch: decode and joins                                                               */
/* ------------------------------------------------------------------------------------------ */
/* LDS tables: a slot holds 1 + the index of a row (or record) with its key, the keys stay where they
 * are.  At most three quarters full, so a probe sequence ends. */
template <typename KeyOf>
__device__ __forceinline__ uint32_t lds_insert(uint32_t* table, uint32_t mask, uint64_t hash, uint64_t key, uint32_t entry, KeyOf key_of) {
  uint32_t slot = (uint32_t)hash & mask;
  for (uint32_t probe = 0; probe <= mask; ++probe) {
    uint32_t cur = __hip_atomic_load(&table[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (cur == 0) { cur = atomicCAS(&table[slot], 0u, entry); if (cur == 0) return slot; }
    if (key_of(cur) == key) return slot;
    slot = (slot + 1u) & mask;
  }
  return KTJ_NOSLOT;
}
template <typename KeyOf>
__device__ __forceinline__ uint32_t lds_find(const uint32_t* table, uint32_t mask, uint64_t hash, uint64_t key, KeyOf key_of) {
  uint32_t slot = (uint32_t)hash & mask;
  for (uint32_t probe = 0; probe <= mask; ++probe) {
    const uint32_t cur = table[slot];
    if (cur == 0) return KTJ_NOSLOT;
    if (key_of(cur) == key) return slot;
    slot = (slot + 1u) & mask;
  }
  return KTJ_NOSLOT;
}

/* The steps and their rules are those of the kernels of a large trace (k_build_cpu_ids, k_build_extcorr,
 * k_join_runtime with its winners, k_link_device, k_after_link, k_dense_*); here the
 * winner of every slot is always known before it is read, so there is one form of each step. */
__global__ void __launch_bounds__(SMALL_JOIN_THREADS) k_small_join(SmallArgs A) {
  if (blockIdx.x != 0) {
    const uint32_t id = (blockIdx.x - 1u) * SMALL_DICT_PER_BLOCK + (threadIdx.x >> 6);
    if (id < A.ctx.dict.n)
      dict_string(A.ctx.dict.raw_blob, A.ctx.dict.raw_off, id, A.entries, const_cast<char*>(A.ctx.dict.name_blob),
                  const_cast<char*>(A.ctx.dict.arg_blob));
    return;
  }
  __shared__ uint64_t s_corr[SMALL_ROWS];             /* runtime rows, then device rows */
  __shared__ uint32_t t_cpu[SMALL_SLOTS], t_full[SMALL_SLOTS], f_first[SMALL_SLOTS], f_stream[SMALL_SLOTS];
  __shared__ uint32_t t_narrow[SMALL_SLOTS], n_ext[SMALL_SLOTS], n_kern[SMALL_SLOTS], n_copy[SMALL_SLOTS];
  __shared__ uint64_t ext_linked[(SMALL_EXT + 63u) / 64u];
  __shared__ uint32_t s_cnt[8];
  enum { C_OOR = 0, C_BAD, C_LINKED, C_VALID, C_UNRESOLVED, C_ORPHANS, C_UNFIT, C_DENSE };
  const uint32_t tid = threadIdx.x, ng = A.ng, nr = A.nr, nd = A.nd, nx = A.nx;
  const uint32_t mask = A.slots - 1u;
  const Columns c = A.c;
  if (tid == 0) stage_clock(A.sc, 0);
  for (uint32_t k = tid; k < A.slots; k += SMALL_JOIN_THREADS) {
    t_cpu[k] = 0; t_full[k] = 0; f_first[k] = 0xFFFFFFFFu; f_stream[k] = 0;
    t_narrow[k] = 0; n_ext[k] = 0; n_kern[k] = 0; n_copy[k] = 0;
  }
  if (tid < 8) s_cnt[tid] = 0;
  __syncthreads();
  auto count = [&](int which, uint32_t mine) { /* all lanes that are here; one LDS atomic per wavefront */
    const uint32_t w = wave_sum_u32(mine);
    if (lane_id() == 0 && w) atomicAdd(&s_cnt[which], w);
  };

  /* decode */
  RowCols rt[SMALL_PER], dv[SMALL_PER];
  {
    uint32_t valid = 0, oor = 0, unfit = 0;
#pragma unroll
    for (uint32_t k = 0; k < SMALL_PER; ++k) {
      const uint32_t i = tid + k * SMALL_JOIN_THREADS;
      if (i < ng) {
        const ktj_generic_rec g = A.g[i];
        const RowCols r = cols_generic(g, A.ctx);
        store_cols(c, i, r);
        valid += r.meta & KTJ_M_VALID ? 1u : 0u;
        unfit |= g.type == KTJ_TYPE_CUDA_SYNC ? 1u : 0u; /* may need a Stream Sync row */
      }
      if (i < nr) {
        rt[k] = cols_runtime(A.r[i], A.clk, A.win_start, A.win_end);
        store_cols(c, ng + i, rt[k]);
        s_corr[i] = rt[k].corr;
        const uint32_t v = rt[k].meta & KTJ_M_VALID ? 1u : 0u;
        valid += v; oor += 1u - v;
      }
      if (i < nd) {
        dv[k] = cols_device(A.d[i], A.clk, A.win_start, A.win_end);
        store_cols(c, ng + nr + i, dv[k]);
        s_corr[nr + i] = dv[k].corr;
        const uint32_t v = dv[k].meta & KTJ_M_VALID ? 1u : 0u;
        valid += v; oor += 1u - v;
      }
    }
    count(C_VALID, valid); count(C_OOR, oor); count(C_UNFIT, unfit);
  }
  __syncthreads();
  if (tid == 0) stage_clock(A.sc, 1);

  auto cpu_key = [&](uint32_t e) { return c.corr[e - 1u]; };
  auto full_key = [&](uint32_t e) { return s_corr[e - 1u]; };
  /* narrow table: entry = 1 + runtime row, or 1 + record with the top bit */
  auto narrow_key = [&](uint32_t e) { return e & 0x80000000u ? A.x[(e & 0x7FFFFFFFu) - 1u].correlation : narrow_corr_key(s_corr[e - 1u]); };

  /* CPU-op ids (activityMap_) */
#pragma unroll
  for (uint32_t k = 0; k < SMALL_PER; ++k) {
    const uint32_t i = tid + k * SMALL_JOIN_THREADS;
    if (i < ng) { const uint64_t key = c.corr[i]; lds_insert(t_cpu, mask, hash64(key), key, i + 1u, cpu_key); }
  }
  __syncthreads();
  /* external correlation: the last record of an id stays; does its external id name a CPU op? */
  for (uint32_t base = 0; base < nx; base += SMALL_JOIN_THREADS) {
    const uint32_t i = base + tid;
    bool linked = false;
    if (i < nx) {
      const ktj_extcorr_rec rec = A.x[i];
      const uint32_t slot = lds_insert(t_narrow, mask, hash64(rec.correlation), rec.correlation, (i + 1u) | 0x80000000u, narrow_key);
      atomicMax(&n_ext[slot], i + 1u);
      linked = lds_find(t_cpu, mask, hash64(rec.external_id), rec.external_id, cpu_key) != KTJ_NOSLOT;
    }
    const uint64_t b = __ballot(linked);
    if (lane_id() == 0 && i < nx) ext_linked[i >> 6] = b;
  }
  /* runtime rows: first row and last stream of an id, last launch and last copy of a narrowed id */
  bool carries_stream = false;
  uint32_t sf_r[SMALL_PER];
#pragma unroll
  for (uint32_t k = 0; k < SMALL_PER; ++k) {
    const uint32_t i = tid + k * SMALL_JOIN_THREADS;
    if (i >= nr) continue;
    const uint64_t key = rt[k].corr;
    const uint32_t sf = lds_insert(t_full, mask, hash64(key), key, i + 1u, full_key);
    sf_r[k] = sf;
    atomicMin(&f_first[sf], i);
    if (rt[k].meta & KTJ_M_HAS_STREAM) { atomicMax(&f_stream[sf], i + 1u); carries_stream = true; }
    const uint32_t kind = (rt[k].meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT;
    if ((rt[k].meta & KTJ_M_VALID) && kind != KTJ_RT_DEFAULT) {
      const uint64_t nk = narrow_corr_key(key);
      const uint32_t sn = lds_insert(t_narrow, mask, hash64(nk), nk, i + 1u, narrow_key);
      atomicMax(kind == KTJ_RT_KERNEL ? &n_kern[sn] : &n_copy[sn], i + 1u);
    }
  }
  const bool have_stream = __syncthreads_or(carries_stream ? 1 : 0) != 0;

  /* what the winners hand over */
  auto external_of = [&](uint32_t sn, bool* linked) -> int32_t { /* the slot's "External id" */
    *linked = false;
    if (sn == KTJ_NOSLOT) return 0;
    const uint32_t x = n_ext[sn];
    if (x == 0 || !((ext_linked[(x - 1u) >> 6] >> ((x - 1u) & 63u)) & 1ull)) return 0;
    *linked = true;
    return (int32_t)(int64_t)A.x[x - 1u].external_id;
  };
  uint32_t n_bad = 0, n_linked = 0, n_unresolved = 0, n_orphans = 0;
#pragma unroll
  for (uint32_t k = 0; k < SMALL_PER; ++k) {
    const uint32_t i = tid + k * SMALL_JOIN_THREADS;
    if (i >= nr) continue;
    const uint64_t nk = narrow_corr_key(rt[k].corr);
    bool linked;
    c.ext[ng + i] = external_of(lds_find(t_narrow, mask, hash64(nk), nk, narrow_key), &linked);
    if (linked && (rt[k].meta & KTJ_M_VALID)) ++n_linked;
    const uint32_t f = f_first[sf_r[k]];
    if (f != i) { const int64_t t1 = c.ts[ng + f]; if (rt[k].ts != 0 && t1 > rt[k].ts) ++n_bad; }
  }
  uint32_t orphan_slot[SMALL_PER];
#pragma unroll
  for (uint32_t k = 0; k < SMALL_PER; ++k) {
    const uint32_t i = tid + k * SMALL_JOIN_THREADS;
    orphan_slot[k] = KTJ_NOSLOT;
    if (i >= nd) continue;
    const bool valid = (dv[k].meta & KTJ_M_VALID) != 0;
    const uint32_t dom = (dv[k].meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT;
    const uint64_t id = dv[k].corr, nk = narrow_corr_key(id);
    const uint32_t sn = lds_find(t_narrow, mask, hash64(nk), nk, narrow_key);
    const uint32_t sf = valid ? lds_insert(t_full, mask, hash64(id), id, nr + i + 1u, full_key) : lds_find(t_full, mask, hash64(id), id, full_key);
    bool linked;
    c.ext[ng + nr + i] = external_of(sn, &linked);
    if (linked && valid) ++n_linked;
    DevLink l;
    l.p[0] = l.p[1] = l.p[2] = 0; l.flags = 0; l.coll = 0;
    if (sn != KTJ_NOSLOT && dom != KTJ_DOM_MEMSET) {
      const uint32_t cp = n_copy[sn], kn = n_kern[sn];
      if (cp) { const ktj_runtime_rec& w = A.r[cp - 1u]; l.flags = KTJ_DL_HAS_SIZE; l.p[0] = w.kind == KTJ_RT_COPY ? w.u.copy.size : w.u.malloc_.size; }
      else if (kn) { l.flags = KTJ_DL_HAS_GRID; pack_grid(A.r[kn - 1u], l.p); }
    }
    A.link[i] = l;
    if (sf != KTJ_NOSLOT) {
      const uint32_t f = f_first[sf]; /* a runtime row's index where some runtime row has the id: final since the barrier */
      if (f < nr) {
        const int64_t t1 = c.ts[ng + f];
        if (valid && dv[k].ts != 0 && t1 > dv[k].ts) ++n_bad;
        const uint32_t ss = f_stream[sf];
        if (have_stream && is_async_op(dom) && dv[k].res == 0 && ss) {
          const ktj_runtime_rec& w = A.r[ss - 1u];
          const uint64_t stream = w.kind == KTJ_RT_KERNEL ? w.u.kernel.stream : w.u.copy.stream;
          if (stream != 0) { dv[k].res = (int64_t)stream; c.res[ng + nr + i] = dv[k].res; }
        }
      } else if (valid) { atomicMin(&f_first[sf], nr + i); orphan_slot[k] = sf; ++n_orphans; }
    }
    if (is_async_op(dom) && dv[k].res == 0) ++n_unresolved;
  }
  count(C_LINKED, n_linked); count(C_UNRESOLVED, n_unresolved); count(C_ORPHANS, n_orphans);
  __syncthreads();
  /* device rows whose id no runtime row has, against the first of them */
#pragma unroll
  for (uint32_t k = 0; k < SMALL_PER; ++k) {
    const uint32_t i = tid + k * SMALL_JOIN_THREADS;
    if (orphan_slot[k] == KTJ_NOSLOT) continue;
    const uint32_t f = f_first[orphan_slot[k]];
    if (f != nr + i) { const int64_t t2 = c.ts[ng + f]; if (t2 != 0 && dv[k].ts > t2) ++n_bad; }
  }
  count(C_BAD, n_bad);
  const bool fill_queues = have_stream && s_cnt[C_UNRESOLVED] != 0;
  if (fill_queues) { /* queue -> stream, where a queue shows one stream only */
    for (uint32_t k = tid; k < A.slots; k += SMALL_JOIN_THREADS) { t_narrow[k] = 0; n_kern[k] = 0xFFFFFFFFu; n_copy[k] = 0; }
    __syncthreads();
    auto queue_key = [&](uint32_t e) { return A.d[e - 1u].queue; };
    uint32_t q_slot[SMALL_PER];
#pragma unroll
    for (uint32_t k = 0; k < SMALL_PER; ++k) {
      const uint32_t i = tid + k * SMALL_JOIN_THREADS;
      q_slot[k] = KTJ_NOSLOT;
      if (i >= nd) continue;
      const uint64_t queue = A.d[i].queue;
      if (!is_async_op((dv[k].meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT) || dv[k].res == 0 || queue == 0) continue;
      q_slot[k] = lds_insert(t_narrow, mask, hash64(queue), queue, i + 1u, queue_key);
      atomicMin(&n_kern[q_slot[k]], i);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < SMALL_PER; ++k)
      if (q_slot[k] != KTJ_NOSLOT && c.res[ng + nr + n_kern[q_slot[k]]] != dv[k].res) n_copy[q_slot[k]] = 1u;
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < SMALL_PER; ++k) {
      const uint32_t i = tid + k * SMALL_JOIN_THREADS;
      if (i >= nd || !is_async_op((dv[k].meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT) || dv[k].res != 0) continue;
      const uint64_t queue = A.d[i].queue;
      const uint32_t s = lds_find(t_narrow, mask, hash64(queue), queue, queue_key);
      if (s != KTJ_NOSLOT && n_copy[s] == 0) { dv[k].res = c.res[ng + nr + n_kern[s]]; c.res[ng + nr + i] = dv[k].res; }
    }
    __syncthreads();
  }
  if (have_stream) { /* dense per-device stream numbers, in order of first appearance */
    for (uint32_t k = tid; k < A.slots; k += SMALL_JOIN_THREADS) { t_full[k] = 0; n_ext[k] = 0xFFFFFFFFu; }
    __syncthreads();
    auto pair_hash = [&](int32_t dev, uint64_t key) { return hash64(key ^ hash64((uint64_t)(int64_t)dev + 0x9E3779B97F4A7C15ULL)); };
    uint32_t p_slot[SMALL_PER];
#pragma unroll
    for (uint32_t k = 0; k < SMALL_PER; ++k) {
      const uint32_t i = tid + k * SMALL_JOIN_THREADS;
      p_slot[k] = KTJ_NOSLOT;
      if (i >= nd) continue;
      const int32_t device = (int32_t)dv[k].dev;
      uint64_t key;
      if (!dense_key((dv[k].meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT, (uint64_t)dv[k].res, A.d[i].queue, &key)) continue;
      /* a pair is equal when device and key are: 0 and not the key tells a row of another device apart */
      auto same = [&](uint32_t e) -> uint64_t {
        const ktj_device_rec& o = A.d[e - 1u];
        if (o.device != device) return ~key;
        const uint64_t res = (uint64_t)c.res[ng + nr + e - 1u];
        return res != 0 ? res : o.queue | (1ULL << 63);
      };
      p_slot[k] = lds_insert(t_full, mask, pair_hash(device, key), key, i + 1u, same);
      atomicMin(&n_ext[p_slot[k]], i);
    }
    __syncthreads();
    uint32_t* list_first = f_first; /* of the pairs: their first rows and devices */
    int32_t* list_dev = reinterpret_cast<int32_t*>(f_stream);
#pragma unroll
    for (uint32_t k = 0; k < SMALL_PER; ++k) {
      const uint32_t i = tid + k * SMALL_JOIN_THREADS;
      if (p_slot[k] != KTJ_NOSLOT && n_ext[p_slot[k]] == i) {
        const uint32_t at = atomicAdd(&s_cnt[C_DENSE], 1u);
        list_first[at] = i; list_dev[at] = (int32_t)dv[k].dev;
      }
    }
    __syncthreads();
    const uint32_t pairs = s_cnt[C_DENSE];
#pragma unroll
    for (uint32_t k = 0; k < SMALL_PER; ++k) {
      const uint32_t i = tid + k * SMALL_JOIN_THREADS;
      if (p_slot[k] == KTJ_NOSLOT || n_ext[p_slot[k]] != i) continue;
      uint32_t rank = 1;
      for (uint32_t j = 0; j < pairs; ++j) rank += list_dev[j] == (int32_t)dv[k].dev && list_first[j] < i ? 1u : 0u;
      n_kern[p_slot[k]] = rank;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < SMALL_PER; ++k)
      if (p_slot[k] != KTJ_NOSLOT) dv[k].res = (int64_t)n_kern[p_slot[k]];
  }
#pragma unroll
  for (uint32_t k = 0; k < SMALL_PER; ++k) { /* resourceId() = stream != 0 ? stream : queue (RocprofActivity.h:100-102) */
    const uint32_t i = tid + k * SMALL_JOIN_THREADS;
    if (i >= nd || !is_async_op((dv[k].meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT)) continue;
    c.res[ng + nr + i] = dv[k].res != 0 ? dv[k].res : (int64_t)A.d[i].queue;
  }
  __syncthreads();
  if (tid == 0) {
    Scalars* s = A.sc;
    s->ts_min_biased = ~0ULL; s->ts_max_biased = 0;
    s->out_of_range = s_cnt[C_OOR]; s->out_of_order = s_cnt[C_BAD]; s->n_linked = s_cnt[C_LINKED]; s->n_valid = s_cnt[C_VALID];
    s->n_flow = 0; s->n_blank_names = 0; s->n_sync_typed = 0;
    s->n_unresolved = s_cnt[C_UNRESOLVED]; s->n_device_orphans = s_cnt[C_ORPHANS];
    s->error = s_cnt[C_UNFIT] ? KTJ_DEVERR_SMALL_UNFIT : 0u;
    s->have_stream_src = have_stream ? 1u : 0u; s->n_dev_ranks = 0; s->n_res_ranks = 0; s->n_dense = s_cnt[C_DENSE];
    s->n_plain = 0; s->runtime_ids_repeat = 0; s->n_queues = 0; s->n_sync_rows = 0; s->ext_ids_repeat = 0;
    for (uint32_t k = 0; k < KTJ_PART_SLOTS; ++k) s->part_done[k] = 0;
    stage_clock(s, 2);
  }
}

/* ------------------------------------------------------------------------------------------ */
/* second launch: canonical order; joined rows and lengths                                      */
/* ------------------------------------------------------------------------------------------ */
#define ROWS_THREADS 512u
#define SORT_ITEMS (SMALL_ROWS / ROWS_THREADS) /* words per thread: word e = thread * SORT_ITEMS + item */
static_assert(SORT_ITEMS == 4u, "the network below exchanges four words per thread");

__device__ __forceinline__ void sort_pair(uint64_t& lo, uint64_t& hi, bool up) {
  const uint64_t a = lo, b = hi;
  const bool swap = (a > b) == up;
  lo = swap ? b : a;
  hi = swap ? a : b;
}
template <uint32_t J> __device__ __forceinline__ void sort_in_thread(uint64_t (&w)[SORT_ITEMS], uint32_t first, uint32_t k) {
#pragma unroll
  for (uint32_t i = 0; i < SORT_ITEMS; ++i)
    if ((i & J) == 0) sort_pair(w[i], w[i | J], ((first + i) & k) == 0);
}
/* Bitonic network over up to 2048 distinct words, four consecutive ones per thread: distances 1 and 2
 * inside a thread, below 256 between the lanes of a wavefront, the three above through LDS.  It ends at
 * the power of two that holds n words.  (Eight words on each of 256 threads: 37 us for 1800 rows with
 * the ranks in front of it, most of it instructions that one wavefront per SIMD issues one by one.) */
__device__ __forceinline__ void sort_words(uint64_t (&w)[SORT_ITEMS], uint32_t n, uint64_t* lds) {
  const uint32_t first = threadIdx.x * SORT_ITEMS;
  for (uint32_t k = 2; (k >> 1) < n; k <<= 1) {
    for (uint32_t j = k >> 1; j > 0; j >>= 1) {
      if (j >= SORT_ITEMS) {
        uint64_t o[SORT_ITEMS];
        if (j >= 64u * SORT_ITEMS) {
          __syncthreads();
#pragma unroll
          for (uint32_t i = 0; i < SORT_ITEMS; ++i) lds[i * ROWS_THREADS + threadIdx.x] = w[i];
          __syncthreads();
#pragma unroll
          for (uint32_t i = 0; i < SORT_ITEMS; ++i) o[i] = lds[i * ROWS_THREADS + (threadIdx.x ^ (j / SORT_ITEMS))];
        } else {
#pragma unroll
          for (uint32_t i = 0; i < SORT_ITEMS; ++i) o[i] = __shfl_xor((unsigned long long)w[i], (int)(j / SORT_ITEMS));
        }
        const bool keep_min = ((first & j) == 0) == ((first & k) == 0); /* the same for a thread's four words */
#pragma unroll
        for (uint32_t i = 0; i < SORT_ITEMS; ++i) w[i] = (o[i] < w[i]) == keep_min ? o[i] : w[i];
      } else if (j == 2u) sort_in_thread<2>(w, first, k);
      else sort_in_thread<1>(w, first, k);
    }
  }
}

__device__ __forceinline__ void small_order(const SmallArgs& A) {
  __shared__ uint32_t t_pair[SMALL_SLOTS], rank_of[SMALL_ROWS], pair_row[SMALL_ROWS];
  __shared__ int64_t s_dev[SMALL_ROWS], s_res[SMALL_ROWS];
  __shared__ uint64_t words[SMALL_ROWS];
  __shared__ uint64_t s_min, s_max;
  __shared__ uint32_t n_pairs;
  const Columns c = A.c;
  const uint32_t n = A.ng + A.nr + A.nd, mask = A.slots - 1u, first = threadIdx.x * SORT_ITEMS;
  if (threadIdx.x == 0) { s_min = ~0ULL; s_max = 0; n_pairs = 0; stage_clock(A.sc, 3); }
  for (uint32_t k = threadIdx.x; k < A.slots; k += ROWS_THREADS) t_pair[k] = 0;
  uint32_t slot[SORT_ITEMS];
  uint64_t ts[SORT_ITEMS];
  int64_t dev[SORT_ITEMS], res[SORT_ITEMS];
  uint32_t meta[SORT_ITEMS];
#pragma unroll
  for (uint32_t i = 0; i < SORT_ITEMS; ++i) { /* all loads in flight together */
    const uint32_t a = first + i;
    const bool in = a < n;
    meta[i] = in ? c.meta[a] : 0u;
    dev[i] = in ? c.dev[a] : 0; res[i] = in ? c.res[a] : 0; ts[i] = in ? (uint64_t)c.ts[a] ^ 0x8000000000000000ULL : 0;
  }
#pragma unroll
  for (uint32_t i = 0; i < SORT_ITEMS; ++i) { s_dev[first + i] = dev[i]; s_res[first + i] = res[i]; }
  __syncthreads();
  uint64_t lo = ~0ULL, hi = 0;
#pragma unroll
  for (uint32_t i = 0; i < SORT_ITEMS; ++i) {
    slot[i] = KTJ_NOSLOT;
    if (!(meta[i] & KTJ_M_VALID)) continue;
    lo = ts[i] < lo ? ts[i] : lo;
    hi = ts[i] > hi ? ts[i] : hi;
    auto same = [&](uint32_t e) -> uint64_t { return s_dev[e - 1u] == dev[i] && s_res[e - 1u] == res[i] ? 1u : 0u; };
    const uint64_t h = ((uint64_t)res[i] ^ ((uint64_t)dev[i] << 17)) * 0x9E3779B97F4A7C15ULL;
    slot[i] = lds_insert(t_pair, mask, h >> 40, 1u, first + i + 1u, same);
    if (t_pair[slot[i]] == first + i + 1u) pair_row[atomicAdd(&n_pairs, 1u)] = first + i; /* this row stands for the pair */
  }
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t l2 = __shfl_xor((unsigned long long)lo, o), h2 = __shfl_xor((unsigned long long)hi, o);
    lo = l2 < lo ? l2 : lo;
    hi = h2 > hi ? h2 : hi;
  }
  if (lane_id() == 0) { atomicMin((unsigned long long*)&s_min, (unsigned long long)lo); atomicMax((unsigned long long*)&s_max, (unsigned long long)hi); }
  __syncthreads();
  const uint32_t m = n_pairs;
  for (uint32_t p = threadIdx.x; p < m; p += ROWS_THREADS) {
    const int64_t pd = s_dev[pair_row[p]], pr = s_res[pair_row[p]];
    uint32_t r = 0;
    for (uint32_t q = 0; q < m; ++q) {
      const int64_t qd = s_dev[pair_row[q]], qr = s_res[pair_row[q]];
      r += qd < pd || (qd == pd && qr < pr) ? 1u : 0u;
    }
    rank_of[pair_row[p]] = r;
  }
  __syncthreads();
  /* word = rank | timestamp above the smallest | arrival index; dropped rows behind everything */
  const uint64_t ts_min = s_min, span = s_max >= s_min ? s_max - s_min : 0;
  const uint32_t ts_bits = span ? 64u - (uint32_t)__builtin_clzll(span) : 0u, rank_bits = m > 1u ? 32u - (uint32_t)__builtin_clz(m - 1u) : 0u;
  if (ts_bits + rank_bits > 52u) { if (threadIdx.x == 0) flag_error(A.sc, KTJ_DEVERR_SMALL_UNFIT); return; }
  uint64_t w[SORT_ITEMS];
#pragma unroll
  for (uint32_t i = 0; i < SORT_ITEMS; ++i)
    w[i] = slot[i] == KTJ_NOSLOT ? ~0ULL - (SMALL_ROWS - 1u) + (first + i)
                                 : ((((uint64_t)rank_of[t_pair[slot[i]] - 1u] << ts_bits) | (ts[i] - ts_min)) << 11) | (first + i);
  sort_words(w, n, words);
#pragma unroll
  for (uint32_t i = 0; i < SORT_ITEMS; ++i)
    if (first + i < n) A.perm[first + i] = (uint32_t)w[i] & (SMALL_ROWS - 1u);
  if (threadIdx.x == 0) stage_clock(A.sc, 4);
}

/* exact byte length, and whether some part of the activity has more pieces than a wavefront has lanes
 * (SegWriter below): SMALL_LEN_PLAIN.  The tail kinds that a large trace keeps in these bits are not needed here. */
#define SMALL_LEN_PLAIN 0x80000000u
#define SMALL_LEN_MASK 0x3FFFFFFFu
struct SegCounter {
  uint64_t n = 0;
  uint32_t segs = 0;
  __device__ KTJ_FI void ch(char) { ++n; ++segs; }
  template <unsigned N> __device__ KTJ_FI void lit(const PackedLit<N>&) { n += N; segs += (N + 15) / 16; }
  __device__ KTJ_FI void dec(uint64_t v) { n += (uint32_t)ndigits_u64(v); ++segs; }
  __device__ KTJ_FI void dec3(uint32_t) { n += 3; ++segs; }
  __device__ KTJ_FI void str(const char*, uint64_t len) { n += len; ++segs; }
  __device__ KTJ_FI void view(const char*, uint64_t len) { n += len; ++segs; }
  __device__ KTJ_FI void name(const char*, uint64_t len) { n += len; ++segs; }
  typedef uint32_t Prepared;
  __device__ KTJ_FI static Prepared prepare(uint64_t v) { return (uint32_t)ndigits_u64(v); }
  __device__ KTJ_FI void num(Prepared len) { n += len; ++segs; }
  __device__ KTJ_FI void relief() {}
};
__device__ __forceinline__ uint32_t small_length(const MatRow& m, const EmitCtx& ctx, Scalars* sc) {
  if (!(m.meta & KTJ_M_VALID)) return 0;
  SegCounter w;
  ActivityParts<SegCounter> parts;
  format_head(w, m, ctx, parts);
  uint32_t most = w.segs;
  w.segs = 0;
  format_args(w, m, ctx, parts);
  most = w.segs > most ? w.segs : most;
  w.segs = 0;
  format_flow(w, m, ctx, parts);
  most = w.segs > most ? w.segs : most;
  if (w.n >= (1ull << 30)) { flag_error(sc, KTJ_DEVERR_RECORD_TOO_LONG); return 0; }
  return (uint32_t)w.n | (most > 64u ? SMALL_LEN_PLAIN : 0u);
}
__device__ __forceinline__ void small_row_done(const SmallArgs& A, uint32_t a, const MatRow& m, bool active) {
  uint32_t flow = 0, blank = 0, plain = 0;
  if (active) {
    A.mat[a] = m;
    const uint32_t len = small_length(m, A.ctx, A.sc);
    A.len[a] = len;
    plain = len & SMALL_LEN_PLAIN ? 1u : 0u;
    if (m.meta & KTJ_M_VALID) {
      flow = m.meta & KTJ_M_FLOW ? 1u : 0u;
      if (!(m.meta & KTJ_M_NAME_BUILTIN) && m.name_id < A.ctx.dict.n && (dict_flags(A.ctx.dict, m.name_id) & KTJ_SF_NAME_UNKNOWN)) blank = 1;
    }
  }
  flow = wave_sum_u32(flow); blank = wave_sum_u32(blank); plain = wave_sum_u32(plain);
  if (lane_id() == 0) {
    if (plain) atomicAdd(&A.sc->n_plain, plain);
    if (flow) atomicAdd(&A.sc->n_flow, (unsigned long long)flow);
    if (blank) atomicAdd(&A.sc->n_blank_names, (unsigned long long)blank);
  }
}
#define ROWS_PER_BLOCK 256u
__global__ void __launch_bounds__(ROWS_THREADS) k_small_rows(SmallArgs A) {
  if (blockIdx.x == 0) { small_order(A); return; }
  if (threadIdx.x >= ROWS_PER_BLOCK) return; /* the rows spread over more CUs, one wavefront per SIMD */
  uint32_t b = blockIdx.x - 1u;
  const uint32_t bg = (A.ng + ROWS_PER_BLOCK - 1u) / ROWS_PER_BLOCK, br = (A.nr + ROWS_PER_BLOCK - 1u) / ROWS_PER_BLOCK;
  const Columns c = A.c;
  MatRow m;
  if (b < bg) {
    const uint32_t i = b * ROWS_PER_BLOCK + threadIdx.x;
    if (i < A.ng) {
      const ktj_generic_rec g = A.g[i];
      m = mat_generic(g, c.dev[i]);
      if (!(c.meta[i] & KTJ_M_VALID)) m.meta &= ~KTJ_M_VALID;
    }
    small_row_done(A, i, m, i < A.ng);
  } else if (b < bg + br) {
    const uint32_t i = (b - bg) * ROWS_PER_BLOCK + threadIdx.x, a = A.ng + i;
    if (i < A.nr) {
      const ktj_runtime_rec rec = A.r[i];
      const bool known = rec.cid < A.api.n_cids;
      const uint32_t name = known ? A.api.cid_name_ids[rec.cid] : KTJ_NONE;
      const bool fstart = known && ((A.api.flow_start_bits[rec.cid >> 5] >> (rec.cid & 31u)) & 1u);
      m = mat_runtime(rec, c.ts[a], c.dur[a], (c.meta[a] & KTJ_M_VALID) != 0, c.ext[a], name, fstart, rec.cid == A.api.malloc_cid);
    }
    small_row_done(A, a, m, i < A.nr);
  } else {
    const uint32_t i = (b - bg - br) * ROWS_PER_BLOCK + threadIdx.x, a = A.ng + A.nr + i;
    if (i < A.nd) {
      const DevLink l = A.link[i];
      m = mat_device_v(A.d[i], c.ts[a], c.dur[a], c.res[a], (c.meta[a] & KTJ_M_VALID) != 0, c.ext[a], (l.flags & KTJ_DL_HAS_GRID) != 0,
                       l.p[0], l.p[1], l.p[2], (l.flags & KTJ_DL_HAS_SIZE) != 0, l.p[0], l.coll);
    }
    small_row_done(A, a, m, i < A.nd);
  }
}

/* ------------------------------------------------------------------------------------------ */
/* third launch: the document                                                                   */
/* ------------------------------------------------------------------------------------------ */
/* One activity formatted by a whole wavefront.  format_activity runs with wavefront-uniform values; every
 * append — sixteen bytes of literal text, a number, a string — becomes the segment of one lane, and
 * flush() turns all of them into bytes at once: numbers to digits, a prefix sum of the lengths, every
 * lane its own bytes (unaligned stores of exactly its length).  An activity with a part (head, args, flow)
 * of more than 64 segments is left to PlainWriter. */
#define SEG_DEC 0x100u
#define SEG_STR 0x200u
struct SegWriter {
  uint64_t a, b;
  uint32_t meta;  /* bytes 0..24, SEG_DEC, or SEG_STR with the address in a and the length in b */
  uint32_t lane, n;
  __device__ KTJ_FI void start() { a = 0; b = 0; meta = 0; n = 0; }
  __device__ KTJ_FI void add(uint64_t lo, uint64_t hi, uint32_t what) {
    /* the count stays a value the compiler knows nothing about: otherwise it compares with constants and
     * keeps hundreds of masks alive across the whole formatter */
    asm volatile("" : "+s"(n));
    const bool me = lane == n;
    a = me ? lo : a; b = me ? hi : b; meta = me ? what : meta;
    ++n;
  }
  __device__ KTJ_FI void ch(char c) { add((uint64_t)(unsigned char)c, 0, 1); }
  template <unsigned N> __device__ KTJ_FI void lit(const PackedLit<N>& l) {
#pragma unroll
    for (unsigned i = 0; i < (N + 15) / 16; ++i)
      add(l.w[2 * i], 2 * i + 1 < (N + 7) / 8 ? l.w[2 * i + 1] : 0, N - 16 * i < 16 ? N - 16 * i : 16);
  }
  __device__ KTJ_FI void dec(uint64_t v) { add(v, 0, SEG_DEC); }
  __device__ KTJ_FI void dec3(uint32_t x) { add((uint64_t)(ascii4(x) >> 8), 0, 3); }
  __device__ KTJ_FI void str(const char* p, uint64_t len) { add((uint64_t)(uintptr_t)p, len, SEG_STR); }
  __device__ KTJ_FI void view(const char* p, uint64_t len) { str(p, len); }
  __device__ KTJ_FI void name(const char* p, uint64_t len) { str(p, len); }
  typedef uint64_t Prepared;
  __device__ KTJ_FI static Prepared prepare(uint64_t v) { return v; }
  __device__ KTJ_FI void num(Prepared v) { dec(v); }
  __device__ KTJ_FI void relief() {}

  __device__ KTJ_FI uint64_t flush(doc_ptr dst) {
    uint64_t w0 = a, w1 = b, w2 = 0;
    uint32_t len = lane < n ? meta & 0xFFu : 0u;
    const bool is_dec = lane < n && (meta & SEG_DEC), is_str = lane < n && (meta & SEG_STR);
    if (is_dec) { /* up to twenty digits, first digit in the lowest byte */
      const uint64_t top = a / 10000000000000000ULL, rest = a - top * 10000000000000000ULL, mid = rest / 100000000ULL;
      const uint64_t p0 = ascii8((uint32_t)top), p1 = ascii8((uint32_t)mid), p2 = ascii8((uint32_t)(rest - mid * 100000000ULL));
      len = (uint32_t)ndigits_u64(a);
      const uint32_t lead = 24u - len, sh = (lead & 7u) * 8u;
      const uint64_t q0 = lead < 8u ? p0 : lead < 16u ? p1 : p2, q1 = lead < 8u ? p1 : lead < 16u ? p2 : 0, q2 = lead < 8u ? p2 : 0;
      w0 = sh ? (q0 >> sh) | (q1 << (64u - sh)) : q0;
      w1 = sh ? (q1 >> sh) | (q2 << (64u - sh)) : q1;
      w2 = q2 >> sh;
    }
    if (is_str) {
      len = (uint32_t)b;
      const text_ptr p = reinterpret_cast<text_ptr>((uintptr_t)a);
      w0 = w1 = w2 = 0;
      if (len <= 24u) { /* at most 7 bytes behind the string are read: the blobs have room for them */
        if (len > 0u) w0 = get8(p);
        if (len > 8u) w1 = get8(p + 8);
        if (len > 16u) w2 = get8(p + 16);
      }
    }
    uint32_t end = len;
    for (int o = 1; o < 64; o <<= 1) { const uint32_t t = __shfl_up(end, o); if (lane >= (uint32_t)o) end += t; }
    const uint32_t total = __shfl(end, 63);
    if (len <= 24u) {
      const doc_ptr p = dst + (end - len);
      if (len >= 8u) put8(p, w0);
      if (len >= 16u) put8(p + 8, w1);
      if (len >= 24u) put8(p + 16, w2);
      put_low(p + (len & ~7u), len < 8u ? w0 : len < 16u ? w1 : w2, len & 7u);
    }
    uint64_t longer = __ballot(is_str && len > 24u);
    while (longer) { /* eight bytes per lane, neighbouring lanes neighbouring bytes */
      const int o = __ffsll((unsigned long long)longer) - 1;
      longer &= longer - 1;
      const uint32_t n_str = __shfl(len, o), at = __shfl(end, o) - n_str;
      const text_ptr p = reinterpret_cast<text_ptr>((uintptr_t)__shfl((unsigned long long)a, o));
      for (uint32_t k = lane * 8u; k < n_str; k += 512u) {
        const uint64_t v = get8(p + k);
        if (k + 8u <= n_str) put8(dst + at + k, v);
        else put_low(dst + at + k, v, n_str - k);
      }
    }
    start();
    return total;
  }
};
/* The same by one lane, byte by byte or nearly so. */
struct PlainWriter {
  doc_ptr p;
  __device__ KTJ_FI void bytes(uint64_t v, uint32_t n) {
    if (n >= 8u) { put8(p, v); p += 8; } else { put_low(p, v, n); p += n; }
  }
  __device__ KTJ_FI void ch(char c) { *p = c; ++p; }
  template <unsigned N> __device__ KTJ_FI void lit(const PackedLit<N>& l) {
    for (unsigned i = 0; i < (N + 7) / 8; ++i) bytes(l.w[i], N - 8 * i < 8 ? N - 8 * i : 8);
  }
  __device__ KTJ_FI void dec(uint64_t v) {
    const uint32_t n = (uint32_t)ndigits_u64(v);
    KTJ_NOUNROLL
    for (uint32_t k = n; k-- > 0;) { p[k] = (char)('0' + v % 10u); v /= 10u; }
    p += n;
  }
  __device__ KTJ_FI void dec3(uint32_t x) { bytes((uint64_t)(ascii4(x) >> 8), 3); }
  __device__ KTJ_FI void str(const char* s, uint64_t len) {
    const text_ptr t = reinterpret_cast<text_ptr>((uintptr_t)s);
    KTJ_NOUNROLL
    for (uint64_t k = 0; k < len; k += 8) bytes(get8(t + k), len - k < 8 ? (uint32_t)(len - k) : 8u);
  }
  __device__ KTJ_FI void view(const char* s, uint64_t len) { str(s, len); }
  __device__ KTJ_FI void name(const char* s, uint64_t len) { str(s, len); }
  typedef uint64_t Prepared;
  __device__ KTJ_FI static Prepared prepare(uint64_t v) { return v; }
  __device__ KTJ_FI void num(Prepared v) { dec(v); }
  __device__ KTJ_FI void relief() {}
};

#define SMALL_EMIT_PER (SMALL_ROWS / KTJ_BLOCK)
/* where every activity of the document begins, behind the prefix; their sum */
__device__ __forceinline__ uint64_t small_offsets(const uint32_t* perm, const uint32_t* len_of, uint32_t n, uint64_t* offs) {
  __shared__ uint64_t wave_tot[KTJ_BLOCK >> 6];
  uint32_t len[SMALL_EMIT_PER];
  const uint32_t first = threadIdx.x * SMALL_EMIT_PER;
#pragma unroll
  for (uint32_t k = 0; k < SMALL_EMIT_PER; ++k) len[k] = first + k < n ? perm[first + k] : KTJ_NOSLOT;
#pragma unroll
  for (uint32_t k = 0; k < SMALL_EMIT_PER; ++k) len[k] = len[k] != KTJ_NOSLOT ? len_of[len[k]] & SMALL_LEN_MASK : 0u;
  unsigned long long x = 0;
#pragma unroll
  for (uint32_t k = 0; k < SMALL_EMIT_PER; ++k) x += len[k];
  const unsigned long long mine = x;
  for (int o = 1; o < 64; o <<= 1) { const unsigned long long y = __shfl_up(x, (unsigned)o); if ((int)lane_id() >= o) x += y; }
  if (lane_id() == 63) wave_tot[threadIdx.x >> 6] = x;
  __syncthreads();
  uint64_t at = x - mine, total = 0;
  for (uint32_t w = 0; w < (KTJ_BLOCK >> 6); ++w) { if (w < (threadIdx.x >> 6)) at += wave_tot[w]; total += wave_tot[w]; }
#pragma unroll
  for (uint32_t k = 0; k < SMALL_EMIT_PER; ++k) { offs[first + k] = at; at += len[k]; }
  __syncthreads();
  return total;
}
__global__ void __launch_bounds__(KTJ_BLOCK) k_small_emit(const MatRow* mat, const uint32_t* perm, const uint32_t* len, Scalars* sc, EmitCtx ctx,
                                                          DocText T) {
  __shared__ uint64_t offs[SMALL_ROWS];
  const uint32_t error = sc->error, n = (uint32_t)sc->n_valid;
  const uint64_t total = error == 0 ? small_offsets(perm, len, n, offs) : 0;
  if (blockIdx.x == 0) { /* what the host waits for; nothing here waits for the other workgroups */
    constexpr uint32_t head_words = (uint32_t)(offsetof(Scalars, shard) / 4);
    if (threadIdx.x == 0) stage_clock(sc, 5);
    __syncthreads();
    const uint32_t* src = reinterpret_cast<const uint32_t*>(sc);
    uint32_t* dst = reinterpret_cast<uint32_t*>(T.h_sc);
    for (uint32_t k = threadIdx.x; k < head_words; k += KTJ_BLOCK) dst[k] = src[k];
    if (threadIdx.x == 0) *T.h_total = total;
  }
  if (error != 0 || T.n_prefix + total + T.n_suffix + 64u > T.out_cap) return; /* the host sees both and decides */
  if (blockIdx.x + 2u >= gridDim.x) {
    if (blockIdx.x + 2u == gridDim.x) put_text_block(T.prefix, T.out, T.n_prefix);
    else put_text_block(T.suffix, T.out + T.n_prefix + total, T.n_suffix);
    if (threadIdx.x == 0) *T.h_end = wall_clock64();
    return;
  }
  const uint32_t p = __builtin_amdgcn_readfirstlane(blockIdx.x * (KTJ_BLOCK >> 6) + (threadIdx.x >> 6));
  if (p >= n) return;
  const uint32_t row = __builtin_amdgcn_readfirstlane(perm[p]);
  if (!(__builtin_amdgcn_readfirstlane(len[row]) & SMALL_LEN_PLAIN)) { /* those are k_small_plain's */
    const MatRow m = mat[row];
    doc_ptr at = reinterpret_cast<doc_ptr>((uintptr_t)(T.out + T.n_prefix + offs[p]));
    SegWriter w;
    w.lane = lane_id();
    w.start();
    ActivityParts<SegWriter> parts;
    format_head(w, m, ctx, parts);
    at += w.flush(at);
    format_args(w, m, ctx, parts);
    at += w.flush(at);
    format_flow(w, m, ctx, parts);
    w.flush(at);
  }
  /* what arrives last stays: the pass's end, to within what the other wavefronts of that workgroup still have to do */
  if (threadIdx.x == 0) *T.h_end = wall_clock64();
}
/* Only when the rows have shown activities with more pieces than lanes (InputShapes of many operands,
 * long arrays): one lane per workgroup writes each of them. */
__global__ void __launch_bounds__(KTJ_BLOCK) k_small_plain(const MatRow* mat, const uint32_t* perm, const uint32_t* len, Scalars* sc, EmitCtx ctx,
                                                           DocText T) {
  __shared__ uint64_t offs[SMALL_ROWS];
  const uint32_t n = (uint32_t)sc->n_valid;
  small_offsets(perm, len, n, offs);
  if (threadIdx.x & 63u) return;
  for (uint32_t p = blockIdx.x * (KTJ_BLOCK >> 6) + (threadIdx.x >> 6); p < n; p += gridDim.x * (KTJ_BLOCK >> 6)) {
    if (!(len[perm[p]] & SMALL_LEN_PLAIN)) continue;
    const MatRow m = mat[perm[p]];
    PlainWriter w;
    w.p = reinterpret_cast<doc_ptr>((uintptr_t)(T.out + T.n_prefix + offs[p]));
    format_activity(w, m, ctx);
  }
  if (threadIdx.x == 0) *T.h_end = wall_clock64();
}

hipError_t small_pass(const SmallArgs& a, uint32_t n_strings, hipStream_t st) {
  const uint64_t n = (uint64_t)a.ng + a.nr + a.nd;
  if (n > SMALL_ROWS || a.nx > SMALL_EXT || a.slots > SMALL_SLOTS || (a.slots & (a.slots - 1u))) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_small_join, dim3(1u + grid_for(n_strings, SMALL_DICT_PER_BLOCK)), dim3(SMALL_JOIN_THREADS), 0, st, a);
  hipLaunchKernelGGL(k_small_rows, dim3(1u + grid_for(a.ng, ROWS_PER_BLOCK) + grid_for(a.nr, ROWS_PER_BLOCK) + grid_for(a.nd, ROWS_PER_BLOCK)), dim3(ROWS_THREADS),
                     0, st, a);
  return KTJ_LAUNCH_CHECK();
}
hipError_t small_emit(const SmallArgs& a, const DocText& t, hipStream_t st) {
  const uint64_t n = (uint64_t)a.ng + a.nr + a.nd; /* a wavefront per activity, two workgroups for the text */
  hipLaunchKernelGGL(k_small_emit, dim3(grid_for(n, KTJ_BLOCK >> 6) + 2u), dim3(KTJ_BLOCK), 0, st, (const MatRow*)a.mat, (const uint32_t*)a.perm,
                     (const uint32_t*)a.len, a.sc, a.ctx, t);
  return KTJ_LAUNCH_CHECK();
}
hipError_t small_plain(const SmallArgs& a, const DocText& t, hipStream_t st) {
  const uint64_t n = (uint64_t)a.ng + a.nr + a.nd;
  hipLaunchKernelGGL(k_small_plain, dim3(grid_for(n, KTJ_BLOCK >> 6)), dim3(KTJ_BLOCK), 0, st, (const MatRow*)a.mat, (const uint32_t*)a.perm,
                     (const uint32_t*)a.len, a.sc, a.ctx, t);
  return KTJ_LAUNCH_CHECK();
}
uint32_t small_slots(uint64_t ng, uint64_t nr, uint64_t nd, uint64_t nx) {
  uint64_t keys = ng > nr + nd ? ng : nr + nd;
  if (nx + nr > keys) keys = nx + nr;
  if (ng + nr + nd > keys) keys = ng + nr + nd;
  uint32_t s = 64;
  while (s < SMALL_SLOTS && s < 2 * keys) s <<= 1;
  return s;
}
bool small_fits(uint64_t ng, uint64_t nr, uint64_t nd, uint64_t nx) {
  return ng + nr + nd > 0 && ng + nr + nd <= SMALL_ROWS && nx <= SMALL_EXT && nx + nr <= SMALL_SLOTS / 4u * 3u;
}

}  // namespace gpu
}  // namespace ktj
