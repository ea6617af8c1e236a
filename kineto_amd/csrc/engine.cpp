/*
 * engine.cpp — host side of the trace post-processing engine behind the C ABI of include/ktj.h:
 * owns device memory, accepts submissions, orders the kernel stages on one HIP stream, formats
 * the handful of non-activity events and moves the finished document to the host / file.
 *
 * There is no CPU implementation of the activity path in this library: if a HIP call fails the
 * entry point returns KTJ_ERR_HIP.
 */
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <cerrno>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <string>
#include <unistd.h>
#include <unordered_map>
#include <utility>
#include <vector>

#include <rocprofiler-sdk/buffer_tracing.h>

#include "../../include/ktj_debug.h"
#include "../../include/ktj_rocprofiler.h"
#include "gpu_stages.h"
#include "host_events.h"
#include "part_queue.h"
#include "sdk_api_rows.h"

using namespace ktj;
using namespace ktj::gpu;

namespace {

#define KTJ_INPUT_ARENA_BYTES (1ull << 20)     /* device memory for the inputs of an engine, to begin with */
#define KTJ_INPUT_ARENA_MAX (64ull << 20)      /* what it may grow to for the engines that follow, room to spare included */
#define KTJ_STAGE_SMALL_BYTES (256u << 10) /* pinned ring that small submissions pass through */
#define KTJ_STAGE_SMALL_MAX (64u << 10)    /* largest submission that does */
/* large submissions: pinned chunks, two per copying thread.  Measured for 1.9 GB of records from
 * ordinary memory (one copy through the runtime's staging: 25 GB/s): chunks of 1 / 2 / 4 / 8 / 16 MiB
 * give 30 / 38 / 42 / 46 / 45 GB/s, 3, 4, 8 or 12 threads the same (each copy handed to the copy
 * engine costs some microseconds whatever its size). */
#define KTJ_STAGE_CHUNK (8ull << 20)
#define KTJ_STAGE_BIG_MIN (16ull << 20)    /* smallest submission that is spread over threads */
#define KTJ_STAGE_THREADS_MAX 4
#define KTJ_STAGE_SLOTS 16
static_assert(KTJ_STAGE_SLOTS >= 2 * KTJ_STAGE_THREADS_MAX, "two per copying thread");
/* Submissions between the ring and KTJ_STAGE_BIG_MIN, and documents on their way to the host, pass
 * through sixteen pinned slots of this size (the first part of the memory that large submissions use
 * whole): the copy engine works on some while the host fills or empties the others. */
#define KTJ_STAGE_SLOT (1ull << 20)
/* Working and document memory that waits for the next engine, per device: a five-hundredth of the card's
 * memory, enough for traces of a few hundred thousand records, which otherwise spend more time in
 * hipMalloc and hipFree than on the GPU.  It and the input arena are given back when KTJ_KIT_LEAN engines in
 * a row could have done with an eighth of them (above KTJ_KIT_SMALL_BYTES), when an allocation of this library
 * fails, and when the program asks for it (ktj_trim). */
#define KTJ_KIT_DEVICE_BYTES_MAX (512ull << 20)
#define KTJ_KIT_SMALL_BYTES (64ull << 20)
#define KTJ_KIT_LEAN 16u
#define KTJ_KIT_PINNED_BYTES_MAX (1ull << 20)  /* same, for the pinned copy of a document (ktj_output_host) */

bool drop_waiting_memory(); /* gives back what the current device's kit holds; true if that was anything */

std::atomic<int> g_failing_allocations{0}; /* ktj_debug_fail_allocations */
hipError_t allocate(void** p, size_t bytes) {
  if (g_failing_allocations.load(std::memory_order_relaxed) > 0 && g_failing_allocations.fetch_sub(1) > 0) return hipErrorOutOfMemory;
  return hipMalloc(p, bytes);
}

/* One working buffer in device memory.  `p` is what the kernels use: either the buffer's own
 * allocation (freed with the engine; the engine's device is current then) or, for the entry point
 * that allocates nothing, a borrowed range that somebody else owns (a piece of the library's static
 * scratch array, or the caller's output buffer).  The own allocation survives a borrow. */
struct DevBuf {
  void* p = nullptr;
  size_t cap = 0;
  void* own = nullptr;
  size_t own_cap = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  DevBuf& operator=(DevBuf&& o) noexcept {
    if (this != &o) { release(); p = o.p; cap = o.cap; own = o.own; own_cap = o.own_cap; o.p = o.own = nullptr; o.cap = o.own_cap = 0; }
    return *this;
  }
  ~DevBuf() { release(); }
  hipError_t ensure(size_t bytes, bool with_slack = true) {
    if (p != own) { p = own; cap = own_cap; } /* back from a borrowed range */
    if (bytes <= cap) return hipSuccess;
    if (own) { hipError_t e = hipFree(own); p = own = nullptr; cap = own_cap = 0; if (e != hipSuccess) return e; }
    size_t want = bytes + (with_slack ? bytes / 8 : 0) + 256;
    hipError_t e = allocate(&own, want);
    if (e == hipErrorOutOfMemory && drop_waiting_memory()) { (void)hipGetLastError(); e = allocate(&own, want); }
    if (e != hipSuccess) { p = own = nullptr; return e; }
    p = own;
    cap = own_cap = want;
    return hipSuccess;
  }
  void borrow(void* ptr, size_t bytes) { p = ptr; cap = bytes; }
  void unborrow() { p = own; cap = own_cap; }
  void release() { if (own) (void)hipFree(own); p = own = nullptr; cap = own_cap = 0; }
  template <typename T> T* as() const { return reinterpret_cast<T*>(p); }
};

/* Device memory for an engine's inputs: one allocation that its arrays are carved out of (a trace of
 * a few records otherwise spends more time in hipMalloc than on the GPU, a session of a few
 * megabytes as much as on its copies).  Pieces are never given back; a new engine that inherits the
 * arena starts at its beginning, and finds it large enough for what its predecessor asked for (as far as
 * KTJ_INPUT_ARENA_MAX goes; an engine whose kit had given the arena back does without). */
struct InputArena {
  DevBuf mem;
  size_t used = 0, missed = 0; /* missed: what it had no room for */
  void* take(size_t bytes) {
    const size_t off = (used + 255) & ~(size_t)255;
    if (!mem.p || off > mem.cap || bytes > mem.cap - off) {
      if (bytes <= KTJ_INPUT_ARENA_MAX) missed += bytes + 256;
      return nullptr;
    }
    used = off + bytes;
    return static_cast<char*>(mem.p) + off;
  }
  size_t asked() const { return used + missed; }
  size_t wanted() const { /* by an engine like this one, with some room to spare; 0: no more than there is */
    const size_t w = std::max<size_t>(std::min<size_t>(asked() + asked() / 4, KTJ_INPUT_ARENA_MAX), KTJ_INPUT_ARENA_BYTES);
    return asked() <= KTJ_INPUT_ARENA_MAX && (missed || !mem.p) && w > mem.cap ? w : 0;
  }
};

/* append-only device array fed from host memory */
struct DevVec {
  DevBuf buf;
  size_t bytes = 0;
  /* room for n more bytes behind what is there; what is there moves along.  A small array takes a
   * piece of the engine's input arena instead of an allocation of its own. */
  hipError_t reserve(size_t n, hipStream_t st, InputArena* arena) {
    if (bytes + n + 16 > buf.cap) { /* 16 spare bytes: string copies load whole aligned words */
      DevBuf nb;
      size_t want = (bytes + n) * 2 + 16;
      void* piece = arena ? arena->take(want) : nullptr;
      hipError_t e = hipSuccess;
      if (piece) nb.borrow(piece, want);
      else e = nb.ensure(want);
      if (e != hipSuccess) return e;
      if (bytes) {
        e = hipMemcpyAsync(nb.p, buf.p, bytes, hipMemcpyDeviceToDevice, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) return e;
      }
      buf = std::move(nb);
    }
    return hipSuccess;
  }
  char* end() const { return static_cast<char*>(buf.p) + bytes; }
  void release() { buf.release(); bytes = 0; }
};

struct RecordSet {
  DevVec owned;
  const void* external = nullptr; /* device pointer supplied by the caller */
  uint64_t n = 0;
  const void* ptr() const { return external ? external : owned.buf.p; }
};

/* read-backs of one pass land in pinned host memory (no staging inside the runtime) */
struct HostCtl {
  Scalars scalars;
  uint64_t act_bytes;
  uint32_t n_out;
  uint32_t weave;                                  /* plan_tables: KTJ_WEAVE_* of this pass */
  uint64_t end_clock;
  alignas(128) uint64_t part_flag[KTJ_PART_SLOTS]; /* copy_parts: what the slots hold */
};
#define KTJ_GUESS_BYTES_PER_ROW 480u /* the fixed text of an event with its flow event */
#define KTJ_PINNED_SMALL_BYTES (256u << 10) /* header/footer text and small tables of a pass that may not allocate */

enum { EV_START = 0, EV_EMIT, EV_COUNT };

}  // namespace

struct ktj_engine {
  std::string out_path, tmp_path, last_error;
  int64_t base_time_ns = 0;
  int device = 0;
  uint32_t flags = 0;
  FILE* sink = nullptr;
  bool bad_sink = false;
  bool started = false;
  bool processed = false;
  hipStream_t stream = nullptr;
  hipEvent_t ev[EV_COUNT] = {};
  hipEvent_t ev_d2h[2] = {};

  /* inputs */
  std::string txt_header, txt_before, txt_after; /* events in front of and behind the activity section, call order */
  bool activities_begun = false;
  DevVec str_blob, str_off; /* str_off holds n_strings + 1 absolute offsets */
  uint64_t n_strings = 0, blob_bytes = 0;
  std::vector<ktj_field> fields;
  std::vector<ktj_schema_desc> schemas;
  DevBuf d_fields, d_schemas;
  bool schemas_dirty = true;
  uint32_t schemas_not_taken = 0;          /* by the weaver, a bit each of the first */
  DevVec args;
  uint64_t n_args = 0;
  std::vector<CollectiveInfo> collectives; /* ktj_add_collective entries */
  bool coll_schemas = false;               /* a schema with a leading KTJ_F_COLLECTIVE field exists */
  bool coll_dirty = true;
  DevBuf d_coll_blob, d_coll_off, d_coll_first, cpu_row;
  /* GPU user annotations: correlation table, span table, finished spans, synthesised records */
  DevBuf u_keys, u_src, sp_hash, sp_first, sp_lo, sp_hi, sp_zero, sp_dev, sp_res, sp_ext, sp_name, sp_out, sp_count, sp_members,
      synth_recs;
  uint64_t n_spans = 0;
  std::vector<uint32_t> coll_first;        /* read back: first use of each entry per backend */
  std::unordered_map<uint64_t, int32_t> sdk_agents;        /* agent handle -> device index */
  std::unordered_map<uint64_t, uint32_t> sdk_kernel_names; /* kernel id -> string id of its name */
  uint32_t sdk_unknown_name = KTJ_NONE;
  std::vector<ktj_device_rec> sdk_rows;                    /* conversion buffer, reused */
  std::vector<ktj_runtime_rec> sdk_api_rows;               /* runtime rows of ktj_submit_sdk_api_record, not yet on the device */
  std::vector<ktj_extcorr_rec> sdk_api_ext, sdk_api_user;  /* their external-correlation pairs */
  std::vector<uint32_t> cid_names, flow_bits;
  uint32_t malloc_cid = KTJ_NONE;
  DevBuf d_cid_names, d_flow_bits;
  bool api_dirty = true;
  ktj_clock_model clock{};
  int64_t win_start = INT64_MIN, win_end = INT64_MAX;
  RecordSet generic, runtime, devrows, extcorr, usercorr;

  /* working buffers */
  DevBuf d_scalars, d_entries, d_name_blob, d_arg_blob;
  DevBuf c_ts, c_dur, c_corr, c_dev, c_res, c_meta, c_ext;
  DevBuf t_full, t_narrow, t_cpu, f_has_runtime, f_first, f_stream_src, f_pay, n_ext_src, n_kern_src, n_copy_src, n_pay, n_head, slot_f, slot_n, dev_link, dev_queue, sync_keys, sync_pos, sync_first;
  DevBuf q_keys, q_stream, q_amb, dn_hash, dn_first, dn_dev, dn_key, dn_rank, dn_list;
  DevBuf s_dev_k, s_dev_r, s_dev_l, s_res_k, s_res_r, s_res_l;
  DevBuf keys_a, keys_b, vals_a, vals_b, hist, scan_tmp;
  bool rows_are_text = false;              /* of the last pass: TextRows in mat */
  bool rows_with_sort = false;             /* likewise: the sort's last launch made rows as well */
  uint64_t not_woven = 0;                  /* number of these records with which a woven pass left too many activities (too_many_left) */
  int some_left = -1;                      /* the last woven pass had activities that the weaver leaves to emit_direct (1, 0; -1: there was none) */
  uint64_t pass_info[4] = {};              /* of the last pass (KTJ_DBG_PASS) */
  uint64_t sort_info[2] = {};              /* and KTJ_DBG_SORT */
  DevBuf mat, schema_book, wide_text, len, len_sorted, kind_sorted, offs, out, tile_start;
  void* pinned_small = nullptr; size_t pinned_small_cap = 0;
  HostCtl* h_ctl = nullptr;                  /* pinned: what the device hands back during a pass */
  HostCtl* h_ctl_dev = nullptr;              /* the same memory as the kernels address it */
  char* pinned_small_dev = nullptr;
  /* ktj_process_noalloc: working buffers are carved out of the library's static scratch array */
  bool noalloc = false;
  char* arena = nullptr; size_t arena_cap = 0, arena_used = 0;
  /* ktj_process: one allocation that the working buffers of a pass are carved out of */
  DevBuf pool;
  size_t pool_used = 0, pool_need = 0;
  bool measuring = false;
  char* pinned_out = nullptr; size_t pinned_out_cap = 0;
  bool host_copy_valid = false;
  /* submissions from ordinary host memory: small ones pass through a pinned ring and are not waited
   * for (the stream orders them before the pass), large ones through pinned chunks that several
   * threads fill while the copy engine empties others */
  InputArena input_arena;
  char* stage_small = nullptr; char* stage_small_dev = nullptr; size_t stage_small_used = 0;
  PieceJobs pieces{}; /* small submissions in the ring that no kernel has moved yet */
  char* stage_big = nullptr; char* stage_big_dev = nullptr; size_t stage_big_bytes = 0;
  uint64_t part_seq = 1; /* what the flags of the next document's parts count from */
  size_t stage_big_used = 0; /* of the slots' memory: uploads that the stream may not have passed yet */
  hipEvent_t ev_stage_big[KTJ_STAGE_SLOTS] = {};
  size_t most_needed = 0;    /* the largest pass's working memory and document */
  uint32_t kit_lean = 0; /* engines in a row, this kit's, that needed little of what it holds */
  bool hip_failed = false; /* a HIP call failed at some point: nothing of this engine is handed on */

  bool small_unfit = false;  /* these records need the launches of a large trace (Scalars::error of a small pass) */
  bool stepwise = false;     /* these records need a pass in which the host looks at the plan of the sort (KTJ_DEVERR_CAREFUL) */
  /* Not 0: all bits by passes, as the order of arrival is not that of the times where many are close together.  To find that out costs a
   * second sort and a wait (KTJ_DEVERR_UNSORTED; 10 000 rows 160 instead of 100 us, 2 million 930 instead of 750), and the next records of a
   * producer mostly come as these did: it is tried again for the 16th of them. */
  uint32_t sort_all_bits = 0;
  uint32_t sort_passes = 0;  /* what these records took in the pass before, where there was one */
  uint32_t sort_passes_most = 0; /* of others before them */
  void other_records() {
    small_unfit = stepwise = no_room_for_text = false; not_woven = 0;
    if (sort_all_bits && sort_passes) --sort_all_bits; /* (there was a pass since) */
    sort_passes_most = std::max(sort_passes_most, sort_passes); sort_passes = 0;
  }
  /* Six passes sort the records of one capture: 2^38 ns, four and a half minutes, beside 9 bits of devices and rows; four
   * do where the lowest sixteen of these 48 bits need none, as the word has room for them beside the index and the rows lie far enough apart.  A
   * pass more than needed costs its three launches, a pass too few the launches behind the sort. */
  uint32_t passes_to_launch(uint64_t n) const { return sort_passes ? sort_passes : std::max(sort_passes_most, n <= 65536u && !sort_all_bits ? 4u : 6u); }
  bool small_last = false;   /* the last pass was a small one: it leaves no intermediate arrays for ktj_debug_fetch */
  bool no_small = false;     /* ktj_debug_fetch makes them */
  bool no_weave = false;     /* joined rows as they are: ktj_debug_fetch */
  bool all_columns = false;  /* ktj_debug_fetch */
  bool columns_are_all = true; /* of the last pass: Columns::all */
  bool no_room_for_text = false; /* and where these records' text rows do not fit into memory */
  hipError_t hip_error = hipSuccess; /* of the last call that failed */
  int64_t last_end_time = 0;
  int wall_clock_khz = 0;

  /* results */
  uint64_t N = 0, prefix_len = 0, act_bytes = 0, total_bytes = 0;
  uint32_t* perm = nullptr; uint64_t* sorted_keys = nullptr;
  int sort_mode = 0; /* 0: key and index in one word; 1: (key, index) pairs */
  Scalars scalars{};
  ktj_stats stats{};
};

namespace {

int fail_hip(ktj_engine* e, hipError_t err, const char* what) {
  e->hip_failed = true;
  e->hip_error = err;
  e->last_error = std::string(what) + ": " + hipGetErrorString(err);
  return KTJ_ERR_HIP;
}
#define HIPCHK(call)                                            \
  do {                                                          \
    hipError_t _e = (call);                                     \
    if (_e != hipSuccess) return fail_hip(e, _e, #call);        \
  } while (0)

/* the ktj_last_error() text for the KTJ_DEVERR_* bits that end a pass */
std::string limit_text(unsigned bits) {
  std::string t;
  auto add = [&](const std::string& x) { t += (t.empty() ? "" : "; ") + x; };
  if (bits & KTJ_DEVERR_STREAMS)
    add("more than KTJ_MAX_STREAM_PAIRS (" + std::to_string(KTJ_MAX_STREAM_PAIRS) + ") distinct (device, stream) pairs among the device records");
  if (bits & KTJ_DEVERR_QUEUES)
    add("more than KTJ_MAX_QUEUES (" + std::to_string(KTJ_MAX_QUEUES) + ") distinct hardware queues among the device records");
  if (bits & KTJ_DEVERR_SYNC_ROWS)
    add("more than KTJ_MAX_SYNC_ROWS (" + std::to_string(KTJ_MAX_SYNC_ROWS) + ") distinct (device, row) pairs of Stream Sync activities");
  if (bits & KTJ_DEVERR_RECORD_TOO_LONG) add("an activity's JSON text is 1 GiB or longer");
  if (bits & KTJ_DEVERR_HASH_COLLISION) add("two (device, stream) pairs share a 64-bit hash");
  if (bits & KTJ_DEVERR_TABLE_FULL) add("a join table sized from the record counts is full (internal error)");
  if (bits & (KTJ_DEVERR_DISTINCT_DEVICES | KTJ_DEVERR_DISTINCT_RESOURCES)) add("distinct-value set overflow after the sort (internal error)");
  return "limit exceeded: " + t + " [bits " + std::to_string(bits) + "]";
}

uint32_t pow2_at_least(uint64_t v) {
  uint64_t c = 1024;
  while (c < v) c <<= 1;
  return (uint32_t)c;
}

/* Runs of sixteen slots that a join table of `cap` slots uses in hash mode, for `slots` slots as its records ask for: no more than these,
 * since all of them are cleared, read and missed in the caches, and a prime number, so that a key's steps reach them all.  Below 2^20 slots,
 * where clearing takes a microsecond and few runs fill unevenly, all that there are.  (11 million kernels of graphs, 17 instead of 33 million
 * slots: join stage 340 -> 285 us; 710 000 records of each class with ids of their own, tables two thirds full instead of one: 363 -> 340; 3
 * million: 2400 -> 2190.) */
uint32_t hash_runs(uint64_t slots, uint32_t cap) {
  uint64_t r = ((slots + 15u) / 16u) | 1u;
  for (bool prime = cap < (1u << 20); !prime;) {
    prime = true;
    for (uint64_t d = 3; d * d <= r; d += 2) if (r % d == 0) { prime = false; r += 2; break; }
  }
  return cap < (1u << 20) || r * 16u > cap ? cap / 16u : (uint32_t)r;
}

std::string default_file_name() { /* output_json.cpp:65-70, 481-483 */
  return "/tmp/libkineto_activities_" + std::to_string((long)getpid()) + ".json";
}

/* Room for `bytes` in a working buffer.  Normally the buffer grows by allocation; in a pass that
 * may not allocate it becomes the next piece of the scratch array (256-byte aligned), or the pass
 * fails with KTJ_ERR_LIMIT. */
int need(ktj_engine* e, DevBuf& b, size_t bytes) {
  if (!e->noalloc) {
    /* The working buffers of a pass share one allocation, the pool: a first pass then makes a handful
     * of allocations instead of sixty.  The pass first asks for everything with `measuring` set, which
     * only adds the sizes up, sizes the pool, and asks again.  What does not fit (buffers whose size a
     * pass learns late) is allocated on its own as before. */
    if (e->measuring) { e->pool_need += (bytes + 255) & ~(size_t)255; return KTJ_OK; }
    const size_t off = (e->pool_used + 255) & ~(size_t)255;
    if (e->pool.p && off <= e->pool.cap && bytes <= e->pool.cap - off) {
      b.borrow(static_cast<char*>(e->pool.p) + off, bytes);
      e->pool_used = off + bytes;
      return KTJ_OK;
    }
    HIPCHK(b.ensure(bytes));
    return KTJ_OK;
  }
  const size_t off = (e->arena_used + 255) & ~(size_t)255;
  if (off > e->arena_cap || bytes > e->arena_cap - off) {
    e->last_error = "ktj_process_noalloc: the trace needs more than the " + std::to_string(e->arena_cap) +
                    " bytes of the static scratch array (asked for " + std::to_string(bytes) + " more at " + std::to_string(off) + ")";
    return KTJ_ERR_LIMIT;
  }
  b.borrow(e->arena + off, bytes);
  e->arena_used = off + bytes;
  return KTJ_OK;
}
#define NEED(buf, bytes)                                  \
  do {                                                    \
    const int _rc = need(e, buf, bytes);                  \
    if (_rc != KTJ_OK) return _rc;                        \
  } while (0)

/* The small submissions gathered in the pinned ring go to their places on the device: one launch for
 * all of them, ordered on the engine's stream like everything else.  Before a pass, before an array
 * they belong to moves, and when the ring or the list is full. */
int put_pending_pieces(ktj_engine* e) {
  if (e->pieces.count == 0) return KTJ_OK;
  HIPCHK(put_pieces(e->pieces, e->stream));
  e->pieces.count = 0;
  return KTJ_OK;
}

/* Is this host memory page-locked for the GPU (ktj_host_alloc, or the caller's own hipHostMalloc)?
 * Such memory is copied from directly. */
bool is_pinned_host(const void* p) {
  hipPointerAttribute_t a;
  memset(&a, 0, sizeof a);
  if (hipPointerGetAttributes(&a, p) != hipSuccess) { (void)hipGetLastError(); return false; }
  return a.type == hipMemoryTypeHost;
}

/* n bytes into the pinned ring of small submissions, to be moved to dst by the next put_pending_pieces;
 * n <= KTJ_STAGE_SMALL_MAX */
int stage_piece(ktj_engine* e, void* dst, const void* src, size_t n) {
  /* the piece sits in the ring where its place on the device does, modulo 16 */
  size_t off = ((e->stage_small_used + 63) & ~(size_t)63) + ((uintptr_t)dst & 15u);
  if (off + n > KTJ_STAGE_SMALL_BYTES || e->pieces.count == KTJ_MAX_PIECES) {
    const int rc = put_pending_pieces(e);
    if (rc != KTJ_OK) return rc;
  }
  if (off + n > KTJ_STAGE_SMALL_BYTES) { /* the ring is full: what is in it has to be on the device first */
    HIPCHK(hipStreamSynchronize(e->stream));
    off = (uintptr_t)dst & 15u;
  }
  memcpy(e->stage_small + off, src, n);
  const uint32_t k = e->pieces.count++;
  e->pieces.src[k] = e->stage_small_dev + off;
  e->pieces.dst[k] = static_cast<char*>(dst);
  e->pieces.n[k] = n;
  e->stage_small_used = off + n;
  return KTJ_OK;
}

/* The pinned slots: at least `bytes` of memory (kept with the kit). */
int ensure_stage(ktj_engine* e, size_t bytes) {
  if (e->stage_big_bytes < bytes) {
    if (e->stage_big) { HIPCHK(hipStreamSynchronize(e->stream)); HIPCHK(hipHostFree(e->stage_big)); }
    e->stage_big = nullptr; e->stage_big_bytes = 0; e->stage_big_used = 0;
    void* p = nullptr;
    HIPCHK(hipHostMalloc(&p, bytes, hipHostMallocDefault));
    e->stage_big = static_cast<char*>(p);
    e->stage_big_bytes = bytes;
    HIPCHK(hipHostGetDevicePointer(&p, e->stage_big, 0));
    e->stage_big_dev = static_cast<char*>(p);
  }
  for (auto& ev : e->ev_stage_big)
    if (!ev) HIPCHK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
  return KTJ_OK;
}

/* uploads out of the slots are on their way: everything else that uses the slots waits for them */
int drain_stage(ktj_engine* e) {
  if (e->stage_big_used) { HIPCHK(hipStreamSynchronize(e->stream)); e->stage_big_used = 0; }
  return KTJ_OK;
}

/* Runs worker(0 .. n_threads - 1), worker 0 on the calling thread; a thread that cannot be started
 * has its share done by the caller. */
template <typename Worker> void run_workers(unsigned n_threads, Worker worker) {
  std::vector<std::thread> pool;
  unsigned started = 1;
  try {
    pool.reserve(n_threads);
    for (; started < n_threads; ++started) pool.emplace_back(worker, started);
  } catch (...) {}
  worker(0);
  for (unsigned t = started; t < n_threads; ++t) worker(t);
  for (auto& th : pool) th.join();
}
unsigned copy_threads(size_t bytes, size_t per_thread, unsigned most) {
  unsigned n = std::thread::hardware_concurrency() / 2;
  if (n > most) n = most;
  if (n > bytes / per_thread) n = (unsigned)(bytes / per_thread);
  return n ? n : 1;
}

/* n bytes of host memory behind a device array.  The caller may free or reuse src when this
 * returns; the copy itself is only ordered on the engine's stream, in front of the next pass.
 *   - up to KTJ_STAGE_SMALL_MAX bytes: into the pinned ring, from where one kernel launch takes all
 *     such pieces to their places (put_pending_pieces; a trace of a few records pays a dozen copies
 *     and stream synchronisations otherwise);
 *   - below KTJ_STAGE_BIG_MIN bytes of ordinary memory: part by part into the pinned slots and on to
 *     the copy engine, not waited for (a copy from ordinary memory is waited for by the runtime, with
 *     nothing overlapped: a session of 30 000 records, 2.8 MB in five arrays, submits in 262 us that way);
 *   - above: threads copy chunks into pinned buffers, two per thread, and hand each to the copy
 *     engine as soon as it is full (one thread's copy through the runtime's own staging reaches about
 *     half of what the link carries);
 *   - page-locked sources: one copy, waited for. */
int append_from_host(ktj_engine* e, DevVec& v, const void* src, size_t n) {
  if (n == 0) return KTJ_OK;
  hipStream_t st = e->stream;
  if (v.bytes + n + 16 > v.buf.cap) { /* the array is about to move: the pieces on their way to it go first */
    const int rc = put_pending_pieces(e);
    if (rc != KTJ_OK) return rc;
  }
  HIPCHK(v.reserve(n, st, &e->input_arena));
  char* dst = v.end();
  if (n <= KTJ_STAGE_SMALL_MAX && e->stage_small) {
    const int rc = stage_piece(e, dst, src, n);
    if (rc != KTJ_OK) return rc;
    v.bytes += n;
    return KTJ_OK;
  }
  if (is_pinned_host(src)) {
    HIPCHK(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, st));
    HIPCHK(hipStreamSynchronize(st)); /* the caller may free src when we return */
    v.bytes += n;
    return KTJ_OK;
  }
  const unsigned n_threads = copy_threads(n, KTJ_STAGE_CHUNK, KTJ_STAGE_THREADS_MAX);
  if (n >= KTJ_STAGE_BIG_MIN && n_threads >= 2) {
    int rc = drain_stage(e);
    if (rc == KTJ_OK) rc = ensure_stage(e, 2 * KTJ_STAGE_THREADS_MAX * KTJ_STAGE_CHUNK);
    if (rc != KTJ_OK) return rc;
    const size_t n_chunks = (n + KTJ_STAGE_CHUNK - 1) / KTJ_STAGE_CHUNK;
    hipError_t err[KTJ_STAGE_THREADS_MAX];
    for (auto& x : err) x = hipSuccess;
    run_workers(n_threads, [&](unsigned t) {
      err[t] = hipSetDevice(e->device);
      /* thread t takes chunks t, t + T, ...; its two pinned slots alternate */
      for (size_t c = t, turn = 0; c < n_chunks && err[t] == hipSuccess; c += n_threads, ++turn) {
        const size_t slot = 2 * (size_t)t + (turn & 1);
        char* stage = e->stage_big + slot * KTJ_STAGE_CHUNK;
        const size_t off = c * KTJ_STAGE_CHUNK, len = n - off < KTJ_STAGE_CHUNK ? n - off : KTJ_STAGE_CHUNK;
        if (turn >= 2) { err[t] = hipEventSynchronize(e->ev_stage_big[slot]); if (err[t] != hipSuccess) break; }
        memcpy(stage, static_cast<const char*>(src) + off, len);
        err[t] = hipMemcpyAsync(dst + off, stage, len, hipMemcpyHostToDevice, st);
        if (err[t] == hipSuccess) err[t] = hipEventRecord(e->ev_stage_big[slot], st);
      }
    });
    /* the slots are free for the next call once the stream has passed them */
    const hipError_t done = hipStreamSynchronize(st);
    for (unsigned t = 0; t < n_threads; ++t) HIPCHK(err[t]);
    HIPCHK(done);
    v.bytes += n;
    return KTJ_OK;
  }
  {
    const int rc = ensure_stage(e, KTJ_STAGE_SLOTS * KTJ_STAGE_SLOT);
    if (rc != KTJ_OK) return rc;
  }
  for (size_t done = 0; done < n;) {
    if (e->stage_big_used == e->stage_big_bytes) { /* all slots are full: wait until the stream has passed them */
      const int rc = drain_stage(e);
      if (rc != KTJ_OK) return rc;
    }
    const size_t len = std::min(std::min<size_t>(n - done, KTJ_STAGE_SLOT), e->stage_big_bytes - e->stage_big_used);
    char* stage = e->stage_big + e->stage_big_used;
    memcpy(stage, static_cast<const char*>(src) + done, len);
    HIPCHK(hipMemcpyAsync(dst + done, stage, len, hipMemcpyHostToDevice, st));
    e->stage_big_used = std::min((e->stage_big_used + len + 255) & ~(size_t)255, e->stage_big_bytes);
    done += len;
  }
  v.bytes += n;
  return KTJ_OK;
}

/* A small host table to the device, in front of the pass that is about to start. */
int upload_small(ktj_engine* e, DevBuf& dst, const void* src, size_t bytes) {
  const size_t room = bytes ? bytes : 16;
  if (e->noalloc) {
    NEED(dst, room);
    if (bytes > e->pinned_small_cap) {
      e->last_error = "ktj_process_noalloc: a table of " + std::to_string(bytes) + " bytes exceeds the pinned staging buffer";
      return KTJ_ERR_LIMIT;
    }
  } else if (!dst.p || dst.cap < room) {
    /* these tables outlive the pass (they are uploaded only when they change), so they are pieces of
     * the engine's input memory and not of the pass's pool */
    void* piece = e->input_arena.take(room + room / 2);
    if (piece) dst.borrow(piece, room + room / 2);
    else HIPCHK(dst.ensure(room));
  }
  if (bytes == 0) return KTJ_OK;
  if (bytes <= KTJ_STAGE_SMALL_MAX) return stage_piece(e, dst.p, src, bytes);
  if (e->noalloc) { memcpy(e->pinned_small, src, bytes); src = e->pinned_small; } /* not the runtime's own staging */
  HIPCHK(hipMemcpyAsync(dst.p, src, bytes, hipMemcpyHostToDevice, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  return KTJ_OK;
}

int bits_for(uint64_t max_value) { /* bits needed to hold values 0..max_value */
  int b = 0;
  while (b < 64 && (max_value >> b) != 0) ++b;
  return b;
}

/* GPU user annotations (GenericActivityProfiler.cpp:277-327, 423-433, 726).  The device groups the
 * in-window device rows by (device, resource, annotation) and reduces each group to its extent;
 * the host puts the finished spans into the order the profiler logs them in — stream by stream
 * (std::map), inside a stream the iteration order of a std::unordered_map keyed by the
 * annotation's id, both filled in the order of the spans' first rows — and hands them back as
 * generic records of type GPU_USER_ANNOTATION whose rows follow the device rows. */
int synthesise_user_spans(ktj_engine* e, Columns c, const EmitCtx& ctx, Table t_cpu, const uint32_t* cpu_row, Scalars* sc,
                          uint64_t first_row) {
  hipStream_t st = e->stream;
  const uint64_t ng = e->generic.n, nr = e->runtime.n, nd = e->devrows.n, nu = e->usercorr.n;
  const ktj_generic_rec* g_recs = static_cast<const ktj_generic_rec*>(e->generic.ptr());
  const ktj_extcorr_rec* u_recs = static_cast<const ktj_extcorr_rec*>(e->usercorr.ptr());
  const uint32_t cap_user = pow2_at_least(2 * nu), cap_span = pow2_at_least(2 * nd);
  NEED(e->u_keys, (cap_user + 1ull) * 8); NEED(e->u_src, (cap_user + 1ull) * 4);
  NEED(e->sp_hash, (cap_span + 1ull) * 8); NEED(e->sp_first, (cap_span + 1ull) * 4);
  NEED(e->sp_lo, (cap_span + 1ull) * 8); NEED(e->sp_hi, (cap_span + 1ull) * 8);
  NEED(e->sp_zero, (cap_span + 1ull) * 4); NEED(e->sp_dev, (cap_span + 1ull) * 4);
  NEED(e->sp_res, (cap_span + 1ull) * 8); NEED(e->sp_ext, (cap_span + 1ull) * 8);
  NEED(e->sp_name, (cap_span + 1ull) * 4); NEED(e->sp_out, (nd + 1ull) * sizeof(SpanOut));
  NEED(e->sp_count, 16);
  SpanTables t{e->u_keys.as<uint64_t>(), e->u_src.as<uint32_t>(), cap_user - 1,
               e->sp_hash.as<uint64_t>(), e->sp_first.as<uint32_t>(), e->sp_lo.as<uint64_t>(), e->sp_hi.as<uint64_t>(),
               e->sp_zero.as<uint32_t>(), cap_span - 1,
               e->sp_dev.as<int32_t>(), e->sp_res.as<int64_t>(), e->sp_ext.as<uint64_t>(), e->sp_name.as<uint32_t>()};
  HIPCHK(fill_u64(t.u_keys, KTJ_EMPTY_KEY, cap_user + 1ull, st)); HIPCHK(fill_u32(t.u_src, 0, cap_user + 1ull, st));
  HIPCHK(fill_u64(t.hash, KTJ_EMPTY_KEY, cap_span + 1ull, st)); HIPCHK(fill_u32(t.first, 0xFFFFFFFFu, cap_span + 1ull, st));
  HIPCHK(fill_u64(t.lo, ~0ull, cap_span + 1ull, st)); HIPCHK(fill_u64(t.hi, 0, cap_span + 1ull, st));
  HIPCHK(fill_u32(t.zero, 0, cap_span + 1ull, st));
  HIPCHK(build_usercorr(u_recs, nu, t, sc, st));
  HIPCHK(group_spans(u_recs, g_recs, nd, c, ng + nr, t_cpu, cpu_row, t, e->sp_out.as<SpanOut>(), e->sp_count.as<uint32_t>(), sc, st));
  HIPCHK(hipMemcpyAsync(&e->h_ctl->n_out, e->sp_count.p, 4, hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  const uint32_t n_out = e->h_ctl->n_out;
  if (n_out == 0) return KTJ_OK;
  std::vector<SpanOut> spans(n_out);
  HIPCHK(hipMemcpyAsync(spans.data(), e->sp_out.p, n_out * sizeof(SpanOut), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  std::sort(spans.begin(), spans.end(), [](const SpanOut& a, const SpanOut& b) { return a.first < b.first; });

  /* insertOrExtendEvent's start rule is `if (ts < start || start == 0) start = ts` (:304-306): the
   * plain minimum unless a row of the span starts at time 0, after which the next row's time is
   * taken whatever it is.  Those spans (rare) are replayed row by row here. */
  bool any_zero = false;
  for (const SpanOut& sp : spans) any_zero = any_zero || sp.zero != 0;
  if (any_zero) {
    NEED(e->sp_members, (nd + 1ull) * sizeof(SpanMember));
    HIPCHK(span_members(u_recs, nd, c, ng + nr, t_cpu, t, e->sp_members.as<SpanMember>(), (uint32_t)nd, e->sp_count.as<uint32_t>(), st));
    HIPCHK(hipMemcpyAsync(&e->h_ctl->n_out, e->sp_count.p, 4, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    const uint32_t n_members = e->h_ctl->n_out;
    std::vector<SpanMember> members(n_members);
    if (n_members) HIPCHK(hipMemcpyAsync(members.data(), e->sp_members.p, n_members * sizeof(SpanMember), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    std::sort(members.begin(), members.end(), [](const SpanMember& a, const SpanMember& b) { return a.row < b.row; });
    std::unordered_map<uint32_t, size_t> by_slot;
    for (size_t k = 0; k < spans.size(); ++k)
      if (spans[k].zero) by_slot[spans[k].zero] = k;
    std::vector<uint8_t> started(spans.size(), 0);
    for (const SpanMember& m : members) {
      const auto it = by_slot.find(m.slot);
      if (it == by_slot.end()) continue;
      SpanOut& sp = spans[it->second];
      if (!started[it->second]) { started[it->second] = 1; sp.start = m.ts; }
      if (m.ts < sp.start || sp.start == 0) sp.start = m.ts;
    }
  }

  /* logEvents order (:313-319) */
  std::map<std::pair<int64_t, int64_t>, std::unordered_map<int64_t, size_t>> streams;
  for (size_t k = 0; k < spans.size(); ++k)
    streams[{(int64_t)spans[k].dev, spans[k].res}].insert({(int64_t)spans[k].ext, k});
  std::vector<ktj_generic_rec> recs;
  recs.reserve(spans.size());
  for (const auto& stream : streams) {
    for (const auto& entry : stream.second) {
      const SpanOut& sp = spans[entry.second];
      ktj_generic_rec r{}; /* createUserGpuSpan (:277-290): no metadata, no flow, no linked activity */
      r.start_ns = sp.start;
      r.end_ns = sp.end;
      r.resource = sp.res;
      r.device = sp.dev;
      r.id = (int32_t)(int64_t)sp.ext;
      r.name_id = sp.name;
      r.schema_id = KTJ_NONE;
      r.type = KTJ_TYPE_GPU_USER_ANNOTATION;
      recs.push_back(r);
    }
  }
  NEED(e->synth_recs, recs.size() * sizeof(ktj_generic_rec) + 16);
  HIPCHK(hipMemcpyAsync(e->synth_recs.p, recs.data(), recs.size() * sizeof(ktj_generic_rec), hipMemcpyHostToDevice, st));
  HIPCHK(hipStreamSynchronize(st));
  DecodeJob job;
  memset(&job, 0, sizeof job);
  job.g = e->synth_recs.as<ktj_generic_rec>(); job.ng = recs.size(); job.first = first_row;
  HIPCHK(decode(job, c, ctx, sc, st));
  e->n_spans = recs.size();
  return KTJ_OK;
}


/* What every engine needs before its first record — a stream, its events, the pinned buffers of the
 * hand-over, the input arena — and what its first pass allocates (the pool of working buffers and
 * the document, while they are small) costs several times what a trace of a few records takes on
 * the GPU.  ktj_destroy leaves one such set per device behind for the next ktj_create, which takes
 * it whole; a second engine alive at the same time makes its own.  Nothing of an engine that saw a
 * HIP error is kept.  What is kept until the process ends: the stream, the events, Scalars and the small
 * pinned buffers, at most 2.5 MiB.  What may be given back before (see KTJ_KIT_LEAN): at most
 * KTJ_KIT_DEVICE_BYTES_MAX of working and document memory, the input arena, KTJ_INPUT_ARENA_MAX at most, and,
 * by ktj_trim only, the pinned slots, 16 or 64 MiB. */
struct Kit {
  bool full = false;
  hipStream_t stream = nullptr;
  hipEvent_t ev[EV_COUNT] = {};
  hipEvent_t ev_d2h[2] = {};
  hipEvent_t ev_stage_big[KTJ_STAGE_SLOTS] = {};
  uint32_t lean = 0;
  void* pinned_small = nullptr; size_t pinned_small_cap = 0; char* pinned_small_dev = nullptr;
  HostCtl* h_ctl = nullptr; HostCtl* h_ctl_dev = nullptr;
  char* pinned_out = nullptr; size_t pinned_out_cap = 0;
  char* stage_small = nullptr; char* stage_small_dev = nullptr;
  char* stage_big = nullptr; char* stage_big_dev = nullptr; size_t stage_big_bytes = 0;
  DevBuf d_scalars, pool, out, arena_mem;
};
std::mutex g_kit_mutex;
std::map<int, Kit*>& kits() { static auto* m = new std::map<int, Kit*>(); return *m; } /* never destroyed: the runtime may be gone by then */

/* the kit's device is current, its mutex held */
bool drop_device_memory(Kit& k) {
  const bool any = k.pool.own_cap + k.out.own_cap + k.arena_mem.own_cap != 0;
  k.pool.release();
  k.out.release();
  k.arena_mem.release();
  return any;
}
bool drop_waiting_memory() {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return false;
  std::lock_guard<std::mutex> lock(g_kit_mutex);
  auto it = kits().find(device);
  return it != kits().end() && it->second->full && drop_device_memory(*it->second);
}

/* the engine's device is current */
bool take_kit(ktj_engine* e) {
  std::lock_guard<std::mutex> lock(g_kit_mutex);
  auto it = kits().find(e->device);
  if (it == kits().end() || !it->second->full) return false;
  Kit& k = *it->second;
  e->stream = k.stream;
  memcpy(e->ev, k.ev, sizeof k.ev); memcpy(e->ev_d2h, k.ev_d2h, sizeof k.ev_d2h);
  memcpy(e->ev_stage_big, k.ev_stage_big, sizeof k.ev_stage_big);
  e->kit_lean = k.lean;
  e->pinned_small = k.pinned_small; e->pinned_small_cap = k.pinned_small_cap; e->pinned_small_dev = k.pinned_small_dev;
  e->h_ctl = k.h_ctl; e->h_ctl_dev = k.h_ctl_dev;
  e->pinned_out = k.pinned_out; e->pinned_out_cap = k.pinned_out_cap;
  e->stage_small = k.stage_small; e->stage_small_dev = k.stage_small_dev;
  e->stage_big = k.stage_big; e->stage_big_dev = k.stage_big_dev; e->stage_big_bytes = k.stage_big_bytes;
  e->d_scalars = std::move(k.d_scalars); e->pool = std::move(k.pool); e->out = std::move(k.out);
  e->input_arena.mem = std::move(k.arena_mem);
  k = Kit();
  return true;
}

/* the engine's device is current and its stream is idle; whatever is not taken stays with the engine */
void give_kit(ktj_engine* e) {
  if (e->hip_failed || !e->stream || !e->h_ctl || !e->pinned_small || !e->stage_small || !e->d_scalars.own) return;
  if (e->pinned_small_cap > KTJ_KIT_PINNED_BYTES_MAX) return; /* grown for an unusually long header: not worth holding */
  for (auto& ev : e->ev) if (!ev) return;
  for (auto& ev : e->ev_d2h) if (!ev) return;
  /* back from whatever they were lent (the pool never is; the document may sit in a caller's buffer) */
  e->pool.unborrow();
  e->out.unborrow();
  const size_t held = e->pool.own_cap + e->out.own_cap + e->input_arena.mem.own_cap;
  if (held > KTJ_KIT_SMALL_BYTES && e->most_needed + e->input_arena.asked() < held / 8) {
    if (++e->kit_lean >= KTJ_KIT_LEAN) { e->pool.release(); e->out.release(); e->input_arena.mem.release(); e->kit_lean = 0; }
  } else e->kit_lean = 0;
  if (const size_t want = e->input_arena.wanted()) { /* room for the inputs of another engine like this one */
    e->input_arena.mem.release();
    if (e->input_arena.mem.ensure(want - 256, false) != hipSuccess) (void)hipGetLastError(); /* ensure adds 256 */
  }
  std::lock_guard<std::mutex> lock(g_kit_mutex);
  Kit* slot = nullptr;
  try {
    Kit*& entry = kits()[e->device];
    if (!entry) entry = new Kit();
    slot = entry;
  } catch (...) { return; }
  if (slot->full) return;
  Kit& k = *slot;
  k.stream = e->stream; e->stream = nullptr;
  memcpy(k.ev, e->ev, sizeof k.ev); memset(e->ev, 0, sizeof e->ev);
  memcpy(k.ev_d2h, e->ev_d2h, sizeof k.ev_d2h); memset(e->ev_d2h, 0, sizeof e->ev_d2h);
  k.lean = e->kit_lean;
  memcpy(k.ev_stage_big, e->ev_stage_big, sizeof k.ev_stage_big); memset(e->ev_stage_big, 0, sizeof e->ev_stage_big);
  k.pinned_small = e->pinned_small; k.pinned_small_cap = e->pinned_small_cap; k.pinned_small_dev = e->pinned_small_dev;
  e->pinned_small = nullptr;
  k.h_ctl = e->h_ctl; k.h_ctl_dev = e->h_ctl_dev; e->h_ctl = nullptr;
  if (e->pinned_out_cap <= KTJ_KIT_PINNED_BYTES_MAX) { k.pinned_out = e->pinned_out; k.pinned_out_cap = e->pinned_out_cap; e->pinned_out = nullptr; }
  k.stage_small = e->stage_small; k.stage_small_dev = e->stage_small_dev; e->stage_small = nullptr;
  k.stage_big = e->stage_big; k.stage_big_dev = e->stage_big_dev; k.stage_big_bytes = e->stage_big_bytes; e->stage_big = nullptr;
  k.d_scalars = std::move(e->d_scalars);
  if (e->pool.own_cap + e->out.own_cap <= KTJ_KIT_DEVICE_BYTES_MAX) {
    k.pool = std::move(e->pool);
    k.out = std::move(e->out);
  }
  k.arena_mem = std::move(e->input_arena.mem);
  k.full = true;
}

}  // namespace

extern "C" {

const char* ktj_version(void) { return "ktj 0.1 (gfx950)"; }

int ktj_create(ktj_engine** out, const char* out_path, int64_t base_time_ns, int hip_device, uint32_t flags) {
  if (!out) return KTJ_ERR_ARG;
  *out = nullptr;
  ktj_engine* e = new (std::nothrow) ktj_engine();
  if (!e) return KTJ_ERR_NOMEM;
  e->out_path = (out_path && out_path[0]) ? out_path : default_file_name();
  e->tmp_path = e->out_path + ".tmp";
  e->base_time_ns = base_time_ns;
  e->device = hip_device;
  e->flags = flags;
  e->sort_mode = (flags & KTJ_CREATE_PAIR_SORT) ? 1 : 0;
  e->clock.scale = 1.0;
  *out = e; /* from here on errors are reported through the handle */
  if (!(flags & KTJ_CREATE_NO_FILE)) { /* openTraceFile, output_json.cpp:485-493 */
    e->sink = fopen(e->tmp_path.c_str(), "w");
    if (!e->sink) { e->bad_sink = true; e->last_error = "Failed to open '" + e->out_path + "': " + strerror(errno); }
  }
  HIPCHK(hipSetDevice(hip_device));
  if (!take_kit(e)) {
    HIPCHK(hipStreamCreate(&e->stream));
    for (auto& ev : e->ev) HIPCHK(hipEventCreate(&ev));
    for (auto& ev : e->ev_d2h) HIPCHK(hipEventCreate(&ev));
    HIPCHK(e->d_scalars.ensure(sizeof(Scalars)));
    HIPCHK(hipHostMalloc(&e->pinned_small, KTJ_PINNED_SMALL_BYTES, hipHostMallocDefault));
    e->pinned_small_cap = KTJ_PINNED_SMALL_BYTES;
    void* p = nullptr;
    HIPCHK(hipHostMalloc(&p, sizeof(HostCtl), hipHostMallocDefault));
    e->h_ctl = static_cast<HostCtl*>(p);
    void* d = nullptr;
    HIPCHK(hipHostGetDevicePointer(&d, e->h_ctl, 0));
    e->h_ctl_dev = static_cast<HostCtl*>(d);
    HIPCHK(hipHostGetDevicePointer(&d, e->pinned_small, 0));
    e->pinned_small_dev = static_cast<char*>(d);
    p = nullptr;
    HIPCHK(hipHostMalloc(&p, KTJ_STAGE_SMALL_BYTES, hipHostMallocDefault));
    e->stage_small = static_cast<char*>(p);
    HIPCHK(hipHostGetDevicePointer(&d, e->stage_small, 0));
    e->stage_small_dev = static_cast<char*>(d);
  }
  if (!e->input_arena.mem.p) HIPCHK(e->input_arena.mem.ensure(KTJ_INPUT_ARENA_BYTES, false));
  memset(e->h_ctl, 0, sizeof(HostCtl));
  { /* this device's copy of the static scratch array (ktj_process_noalloc) */
    void* p = nullptr;
    size_t bytes = 0;
    HIPCHK(scratch_address(hip_device, &p, &bytes));
    e->arena = static_cast<char*>(p);
    e->arena_cap = bytes;
  }
  return KTJ_OK;
}

void ktj_destroy(ktj_engine* e) {
  if (!e) return;
  (void)hipSetDevice(e->device);
  if (e->stream) (void)hipStreamSynchronize(e->stream);
  give_kit(e); /* what the next engine on this device can start from; the rest is freed here */
  /* device buffers free themselves when the engine is deleted below */
  if (e->pinned_small) (void)hipHostFree(e->pinned_small);
  if (e->h_ctl) (void)hipHostFree(e->h_ctl);
  if (e->pinned_out) (void)hipHostFree(e->pinned_out);
  if (e->stage_small) (void)hipHostFree(e->stage_small);
  if (e->stage_big) (void)hipHostFree(e->stage_big);
  for (auto& ev : e->ev_stage_big) if (ev) (void)hipEventDestroy(ev);
  for (auto& ev : e->ev) if (ev) (void)hipEventDestroy(ev);
  for (auto& ev : e->ev_d2h) if (ev) (void)hipEventDestroy(ev);
  if (e->stream) (void)hipStreamDestroy(e->stream);
  if (e->sink) { fclose(e->sink); remove(e->tmp_path.c_str()); }
  delete e;
}

int ktj_trim(int hip_device) {
  int current = 0;
  if (hipGetDevice(&current) != hipSuccess) return KTJ_ERR_HIP;
  std::lock_guard<std::mutex> lock(g_kit_mutex);
  auto it = kits().find(hip_device);
  if (it == kits().end() || !it->second->full) return KTJ_OK;
  if (hipSetDevice(hip_device) != hipSuccess) return KTJ_ERR_HIP;
  Kit& k = *it->second;
  (void)drop_device_memory(k);
  hipError_t err = k.stage_big ? hipHostFree(k.stage_big) : hipSuccess;
  k.stage_big = k.stage_big_dev = nullptr;
  k.stage_big_bytes = 0;
  if (err == hipSuccess) err = hipSetDevice(current);
  return err == hipSuccess ? KTJ_OK : KTJ_ERR_HIP;
}

const char* ktj_last_error(const ktj_engine* e) { return e ? e->last_error.c_str() : "null engine"; }

int ktj_trace_start(ktj_engine* e, const char* const* meta_kv, size_t n_kv, const char* device_properties) {
  if (!e || (n_kv && !meta_kv)) return KTJ_ERR_ARG;
  if (e->bad_sink) return KTJ_OK;
  e->txt_header.clear();
  append_trace_start(e->txt_header, meta_kv, n_kv, device_properties, e->base_time_ns, (e->flags & KTJ_CREATE_DISPLAY_NS) != 0);
  e->started = true;
  e->processed = false;
  return KTJ_OK;
}

int ktj_intern_strings(ktj_engine* e, const char* blob, const uint64_t* offsets, size_t n, uint32_t* first_id) {
  if (!e || (n && (!blob || !offsets))) return KTJ_ERR_ARG;
  if (first_id) *first_id = (uint32_t)e->n_strings;
  if (e->bad_sink || n == 0) return KTJ_OK;
  if (e->n_strings + n >= KTJ_NONE) return KTJ_ERR_LIMIT;
  HIPCHK(hipSetDevice(e->device));
  const uint64_t src0 = offsets[0], nbytes = offsets[n] - offsets[0];
  std::vector<uint64_t> abs_off(n + 1);
  for (size_t i = 0; i <= n; ++i) {
    if (offsets[i] < src0 || (i && offsets[i] < offsets[i - 1])) return KTJ_ERR_ARG;
    abs_off[i] = e->blob_bytes + (offsets[i] - src0);
  }
  { const int rc = append_from_host(e, e->str_blob, blob + src0, nbytes); if (rc != KTJ_OK) return rc; }
  {
    /* entry n_strings already equals blob_bytes */
    const int rc = e->n_strings == 0 ? append_from_host(e, e->str_off, abs_off.data(), (n + 1) * 8)
                                     : append_from_host(e, e->str_off, abs_off.data() + 1, n * 8);
    if (rc != KTJ_OK) return rc;
  }
  e->n_strings += n;
  e->blob_bytes += nbytes;
  e->processed = false;
  return KTJ_OK;
}

int ktj_register_schema(ktj_engine* e, const ktj_field* f, size_t n_fields, uint32_t* schema_id) {
  if (!e || (n_fields && !f)) return KTJ_ERR_ARG;
  if (n_fields > KTJ_MAX_SCHEMA_FIELDS) return KTJ_ERR_LIMIT;
  int depth = 0;
  for (size_t i = 0; i < n_fields; ++i) {
    const uint16_t t = f[i].type;
    if (t > KTJ_F_UNSUPPORTED) return KTJ_ERR_ARG;
    const bool no_slots = t == KTJ_F_DICT_BEGIN || t == KTJ_F_DICT_END || t == KTJ_F_UNSUPPORTED;
    const bool array = t == KTJ_F_I64_ARRAY || t == KTJ_F_STR_ARRAY;
    if (no_slots ? f[i].count != 0 : array ? false : f[i].count != 1) return KTJ_ERR_ARG; /* arrays may be empty */
    if ((t == KTJ_F_DICT_BEGIN || t == KTJ_F_UNSUPPORTED) && f[i].key_id == KTJ_NONE) return KTJ_ERR_ARG;
    if (t == KTJ_F_DICT_BEGIN) ++depth;
    if (t == KTJ_F_DICT_END && --depth < 0) return KTJ_ERR_ARG;
  }
  if (depth != 0) return KTJ_ERR_ARG; /* every dict is closed */
  if (n_fields && f[0].type == KTJ_F_COLLECTIVE) e->coll_schemas = true;
  ktj_schema_desc d;
  d.first_field = (uint32_t)e->fields.size();
  d.n_fields = (uint32_t)n_fields;
  e->fields.insert(e->fields.end(), f, f + n_fields);
  if (schema_id) *schema_id = (uint32_t)e->schemas.size();
  e->schemas.push_back(d);
  e->schemas_dirty = true;
  e->processed = false;
  return KTJ_OK;
}

int ktj_add_collective(ktj_engine* e, const ktj_collective_meta* meta, uint32_t* index) {
  if (!e || !meta) return KTJ_ERR_ARG;
  if (e->collectives.size() >= KTJ_MAX_COLLECTIVES) return KTJ_ERR_LIMIT; /* the join tables keep 1 + index in 29 bits */
  if (index) *index = (uint32_t)e->collectives.size();
  e->collectives.push_back(make_collective(*meta));
  e->coll_dirty = true;
  e->processed = false;
  return KTJ_OK;
}

int ktj_submit_args(ktj_engine* e, const uint64_t* slots, size_t n_slots, uint64_t* first_slot) {
  if (!e || (n_slots && !slots)) return KTJ_ERR_ARG;
  if (first_slot) *first_slot = e->n_args;
  if (e->bad_sink || n_slots == 0) return KTJ_OK;
  HIPCHK(hipSetDevice(e->device));
  { const int rc = append_from_host(e, e->args, slots, n_slots * 8); if (rc != KTJ_OK) return rc; }
  e->n_args += n_slots;
  e->processed = false;
  return KTJ_OK;
}

int ktj_set_api_table(ktj_engine* e, const uint32_t* cid_name_ids, size_t n_cids, const uint32_t* flow_start_cids,
                      size_t n_flow_start, uint32_t malloc_cid) {
  if (!e || (n_cids && !cid_name_ids) || (n_flow_start && !flow_start_cids)) return KTJ_ERR_ARG;
  e->cid_names.assign(cid_name_ids, cid_name_ids + n_cids);
  e->flow_bits.assign((n_cids + 31) / 32 + 1, 0u);
  for (size_t i = 0; i < n_flow_start; ++i)
    if (flow_start_cids[i] < n_cids) e->flow_bits[flow_start_cids[i] >> 5] |= 1u << (flow_start_cids[i] & 31u);
  e->malloc_cid = malloc_cid;
  e->api_dirty = true;
  e->processed = false;
  return KTJ_OK;
}

int ktj_set_clock_model(ktj_engine* e, const ktj_clock_model* m) {
  if (!e || !m) return KTJ_ERR_ARG;
  if (m->runtime_mode > KTJ_CLOCK_OFFSET || m->device_mode > KTJ_CLOCK_OFFSET) return KTJ_ERR_ARG;
  e->clock = *m;
  e->processed = false;
  return KTJ_OK;
}

int ktj_set_window(ktj_engine* e, int64_t start_ns, int64_t end_ns) {
  if (!e) return KTJ_ERR_ARG;
  e->win_start = start_ns;
  e->win_end = end_ns;
  e->processed = false;
  return KTJ_OK;
}

static RecordSet* record_set(ktj_engine* e, int rec_class, size_t* rec_size) {
  switch (rec_class) {
    case KTJ_REC_GENERIC: *rec_size = sizeof(ktj_generic_rec); return &e->generic;
    case KTJ_REC_RUNTIME: *rec_size = sizeof(ktj_runtime_rec); return &e->runtime;
    case KTJ_REC_DEVICE: *rec_size = sizeof(ktj_device_rec); return &e->devrows;
    case KTJ_REC_EXTCORR: *rec_size = sizeof(ktj_extcorr_rec); return &e->extcorr;
    case KTJ_REC_USERCORR: *rec_size = sizeof(ktj_extcorr_rec); return &e->usercorr;
    default: return nullptr;
  }
}

static int flush_sdk_api_rows(ktj_engine* e);
/* rows of ktj_submit_sdk_api_record that wait on the host arrived before anything submitted now */
static bool class_has_buffered_sdk_rows(int rec_class) {
  return rec_class == KTJ_REC_RUNTIME || rec_class == KTJ_REC_EXTCORR || rec_class == KTJ_REC_USERCORR;
}

int ktj_submit_records(ktj_engine* e, int rec_class, const void* packed, size_t n_records) {
  if (!e || (n_records && !packed)) return KTJ_ERR_ARG;
  size_t rs = 0;
  RecordSet* set = record_set(e, rec_class, &rs);
  if (!set) return KTJ_ERR_ARG;
  if (e->bad_sink || n_records == 0) return KTJ_OK;
  if (class_has_buffered_sdk_rows(rec_class)) {
    const int flushed = flush_sdk_api_rows(e);
    if (flushed != KTJ_OK) return flushed;
  }
  if (set->external) return KTJ_ERR_STATE;
  HIPCHK(hipSetDevice(e->device));
  { const int rc = append_from_host(e, set->owned, packed, n_records * rs); if (rc != KTJ_OK) return rc; }
  set->n += n_records;
  e->other_records();
  if (rec_class == KTJ_REC_GENERIC || rec_class == KTJ_REC_RUNTIME || rec_class == KTJ_REC_DEVICE) e->activities_begun = true;
  e->processed = false;
  return KTJ_OK;
}

int ktj_host_alloc(ktj_engine* e, size_t n_bytes, void** host_ptr) {
  if (!e || !host_ptr) return KTJ_ERR_ARG;
  *host_ptr = nullptr;
  HIPCHK(hipSetDevice(e->device));
  void* p = nullptr;
  const hipError_t rc = hipHostMalloc(&p, n_bytes ? n_bytes : 16, hipHostMallocDefault);
  if (rc != hipSuccess) { e->last_error = std::string("hipHostMalloc: ") + hipGetErrorString(rc); return KTJ_ERR_NOMEM; }
  *host_ptr = p;
  return KTJ_OK;
}

int ktj_host_free(ktj_engine* e, void* host_ptr) {
  if (!e) return KTJ_ERR_ARG;
  if (!host_ptr) return KTJ_OK;
  HIPCHK(hipSetDevice(e->device));
  HIPCHK(hipHostFree(host_ptr));
  return KTJ_OK;
}

int ktj_submit_records_device(ktj_engine* e, int rec_class, const void* device_ptr, size_t n_records) {
  if (!e || (n_records && !device_ptr)) return KTJ_ERR_ARG;
  size_t rs = 0;
  RecordSet* set = record_set(e, rec_class, &rs);
  if (!set) return KTJ_ERR_ARG;
  if (((uintptr_t)device_ptr & 15u) != 0) return KTJ_ERR_ARG; /* kernels read 16-byte lanes */
  if (e->bad_sink) return KTJ_OK;
  if (class_has_buffered_sdk_rows(rec_class)) {
    const int flushed = flush_sdk_api_rows(e);
    if (flushed != KTJ_OK) return flushed;
  }
  if (set->owned.bytes != 0) return KTJ_ERR_STATE;
  set->external = n_records ? device_ptr : nullptr;
  set->n = n_records;
  e->other_records();
  if (n_records && (rec_class == KTJ_REC_GENERIC || rec_class == KTJ_REC_RUNTIME || rec_class == KTJ_REC_DEVICE)) e->activities_begun = true;
  e->processed = false;
  return KTJ_OK;
}

/* ---- rocprofiler-sdk buffer records (include/ktj_rocprofiler.h) ---- */

int ktj_set_sdk_agents(ktj_engine* e, const uint64_t* agent_handles, const int32_t* device_ids, size_t n) {
  if (!e || (n && (!agent_handles || !device_ids))) return KTJ_ERR_ARG;
  e->sdk_agents.clear();
  for (size_t i = 0; i < n; ++i) e->sdk_agents[agent_handles[i]] = device_ids[i];
  return KTJ_OK;
}

int ktj_set_sdk_kernel_names(ktj_engine* e, const uint64_t* kernel_ids, const uint32_t* name_ids, size_t n,
                             uint32_t unknown_name_id) {
  if (!e || (n && (!kernel_ids || !name_ids))) return KTJ_ERR_ARG;
  for (size_t i = 0; i < n; ++i) e->sdk_kernel_names[kernel_ids[i]] = name_ids[i];
  e->sdk_unknown_name = unknown_name_id;
  return KTJ_OK;
}

/* RocprofLogger::buffer_callback (libkineto/src/RocprofLogger.cpp:681-749): the fields of a
 * rocprofAsyncRow (src/RocLogger.h:216-240) from a kernel-dispatch or memory-copy record. */
int ktj_submit_sdk_buffer(ktj_engine* e, void* const* headers, size_t num_headers, uint64_t* n_rows) {
  if (n_rows) *n_rows = 0;
  if (!e || (num_headers && !headers)) return KTJ_ERR_ARG;
  std::vector<ktj_device_rec>& rows = e->sdk_rows;
  rows.clear();
  rows.reserve(num_headers);
  auto device_of = [e](uint64_t agent_handle) {
    const auto it = e->sdk_agents.find(agent_handle);
    return it != e->sdk_agents.end() ? it->second : -1;
  };
  for (size_t i = 0; i < num_headers; ++i) {
    const rocprofiler_record_header_t* h = static_cast<const rocprofiler_record_header_t*>(headers[i]);
    if (!h || h->category != ROCPROFILER_BUFFER_CATEGORY_TRACING || !h->payload) continue;
    ktj_device_rec r{};
    if (h->kind == ROCPROFILER_BUFFER_TRACING_KERNEL_DISPATCH) {
      const auto& rec = *static_cast<const rocprofiler_buffer_tracing_kernel_dispatch_record_t*>(h->payload);
      const auto name = e->sdk_kernel_names.find(rec.dispatch_info.kernel_id);
      r.id = rec.correlation_id.internal;
      r.begin = rec.start_timestamp;
      r.end = rec.end_timestamp;
      r.domain = KTJ_DOM_KERNEL_DISPATCH;
      r.op = static_cast<uint32_t>(rec.operation);
      r.device = device_of(rec.dispatch_info.agent_id.handle);
      r.name_id = name != e->sdk_kernel_names.end() ? name->second : e->sdk_unknown_name;
      r.queue = rec.dispatch_info.queue_id.handle;
    } else if (h->kind == ROCPROFILER_BUFFER_TRACING_MEMORY_COPY) {
      const auto& rec = *static_cast<const rocprofiler_buffer_tracing_memory_copy_record_t*>(h->payload);
      r.id = rec.correlation_id.internal;
      r.begin = rec.start_timestamp;
      r.end = rec.end_timestamp;
      r.domain = KTJ_DOM_MEMORY_COPY;
      r.op = static_cast<uint32_t>(rec.operation);
      r.device = device_of(rec.dst_agent_id.handle);
      r.name_id = KTJ_NONE; /* the row's name is empty; the copy direction names the activity */
      r.queue = 0;
    } else {
      continue;
    }
    rows.push_back(r);
  }
  if (n_rows) *n_rows = rows.size();
  return ktj_submit_records(e, KTJ_REC_DEVICE, rows.data(), rows.size());
}

/* Runtime rows and correlation pairs that ktj_submit_sdk_api_record collected go to the device.  The
 * vectors are taken out first: the submit calls below flush whatever is buffered before they append. */
static int flush_sdk_api_rows(ktj_engine* e) {
  if (e->sdk_api_rows.empty() && e->sdk_api_ext.empty() && e->sdk_api_user.empty()) return KTJ_OK;
  std::vector<ktj_runtime_rec> rows; rows.swap(e->sdk_api_rows);
  std::vector<ktj_extcorr_rec> ext, user; ext.swap(e->sdk_api_ext); user.swap(e->sdk_api_user);
  int rc = KTJ_OK;
  if (!rows.empty()) rc = ktj_submit_records(e, KTJ_REC_RUNTIME, rows.data(), rows.size());
  if (rc == KTJ_OK && !ext.empty()) rc = ktj_submit_records(e, KTJ_REC_EXTCORR, ext.data(), ext.size());
  if (rc == KTJ_OK && !user.empty()) rc = ktj_submit_records(e, KTJ_REC_USERCORR, user.data(), user.size());
  if (rc != KTJ_OK) { /* nothing is lost: what a later flush finds is what this one could not place */
    e->sdk_api_rows.swap(rows); e->sdk_api_ext.swap(ext); e->sdk_api_user.swap(user);
  } else { /* keep the capacity for the next batch */
    rows.clear(); e->sdk_api_rows.swap(rows);
  }
  return rc;
}

int ktj_flush(ktj_engine* e) {
  if (!e) return KTJ_ERR_ARG;
  if (e->bad_sink) return KTJ_OK;
  return flush_sdk_api_rows(e);
}

#define KTJ_SDK_API_BATCH 65536u
int ktj_submit_sdk_api_record(ktj_engine* e, const void* record, uint64_t begin, uint64_t end, uint32_t pid, uint32_t tid,
                              const uint64_t* external_id, const uint64_t* user_external_id) {
  if (!e || !record) return KTJ_ERR_ARG;
  if (e->bad_sink) return KTJ_OK;
  const auto& rec = *static_cast<const rocprofiler_callback_tracing_record_t*>(record);
  if (rec.kind != ROCPROFILER_CALLBACK_TRACING_HIP_RUNTIME_API || !rec.payload) return KTJ_OK; /* RocprofLogger.cpp:567 */
  const auto& data = *static_cast<const rocprofiler_callback_tracing_hip_api_data_t*>(rec.payload);
  ktj_runtime_rec row;
  sdk_api::runtime_row(static_cast<uint32_t>(rec.operation), rec.correlation_id.internal, data.args, begin, end, pid, tid, &row);
  e->sdk_api_rows.push_back(row);
  if (external_id) e->sdk_api_ext.push_back(ktj_extcorr_rec{rec.correlation_id.internal, *external_id});
  if (user_external_id) e->sdk_api_user.push_back(ktj_extcorr_rec{rec.correlation_id.internal, *user_external_id});
  e->activities_begun = true;
  e->processed = false;
  return e->sdk_api_rows.size() >= KTJ_SDK_API_BATCH ? flush_sdk_api_rows(e) : KTJ_OK;
}

int ktj_begin_activities(ktj_engine* e) {
  if (!e) return KTJ_ERR_ARG;
  e->activities_begun = true;
  return KTJ_OK;
}

int ktj_submit_info(ktj_engine* e, int info_kind, const void* info) {
  if (!e || !info) return KTJ_ERR_ARG;
  if (e->bad_sink) return KTJ_OK;
  std::string& txt = e->activities_begun ? e->txt_after : e->txt_before;
  switch (info_kind) {
    case KTJ_INFO_DEVICE: append_device_info(txt, *static_cast<const ktj_device_info*>(info), e->base_time_ns); break;
    case KTJ_INFO_RESOURCE: append_resource_info(txt, *static_cast<const ktj_resource_info*>(info), e->base_time_ns); break;
    case KTJ_INFO_OVERHEAD: append_overhead_info(txt, *static_cast<const ktj_overhead_info*>(info), e->base_time_ns); break;
    case KTJ_INFO_SPAN: append_trace_span(txt, *static_cast<const ktj_trace_span*>(info), e->base_time_ns); break;
    default: return KTJ_ERR_ARG;
  }
  e->processed = false;
  return KTJ_OK;
}

/* A complete stream in one call (include/ktj_stream.h), in the call order of the buffering logger's
 * replay (libkineto/src/output_membuf.h:91-107): device and resource infos, the activities, the spans. */
int ktj_submit_stream(ktj_engine* e, const ktj_stream* s) {
  if (!e || !s) return KTJ_ERR_ARG;
  int rc = KTJ_OK;
  uint32_t id;
  uint64_t slot;
  /* the calls that follow one that failed are not made; ktj_last_error says which one it was (the calls leave a
   * text of their own only for a failed HIP call) */
  auto call = [&](const char* name, auto make) {
    if (rc != KTJ_OK) return;
    rc = make();
    if (rc != KTJ_OK) e->last_error = std::string("ktj_submit_stream: ") + name + (rc == KTJ_ERR_HIP ? ": " + e->last_error : " returned " + std::to_string(rc));
  };
  auto records = [&](const char* name, int rec_class, const void* packed, uint64_t n) {
    call(name, [&] { return ktj_submit_records(e, rec_class, packed, n); });
  };
  auto infos = [&](const char* name, int kind, auto* first, uint64_t n) {
    for (uint64_t i = 0; i < n && rc == KTJ_OK; ++i) call(name, [&] { return ktj_submit_info(e, kind, first + i); });
  };
  call("ktj_trace_start", [&] { return ktj_trace_start(e, s->meta_kv, s->n_meta, s->device_properties); });
  call("ktj_intern_strings", [&] { return ktj_intern_strings(e, s->str_blob, s->str_off, s->n_strings, &id); });
  for (uint64_t i = 0; i < s->n_schemas && rc == KTJ_OK; ++i)
    call("ktj_register_schema", [&] { return ktj_register_schema(e, s->fields + s->schemas[i].first_field, s->schemas[i].n_fields, &id); });
  for (uint64_t i = 0; i < s->n_collectives && rc == KTJ_OK; ++i)
    call("ktj_add_collective", [&] { return ktj_add_collective(e, &s->collectives[i], nullptr); });
  call("ktj_submit_args", [&] { return ktj_submit_args(e, s->args, s->n_args, &slot); });
  call("ktj_set_api_table",
       [&] { return ktj_set_api_table(e, s->cid_name_ids, s->n_cids, s->flow_start_cids, s->n_flow_start, s->malloc_cid); });
  call("ktj_set_clock_model", [&] { return ktj_set_clock_model(e, &s->clock); });
  call("ktj_set_window", [&] { return ktj_set_window(e, s->window_start_ns, s->window_end_ns); });
  infos("ktj_submit_info (device)", KTJ_INFO_DEVICE, s->device_infos, s->n_device_infos);
  infos("ktj_submit_info (resource)", KTJ_INFO_RESOURCE, s->resource_infos, s->n_resource_infos);
  infos("ktj_submit_info (overhead)", KTJ_INFO_OVERHEAD, s->overhead_infos, s->n_overhead_infos);
  call("ktj_begin_activities", [&] { return ktj_begin_activities(e); });
  records("ktj_submit_records (generic)", KTJ_REC_GENERIC, s->generic, s->n_generic);
  records("ktj_submit_records (runtime)", KTJ_REC_RUNTIME, s->runtime, s->n_runtime);
  records("ktj_submit_records (device)", KTJ_REC_DEVICE, s->device, s->n_device);
  records("ktj_submit_records (external correlation)", KTJ_REC_EXTCORR, s->extcorr, s->n_extcorr);
  records("ktj_submit_records (user correlation)", KTJ_REC_USERCORR, s->usercorr, s->n_usercorr);
  infos("ktj_submit_info (span)", KTJ_INFO_SPAN, s->spans, s->n_spans);
  return rc;
}

/* page-locked room for the document's header, infos and footer */
static int ensure_text(ktj_engine* e, size_t bytes) {
  if (bytes <= e->pinned_small_cap) return KTJ_OK;
  if (e->noalloc) {
    e->last_error = "ktj_process_noalloc: header and footer text of " + std::to_string(bytes) + " bytes exceeds the pinned staging buffer";
    return KTJ_ERR_LIMIT;
  }
  if (e->pinned_small) HIPCHK(hipHostFree(e->pinned_small));
  e->pinned_small = nullptr;
  e->pinned_small_cap = 0;
  HIPCHK(hipHostMalloc(&e->pinned_small, bytes * 2 + 4096, hipHostMallocDefault));
  e->pinned_small_cap = bytes * 2 + 4096;
  void* d = nullptr;
  HIPCHK(hipHostGetDevicePointer(&d, e->pinned_small, 0));
  e->pinned_small_dev = static_cast<char*>(d);
  return KTJ_OK;
}
/* header and footer into page-locked memory, for the kernels that put them in front of and behind the activities */
static int document_text(ktj_engine* e, const std::string& prefix, const std::string& suffix, DocText* text) {
  const size_t at_suffix = (prefix.size() + 15) & ~(size_t)15;
  const int rc = ensure_text(e, at_suffix + suffix.size() + 64);
  if (rc != KTJ_OK) return rc;
  memcpy(e->pinned_small, prefix.data(), prefix.size());
  memcpy(static_cast<char*>(e->pinned_small) + at_suffix, suffix.data(), suffix.size());
  text->prefix = e->pinned_small_dev; text->n_prefix = prefix.size();
  text->suffix = e->pinned_small_dev + at_suffix; text->n_suffix = suffix.size();
  text->h_sc = &e->h_ctl_dev->scalars; text->h_total = &e->h_ctl_dev->act_bytes; text->h_end = &e->h_ctl_dev->end_clock;
  return KTJ_OK;
}
static int short_output(ktj_engine* e) {
  e->last_error = "ktj_process_noalloc: the document has " + std::to_string(e->total_bytes) + " bytes and needs an output buffer of " +
                  std::to_string(e->total_bytes + 64);
  return KTJ_ERR_LIMIT;
}
/* per row the fixed text of an event and one string of average length, at most 2 KB */
static uint64_t guess_per_row(const ktj_engine* e) {
  const uint64_t avg_string = e->n_strings ? e->blob_bytes / e->n_strings : 0;
  return std::min<uint64_t>(KTJ_GUESS_BYTES_PER_ROW + avg_string, 2048);
}
static EmitCtx emit_context(const ktj_engine* e, uint32_t n_coll) {
  EmitCtx ctx;
  memset(&ctx, 0, sizeof ctx);
  ctx.dict.name_blob = e->d_name_blob.as<char>(); ctx.dict.arg_blob = e->d_arg_blob.as<char>();
  ctx.dict.raw_blob = e->str_blob.buf.as<char>(); ctx.dict.raw_off = e->str_off.buf.as<uint64_t>();
  ctx.dict.entries = e->d_entries.as<DictEntry>(); ctx.dict.n = (uint32_t)e->n_strings;
  ctx.fields = e->d_fields.as<ktj_field>(); ctx.schemas = e->d_schemas.as<ktj_schema_desc>();
  ctx.n_schemas = (uint32_t)e->schemas.size();
  ctx.args = e->args.buf.as<uint64_t>(); ctx.n_args = e->n_args;
  ctx.base_time_ns = e->base_time_ns;
  ctx.create_flags = e->flags;
  ctx.coll_blob = e->d_coll_blob.as<char>(); ctx.coll_off = e->d_coll_off.as<uint64_t>(); ctx.n_coll = n_coll;
  return ctx;
}
static ClockDev clock_of(const ktj_engine* e) {
  ClockDev clk;
  clk.t0_approx = e->clock.t0_approx; clk.t0 = e->clock.t0;
  memcpy(&clk.scale_bits, &e->clock.scale, 8);
  clk.async_offset = e->clock.async_offset; clk.runtime_mode = e->clock.runtime_mode; clk.device_mode = e->clock.device_mode;
  return clk;
}
static Columns columns_of(const ktj_engine* e) {
  Columns c;
  c.ts = e->c_ts.as<int64_t>(); c.dur = e->c_dur.as<int64_t>(); c.corr = e->c_corr.as<uint64_t>();
  c.dev = e->c_dev.as<int64_t>(); c.res = e->c_res.as<int64_t>(); c.meta = e->c_meta.as<uint32_t>();
  c.ext = e->c_ext.as<int32_t>();
  c.all = e->columns_are_all;
  return c;
}
static hipError_t know_wall_clock(ktj_engine* e) {
  return e->wall_clock_khz > 0 ? hipSuccess : hipDeviceGetAttribute(&e->wall_clock_khz, hipDeviceAttributeWallClockRate, e->device);
}
static float clock_ms(const ktj_engine* e, unsigned long long from, unsigned long long to) {
  return to > from ? (float)((double)(to - from) / e->wall_clock_khz) : 0.0f;
}
static void count_stats(ktj_engine* e, uint64_t N) {
  const uint64_t ng = e->generic.n, nr = e->runtime.n, nd = e->devrows.n, nx = e->extcorr.n;
  ktj_stats& s = e->stats;
  memset(&s, 0, sizeof s);
  s.n_generic = ng; s.n_runtime = nr; s.n_device = nd; s.n_extcorr = nx;
  s.n_emitted = e->scalars.n_valid;
  s.out_of_range_events = e->scalars.out_of_range;
  s.gpu_and_cpu_op_out_of_order = e->scalars.out_of_order;
  s.n_flow_events = e->scalars.n_flow;
  s.n_linked = e->scalars.n_linked;
  s.n_blank_names = e->scalars.n_blank_names;
  s.output_bytes = e->total_bytes;
  s.activity_bytes = e->act_bytes;
  const uint64_t raw_in = ng * sizeof(ktj_generic_rec) + nr * sizeof(ktj_runtime_rec) + nd * sizeof(ktj_device_rec);
  s.stage_bytes[KTJ_STAGE_DICT] = e->blob_bytes * 3;
  /* clock conversion and window filter run inside the decode kernels on values that are in registers
   * there: their bytes (two timestamps in, two out) are bytes of the decode stage already */
  s.stage_bytes[KTJ_STAGE_DECODE] = raw_in + N * 48;
  s.stage_bytes[KTJ_STAGE_CONVERT] = 0;
  s.stage_bytes[KTJ_STAGE_JOIN] = nx * 12 + ng * 12 + nr * 12 + (nr + nd) * 12 * 2 +
                                   nr * (sizeof(ktj_runtime_rec) + 48 + sizeof(MatRow) + 4); /* incl. the runtime rows' joined rows */
  const uint64_t last_launch = e->rows_with_sort ? N * 12 : 0; /* a word in, an index out: counted where its time is */
  s.stage_bytes[KTJ_STAGE_SORT] = N * 56 - last_launch;
  s.stage_bytes[KTJ_STAGE_SIZE] = last_launch + (ng * sizeof(ktj_generic_rec) + nd * sizeof(ktj_device_rec)) + (ng + nd) * 48 +
                                   (ng + nd) * (sizeof(MatRow) + 4) + N * 8;
  s.stage_bytes[KTJ_STAGE_SCAN] = N * 12;
  s.stage_bytes[KTJ_STAGE_EMIT] = e->scalars.n_valid * (sizeof(MatRow) + 12) + e->act_bytes;
}

/* The pass of a small trace: three launches and one wait (small.hip).  *done stays false where the trace
 * turns out to need the launches of a large one. */
static int process_small(ktj_engine* e, int64_t end_time_ns, void* out_device, uint64_t out_cap, bool* done) {
  hipStream_t st = e->stream;
  const uint64_t ng = e->generic.n, nr = e->runtime.n, nd = e->devrows.n, nx = e->extcorr.n, N = ng + nr + nd;
  const uint32_t ns = (uint32_t)e->n_strings;
  size_t pass_bytes = 0;
  e->pool_used = 0;
  for (int phase = e->noalloc ? 1 : 0; phase < 2; ++phase) {
    e->measuring = phase == 0;
    e->pool_need = 0;
    NEED(e->d_entries, (ns + 1ull) * sizeof(DictEntry));
    NEED(e->d_name_blob, e->blob_bytes * 2 + KTJ_DICT_ROOM * (ns + 1ull)); NEED(e->d_arg_blob, e->blob_bytes + KTJ_DICT_ROOM * (ns + 1ull));
    NEED(e->c_ts, N * 8); NEED(e->c_dur, N * 8); NEED(e->c_corr, N * 8); NEED(e->c_dev, N * 8); NEED(e->c_res, N * 8);
    NEED(e->c_meta, N * 4); NEED(e->c_ext, N * 4);
    NEED(e->dev_link, nd * sizeof(DevLink) + 16); NEED(e->mat, N * sizeof(MatRow)); NEED(e->len, N * 4); NEED(e->vals_a, N * 4);
    if (e->measuring) {
      e->measuring = false;
      pass_bytes = e->pool_need;
      if (e->pool.cap < pass_bytes + 4096) HIPCHK(e->pool.ensure(pass_bytes + 4096));
    }
  }
  const std::string prefix = e->txt_header + e->txt_before;
  std::string suffix = e->txt_after;
  append_trace_end(suffix, end_time_ns, e->base_time_ns, e->out_path, std::string());
  DocText text;
  { const int rc = document_text(e, prefix, suffix, &text); if (rc != KTJ_OK) return rc; }
  if (out_device) e->out.borrow(out_device, out_cap);
  else HIPCHK(e->out.ensure(N * guess_per_row(e) + prefix.size() + suffix.size() + (64u << 10), false));

  Scalars* sc = e->d_scalars.as<Scalars>();
  SmallArgs a;
  a.g = static_cast<const ktj_generic_rec*>(e->generic.ptr()); a.r = static_cast<const ktj_runtime_rec*>(e->runtime.ptr());
  a.d = static_cast<const ktj_device_rec*>(e->devrows.ptr()); a.x = static_cast<const ktj_extcorr_rec*>(e->extcorr.ptr());
  a.ng = (uint32_t)ng; a.nr = (uint32_t)nr; a.nd = (uint32_t)nd; a.nx = (uint32_t)nx;
  a.slots = small_slots(ng, nr, nd, nx);
  a.c = columns_of(e);
  a.link = e->dev_link.as<DevLink>();
  a.clk = clock_of(e); a.win_start = e->win_start; a.win_end = e->win_end;
  a.ctx = emit_context(e, 0);
  a.entries = e->d_entries.as<DictEntry>();
  a.api = ApiTable{e->d_cid_names.as<uint32_t>(), (uint32_t)e->cid_names.size(), e->d_flow_bits.as<uint32_t>(), e->malloc_cid};
  a.mat = e->mat.as<MatRow>(); a.len = e->len.as<uint32_t>(); a.perm = e->vals_a.as<uint32_t>();
  a.sc = sc;
  text.out = e->out.as<char>(); text.out_cap = e->out.cap;
  e->h_ctl->end_clock = 0;
  HIPCHK(small_pass(a, ns, st));
  HIPCHK(small_emit(a, text, st));
  HIPCHK(hipStreamSynchronize(st));
  e->stage_small_used = 0;
  e->stage_big_used = 0;
  e->scalars = e->h_ctl->scalars;
  if (e->scalars.error & KTJ_DEVERR_SMALL_UNFIT) { e->small_unfit = true; return KTJ_OK; }
  if (e->scalars.error) { e->last_error = limit_text(e->scalars.error); return KTJ_ERR_LIMIT; }
  e->act_bytes = e->h_ctl->act_bytes;
  e->prefix_len = prefix.size();
  e->total_bytes = prefix.size() + e->act_bytes + suffix.size();
  if (e->total_bytes + 64 > text.out_cap) { /* nothing has been written */
    if (out_device) return short_output(e);
    HIPCHK(e->out.ensure(e->total_bytes + 64));
    text.out = e->out.as<char>(); text.out_cap = e->out.cap;
    HIPCHK(small_emit(a, text, st));
    HIPCHK(hipStreamSynchronize(st));
  }
  if (e->scalars.n_plain) {
    HIPCHK(small_plain(a, text, st));
    HIPCHK(hipStreamSynchronize(st));
  }
  if (!out_device) e->most_needed = std::max(e->most_needed, pass_bytes + (size_t)e->total_bytes);
  count_stats(e, N);
  HIPCHK(know_wall_clock(e));
  /* by the device's clock: decode includes the dictionary, which is made beside it; size is what making
   * the joined rows takes beyond the sort that runs beside it */
  const unsigned long long* ck = e->scalars.clock;
  auto ms = [&](unsigned long long from, unsigned long long to) { return clock_ms(e, from, to); };
  ktj_stats& s = e->stats;
  if (!(e->flags & KTJ_CREATE_NO_STAGE_TIMES)) {
    s.stage_ms[KTJ_STAGE_DECODE] = ms(ck[0], ck[1]);
    s.stage_ms[KTJ_STAGE_JOIN] = ms(ck[1], ck[2]);
    s.stage_ms[KTJ_STAGE_SORT] = ms(ck[3], ck[4]);
    s.stage_ms[KTJ_STAGE_SIZE] = ms(ck[4], ck[5]);
    s.stage_ms[KTJ_STAGE_EMIT] = ms(ck[5], e->h_ctl->end_clock);
  }
  s.stage_ms[KTJ_STAGE_TOTAL_GPU] = ms(ck[0], e->h_ctl->end_clock);
  e->small_last = true;
  e->processed = true;
  *done = true;
  return KTJ_OK;
}

/* One pass of the whole path.  out_device == nullptr: the document goes into the engine's own
 * buffer and working memory is allocated as needed (ktj_process).  Otherwise (ktj_process_noalloc,
 * e->noalloc set by the caller): the document goes into the caller's buffer of out_cap bytes and
 * every working buffer is a piece of the scratch array. */
static int process_pass(ktj_engine* e, int64_t end_time_ns, void* out_device, uint64_t out_cap) {
  HIPCHK(hipSetDevice(e->device));
  hipStream_t st = e->stream;
  e->arena_used = 0;
  e->processed = false;
  e->total_bytes = 0;
  if (e->noalloc) e->schemas_dirty = e->api_dirty = e->coll_dirty = true; /* small tables live in the scratch array too */
  const uint64_t ng = e->generic.n, nr = e->runtime.n, nd = e->devrows.n, nx = e->extcorr.n, nu = e->usercorr.n;
  uint64_t N = ng + nr + nd; /* grows by the synthesised GPU user-annotation spans, at most one per device row */
  const uint64_t max_spans = nu ? nd : 0;
  if (N + max_spans >= 0xFFFFFFF0ull) { e->last_error = "more than 2^32 - 16 records"; return KTJ_ERR_LIMIT; }
  e->N = N;
  e->n_spans = 0;
  e->host_copy_valid = false;
  /* The document of the pass before may lie in a buffer of ktj_process_noalloc's caller, which that caller has had
   * back since: a pass of ktj_process begins with the engine's own buffer (or none). */
  if (!out_device) e->out.unborrow();
  const uint64_t Na = N + max_spans ? N + max_spans : 1;

  /* small tables */
  if (e->schemas_dirty) {
    int rc = upload_small(e, e->d_fields, e->fields.data(), e->fields.size() * sizeof(ktj_field));
    if (rc) return rc;
    rc = upload_small(e, e->d_schemas, e->schemas.data(), e->schemas.size() * sizeof(ktj_schema_desc));
    if (rc) return rc;
    e->schemas_not_taken = weave::schemas_not_taken(e->fields.data(), e->schemas.data(), (uint32_t)e->schemas.size());
    e->schemas_dirty = false;
  }
  if (e->api_dirty) {
    int rc = upload_small(e, e->d_cid_names, e->cid_names.data(), e->cid_names.size() * 4);
    if (rc) return rc;
    if (e->flow_bits.empty()) e->flow_bits.assign(1, 0u);
    rc = upload_small(e, e->d_flow_bits, e->flow_bits.data(), e->flow_bits.size() * 4);
    if (rc) return rc;
    e->api_dirty = false;
  }

  /* collective metadata is looked at only if both entries and a schema that refers to them exist */
  const uint32_t n_coll = e->coll_schemas ? (uint32_t)e->collectives.size() : 0u;
  if (n_coll && e->coll_dirty) {
    std::string blob;
    std::vector<uint64_t> off(e->collectives.size() + 1, 0);
    for (size_t k = 0; k < e->collectives.size(); ++k) { blob += e->collectives[k].args; off[k + 1] = blob.size(); }
    blob.append(16, '\0'); /* string copies load whole aligned words */
    int rc = upload_small(e, e->d_coll_blob, blob.data(), blob.size());
    if (rc == KTJ_OK) rc = upload_small(e, e->d_coll_off, off.data(), off.size() * 8);
    if (rc != KTJ_OK) return rc;
    e->coll_dirty = false;
  }
  { const int rc = put_pending_pieces(e); if (rc != KTJ_OK) return rc; }
  e->last_end_time = end_time_ns;
  e->sort_info[0] = e->sort_info[1] = 0;
  e->small_last = false;
  e->rows_are_text = e->rows_with_sort = false;
  if (!e->small_unfit && !e->no_small && nu == 0 && n_coll == 0 && small_fits(ng, nr, nd, nx) && !sort_packed_passes_forced() &&
      !(e->flags & (KTJ_CREATE_TILE_EMIT | KTJ_CREATE_HASH_JOIN | KTJ_CREATE_PAIR_SORT))) {
    bool done = false;
    const size_t tables = e->arena_used; /* of the scratch array */
    const int rc = process_small(e, end_time_ns, out_device, out_cap, &done);
    if (rc != KTJ_OK || done) return rc;
    e->arena_used = tables;
  }

  /* working memory */
  const uint32_t ns = (uint32_t)e->n_strings;
  if (nx >= 0x7FFFFFFFull || nr >= 0x7FFFFFFFull) { e->last_error = "more than 2^31 - 2 records of one class"; return KTJ_ERR_LIMIT; }
  /* capacities for the hash mode (load <= 2/3); the direct mode uses a prefix of the same buffers */
  const uint64_t slots_full = (nr + nd) + (nr + nd) / 2, slots_narrow = (nx + nr) + (nx + nr) / 2, slots_cpu = 2 * ng;
  const uint32_t cap_full = pow2_at_least(slots_full), cap_narrow = pow2_at_least(slots_narrow), cap_cpu = pow2_at_least(slots_cpu);
  /* Joined rows as text for the weaver, but where something reads them as they are, and where their 32 bytes more
   * would not fit the scratch array with as many records. */
  const bool woven = n_coll == 0 && !e->noalloc && !e->no_weave && !e->no_room_for_text && !(e->flags & KTJ_CREATE_TILE_EMIT) && (e->not_woven == 0 || e->not_woven != ng + nr + nd);
  e->rows_are_text = woven;
  e->pass_info[0] = woven; e->pass_info[1] = e->pass_info[2] = e->pass_info[3] = 0;
  e->columns_are_all = e->all_columns || max_spans != 0 || e->noalloc;
  const bool wide = woven && std::any_of(e->fields.begin(), e->fields.end(), [](const ktj_field& f) { return f.type == KTJ_F_F64; });
  e->pool_used = 0;
  size_t pass_bytes = 0;
  for (int phase = e->noalloc ? 1 : 0; phase < 2; ++phase) { /* 0: add the sizes up and size the pool; 1: hand the buffers out */
  e->measuring = phase == 0;
  e->pool_need = 0;
  NEED(e->d_entries, (ns + 1ull) * sizeof(DictEntry));
  NEED(e->d_name_blob, e->blob_bytes * 2 + KTJ_DICT_ROOM * (ns + 1ull)); NEED(e->d_arg_blob, e->blob_bytes + KTJ_DICT_ROOM * (ns + 1ull));
  NEED(e->c_ts, Na * 8); NEED(e->c_dur, e->columns_are_all ? Na * 8 : 16); NEED(e->c_corr, Na * 8);
  NEED(e->c_dev, Na * 8); NEED(e->c_res, Na * 8); NEED(e->c_meta, Na * 4);
  NEED(e->c_ext, Na * 4);
  NEED(e->t_full, (cap_full + 1ull) * 8); NEED(e->t_narrow, (cap_narrow + 1ull) * 8);
  NEED(e->t_cpu, (cap_cpu + 1ull) * 8);
  NEED(e->f_first, (cap_full + 1ull) * 4); NEED(e->f_stream_src, (cap_full + 1ull) * 4);
  NEED(e->f_pay, (cap_full + 1ull) * sizeof(FullPay));
  NEED(e->f_has_runtime, (cap_full / 32 + 2ull) * 4);
  NEED(e->n_ext_src, (cap_narrow + 1ull) * 4); NEED(e->n_kern_src, (cap_narrow + 1ull) * 4);
  NEED(e->n_copy_src, (cap_narrow + 1ull) * 4); NEED(e->n_pay, (cap_narrow + 1ull) * sizeof(NarrowPay));
  if (!e->noalloc) NEED(e->n_head, (cap_narrow + 1ull) * sizeof(NarrowHead)); /* (the scratch array has as many records without) */
  NEED(e->slot_f, nr * 4 + 16); NEED(e->slot_n, nr * 4 + 16);
  NEED(e->dev_link, nd * sizeof(DevLink) + 16);
  NEED(e->dev_queue, nd * 8 + 16);
  NEED(e->q_keys, (KTJ_QUEUE_CAP + 1ull) * 8); NEED(e->q_stream, (KTJ_QUEUE_CAP + 1ull) * 8);
  NEED(e->q_amb, (KTJ_QUEUE_CAP + 1ull) * 4);
  NEED(e->dn_hash, (KTJ_DENSE_CAP + 1ull) * 8); NEED(e->dn_first, (KTJ_DENSE_CAP + 1ull) * 4);
  NEED(e->dn_dev, (KTJ_DENSE_CAP + 1ull) * 4); NEED(e->dn_key, (KTJ_DENSE_CAP + 1ull) * 8);
  NEED(e->dn_rank, (KTJ_DENSE_CAP + 1ull) * 4); NEED(e->dn_list, KTJ_MAX_STREAM_PAIRS * 4ull);
  NEED(e->s_dev_k, (KTJ_SET_CAP + 1ull) * 8); NEED(e->s_dev_r, (KTJ_SET_CAP + 1ull) * 4); NEED(e->s_dev_l, KTJ_SET_MAX * 4ull);
  NEED(e->s_res_k, (KTJ_SET_CAP + 1ull) * 8); NEED(e->s_res_r, (KTJ_SET_CAP + 1ull) * 4); NEED(e->s_res_l, KTJ_SET_MAX * 4ull);
  NEED(e->keys_a, Na * 8); NEED(e->keys_b, Na * 8);
  NEED(e->vals_a, Na * 4); NEED(e->vals_b, Na * 4);
  NEED(e->hist, radix_tmp_elems(Na) * 4);
  {
    uint64_t m = scan_tmp_elems(radix_tmp_elems(Na));
    const uint64_t m2 = offsets_tmp_elems(Na);
    if (m2 > m) m = m2;
    NEED(e->scan_tmp, m * 8);
  }
  NEED(e->mat, Na * (woven ? sizeof(weave::TextRow) : sizeof(MatRow)));
  if (woven) NEED(e->schema_book, sizeof(weave::SchemaBook));
  if (wide) NEED(e->wide_text, ng * sizeof(weave::WideText));
  NEED(e->len, Na * 4); NEED(e->len_sorted, Na * 4); NEED(e->kind_sorted, Na + 16);
  NEED(e->offs, (Na + 1) * 8);
  if (e->measuring) {
    e->measuring = false;
    if (e->pool.cap < e->pool_need + 4096) HIPCHK(e->pool.ensure(e->pool_need + 4096));
    pass_bytes = e->pool_need;
  }
  }

  Scalars* sc = e->d_scalars.as<Scalars>();
  const bool stage_times = !(e->flags & KTJ_CREATE_NO_STAGE_TIMES);
  const Columns c = columns_of(e);
  const ktj_generic_rec* g_recs = static_cast<const ktj_generic_rec*>(e->generic.ptr());
  const ktj_runtime_rec* r_recs = static_cast<const ktj_runtime_rec*>(e->runtime.ptr());
  const ktj_device_rec* d_recs = static_cast<const ktj_device_rec*>(e->devrows.ptr());
  const ktj_extcorr_rec* x_recs = static_cast<const ktj_extcorr_rec*>(e->extcorr.ptr());

  HIPCHK(hipEventRecord(e->ev[EV_START], st));

  /* ---- the start, stage 0: dictionary ---- */
  const EmitCtx ctx = emit_context(e, n_coll);
  uint32_t* cpu_row = nullptr; /* last CPU op per id: only where something is read from that op */
  if (n_coll || max_spans) {
    NEED(e->cpu_row, (cap_cpu + 1ull) * 4);
    cpu_row = e->cpu_row.as<uint32_t>();
    HIPCHK(fill_u32(cpu_row, 0, cap_cpu + 1ull, st));
  }
  if (n_coll) NEED(e->d_coll_first, 2ull * n_coll * 4);
  StreamTables stt{e->q_keys.as<uint64_t>(), e->q_stream.as<uint64_t>(), e->q_amb.as<uint32_t>(), e->dn_hash.as<uint64_t>(),
                   e->dn_first.as<uint32_t>(), e->dn_dev.as<int32_t>(), e->dn_key.as<uint64_t>(), e->dn_rank.as<uint32_t>(),
                   e->dn_list.as<uint32_t>()};
  SortSets sets{e->s_dev_k.as<uint64_t>(), e->s_dev_r.as<uint32_t>(), e->s_res_k.as<uint64_t>(), e->s_res_r.as<uint32_t>(),
                e->s_dev_l.as<uint32_t>(), e->s_res_l.as<uint32_t>()};
  FillJobs fills;
  fills.count = 0;
  fills.add(stt.q_keys, KTJ_EMPTY_KEY, KTJ_QUEUE_CAP + 1ull, 8); fills.add(stt.q_stream, 0, KTJ_QUEUE_CAP + 1ull, 8);
  fills.add(stt.q_amb, 0, KTJ_QUEUE_CAP + 1ull, 4);
  fills.add(stt.d_hash, KTJ_EMPTY_KEY, KTJ_DENSE_CAP + 1ull, 8); fills.add(stt.d_first, 0xFFFFFFFFu, KTJ_DENSE_CAP + 1ull, 4);
  fills.add(stt.d_rank, 0, KTJ_DENSE_CAP + 1ull, 4);
  fills.add(sets.dev_keys, KTJ_EMPTY_KEY, KTJ_SET_CAP + 1ull, 8); fills.add(sets.res_keys, KTJ_EMPTY_KEY, KTJ_SET_CAP + 1ull, 8);
  HIPCHK(begin_pass(sc, fills, e->str_blob.buf.as<char>(), e->str_off.buf.as<uint64_t>(), ns, e->d_entries.as<DictEntry>(),
                    e->d_name_blob.as<char>(), e->d_arg_blob.as<char>(), st));

  /* ---- stage 1: decode; stage 2a, clock conversion and window filter, happens inside ---- */
  {
    DecodeJob job;
    memset(&job, 0, sizeof job);
    job.g = g_recs; job.r = r_recs; job.d = d_recs; job.x = x_recs;
    job.ng = ng; job.nr = nr; job.nd = nd; job.nx = nx;
    job.whole_pass = true;
    job.text = woven;
    job.schemas_not_taken = e->schemas_not_taken; job.n_cids = (uint32_t)e->cid_names.size();
    job.queue = e->dev_queue.as<uint64_t>();
    job.clk = clock_of(e); job.win_start = e->win_start; job.win_end = e->win_end;
    HIPCHK(decode(job, c, ctx, sc, st));
  }

  /* ---- stage 2b: joins ---- */
  Table tf{e->t_full.as<uint64_t>(), cap_full - 1, hash_runs(slots_full, cap_full), 0u, &sc->plan.ctl[KTJ_TBL_FULL]};
  Table tn{e->t_narrow.as<uint64_t>(), cap_narrow - 1, hash_runs(slots_narrow, cap_narrow), 0u, &sc->plan.ctl[KTJ_TBL_NARROW]};
  Table t_cpu{e->t_cpu.as<uint64_t>(), cap_cpu - 1, hash_runs(slots_cpu, cap_cpu), 1u, &sc->plan.ctl[KTJ_TBL_CPU]};
  FullCols fc{e->f_has_runtime.as<uint32_t>(), e->f_first.as<uint32_t>(), e->f_stream_src.as<uint32_t>(), e->f_pay.as<FullPay>()};
  NarrowCols nc{e->n_ext_src.as<uint32_t>(), e->n_kern_src.as<uint32_t>(), e->n_copy_src.as<uint32_t>(), e->n_pay.as<NarrowPay>(),
                e->noalloc ? nullptr : e->n_head.as<NarrowHead>()};
  e->h_ctl->weave = KTJ_WEAVE_UNKNOWN;
  HIPCHK(plan_tables(tf, fc, tn, nc, t_cpu, (e->flags & KTJ_CREATE_HASH_JOIN) != 0, woven ? ng + nr + nd : 0u, &e->h_ctl_dev->weave, sc, st));
  ApiTable api{e->d_cid_names.as<uint32_t>(), (uint32_t)e->cid_names.size(), e->d_flow_bits.as<uint32_t>(), e->malloc_cid};
  weave::SchemaBook* book = woven ? e->schema_book.as<weave::SchemaBook>() : nullptr;
  const Rows rows{e->mat.p, book, wide ? e->wide_text.as<weave::WideText>() : nullptr};
  const MatRow* mat = e->mat.as<MatRow>();
  /* places of the rows that are not text: in the sort's buffer that does not hold its result */
  auto left = [&]() -> uint32_t* { return !woven ? nullptr : e->sorted_keys == e->keys_b.p ? e->keys_a.as<uint32_t>() : e->keys_b.as<uint32_t>(); };
  /* only external-correlation records and user spans ask for the CPU ops' ids (5 M records without any: 58 us) */
  if (nx || max_spans) HIPCHK(build_cpu_ids(g_recs, ng, t_cpu, cpu_row, sc, st));
  HIPCHK(build_extcorr(x_recs, nx, tn, nc, t_cpu, cpu_row, g_recs, ctx, sc, st));
  HIPCHK(join_runtime_rows(r_recs, nr, c, ng, api, tf, fc, tn, nc, e->slot_f.as<uint32_t>(), e->slot_n.as<uint32_t>(), clock_of(e), ctx, rows,
                           e->len.as<uint32_t>(), sc, st));
  HIPCHK(republish_runtime_rows(r_recs, nr, c, ng, fc, nc, e->slot_f.as<uint32_t>(), e->slot_n.as<uint32_t>(), sc, st));
  unsigned long long* orphans = e->keys_a.as<unsigned long long>(); /* a bit per device row: the sort's words come later */
  HIPCHK(link_device_rows(nd, c, ng + nr, tf, fc, tn, nc, links_in(e->dev_link.p, nd), orphans, sc, st));
  HIPCHK(backfill_streams(e->dev_queue.as<uint64_t>(), nd, max_spans != 0, c, ng + nr, tf, fc, orphans, stt, sc, st));
  if (max_spans) {
    const int rc = synthesise_user_spans(e, c, ctx, t_cpu, cpu_row, sc, N);
    if (rc != KTJ_OK) return rc;
    N += e->n_spans;
    e->N = N;
  }

  /* ---- stage 3: canonical order ---- */
  /* The rest of the pass is put into the stream in one go where its launches can be told beforehand:
   * the widths of the sort's keys stay on the device, the kernels behind it read what they need from
   * there, and the host waits once, for the finished document.  (With a wait before the sort and one
   * before emit the GPU stood still for 25 us each: 30 000 records took 346 us.)  It cannot be told with
   * collective entries (the footer names those in use) and synthesised spans, and what else only the
   * device sees, it flags: more sort passes than launched, keys too wide for the one-word sort, CUDA_SYNC
   * activities, too many distinct values.  Such records take the stepwise rest of the pass from here on. */
  bool has_room = true;
  if (!out_device && e->out.cap == 0) {
    /* An engine's first pass has no document buffer yet, and how long the document is comes out of
     * the scan.  A first guess is allocated here, while the GPU is busy with the join.  If that turns out too
     * small the buffer is allocated where its size is known, as in later passes; if it cannot be had, the
     * stepwise rest does that from the start. */
    has_room = e->out.ensure(N * guess_per_row(e) + (1u << 20), false) == hipSuccess;
    if (!has_room) (void)hipGetLastError();
  }
  /* (settled here: collect_distinct flags what only a host that does not look would get wrong) */
  const bool straight = has_room && n_coll == 0 && max_spans == 0 && !e->stepwise && !(e->flags & KTJ_CREATE_TILE_EMIT) && e->sort_mode != 1;
  const Backfill fill{e->dev_queue.as<uint64_t>(), ng + nr, max_spans ? 0 : nd, stt};
  HIPCHK(collect_distinct(c, N, nd, fill, sets, sc, straight, ctx, book, st));
  /* The document's activities, but for the tile variant: what the weaver prints, and at most n_left others. */
  auto put_activities = [&](uint64_t n_most, uint64_t n_left, uint64_t at, bool weave = true) -> int {
    if (woven && n_most && weave)
      HIPCHK(weave_activities(e->mat.as<weave::TextRow>(), e->perm, e->offs.as<uint64_t>(), e->kind_sorted.as<uint8_t>(), n_most, ctx, e->out.as<char>(), at, sc, book, rows.wide, st));
    HIPCHK(emit_direct(rows.p, e->perm, e->offs.as<uint64_t>(), e->kind_sorted.as<uint8_t>(), woven ? n_left : n_most, ctx, e->out.as<char>(), at, sc, left(), st));
    return KTJ_OK;
  };
  /* when the scalars are the host's: how many others there are */
  auto was_woven = [&]() -> uint64_t {
    if (!woven) return 0;
    const uint64_t n = e->scalars.no_text ? e->scalars.n_valid : e->scalars.n_left;
    e->not_woven = too_many_left(n, e->scalars.n_valid) ? ng + nr + nd : 0u;
    e->pass_info[1] = e->scalars.no_text; e->pass_info[2] = n;
    return n;
  };
  bool emitted = false;
  if (straight) {
    const std::string prefix = e->txt_header + e->txt_before;
    std::string suffix = e->txt_after;
    append_trace_end(suffix, end_time_ns, e->base_time_ns, e->out_path, std::string());
    DocText text;
    { const int rc = document_text(e, prefix, suffix, &text); if (rc != KTJ_OK) return rc; }
    if (out_device) e->out.borrow(out_device, out_cap);
    e->perm = e->vals_a.as<uint32_t>();
    e->sorted_keys = nullptr;
    auto sort = [&](RowsJob* job) { return sort_packed(c, N, sets, sc, e->passes_to_launch(N), !e->sort_all_bits, e->keys_a.as<uint64_t>(), e->keys_b.as<uint64_t>(), e->perm, e->hist.as<uint32_t>(), e->offs.as<uint32_t>(), job, st); };
    RowsJob job{g_recs, ng, d_recs, nd, c, ng + nr, links_in(e->dev_link.p, nd), clock_of(e), ctx, rows, e->len.as<uint32_t>(), false};
    HIPCHK(sort(&job));
    e->rows_with_sort = job.made;
    if (!job.made) HIPCHK(mat_rows(g_recs, ng, 0, nullptr, d_recs, nd, c, ng + nr, links_in(e->dev_link.p, nd), clock_of(e), ctx, rows, e->len.as<uint32_t>(), sc, st));
    for (;;) {
      text.out = e->out.as<char>(); text.out_cap = e->out.cap;
      HIPCHK(gather_offsets(e->perm, e->len.as<uint32_t>(), N, e->len_sorted.as<uint32_t>(), e->kind_sorted.as<uint8_t>(),
                            e->scan_tmp.as<uint64_t>(), e->offs.as<uint64_t>(), left(), sc, text, st));
      /* Mostly there are no others, and a launch that finds its list empty takes 4 us, 20 with 22 million rows.  What k_decode
       * has counted is here by now or soon: in the first pass of an engine that is waited for, with ten launches and more behind
       * it in the stream.  Others that it cannot know of are printed behind a wait of their own the first time.  (No look at the count: 30 000 records of which some are left
       * 217 instead of 200 us; the launch in every first pass: 180 instead of 176 us with none left.) */
      auto look = [&]() -> uint32_t { return woven ? __atomic_load_n(&e->h_ctl->weave, __ATOMIC_ACQUIRE) : (uint32_t)KTJ_WEAVE_UNKNOWN; };
      uint32_t counted = look();
      if (woven && e->some_left < 0)
        for (const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(1); counted == KTJ_WEAVE_UNKNOWN && std::chrono::steady_clock::now() < until;) counted = look();
      const bool others = counted >= KTJ_WEAVE_MOST || (counted == KTJ_WEAVE_ALL ? e->some_left > 0 : e->some_left != 0);
      { const int rc = put_activities(N, others ? N : 0u, prefix.size(), counted != KTJ_WEAVE_NONE); if (rc != KTJ_OK) return rc; }
      HIPCHK(hipEventRecord(e->ev[EV_EMIT], st));
      HIPCHK(hipStreamSynchronize(st));
      e->scalars = e->h_ctl->scalars;
      if (e->scalars.error == KTJ_DEVERR_UNSORTED) { /* the rows are made: what needs their order comes again, with passes over all bits */
        e->sort_all_bits = 16; e->sort_info[1] = 1;
        e->sort_passes = sort_packed_passes(e->scalars.sort, false);
        HIPCHK(clear_error_bits(sc, KTJ_DEVERR_UNSORTED, st));
        HIPCHK(sort(nullptr));
        e->rows_with_sort = false;
        continue;
      }
      if (e->scalars.error) break;
      e->act_bytes = e->h_ctl->act_bytes;
      e->prefix_len = prefix.size();
      e->total_bytes = prefix.size() + e->act_bytes + suffix.size();
      emitted = e->total_bytes + 64 <= text.out_cap;
      if (emitted) {
        const uint64_t n_left = was_woven();
        if (woven) e->some_left = n_left != 0 ? 1 : 0;
        if (n_left != 0 && !others) {
          e->pass_info[3] = 1;
          { const int rc = put_activities(0, n_left, prefix.size()); if (rc != KTJ_OK) return rc; }
          HIPCHK(hipEventRecord(e->ev[EV_EMIT], st));
          HIPCHK(hipStreamSynchronize(st));
        }
        break;
      }
      if (out_device) return short_output(e); /* nothing has been written */
      HIPCHK(e->out.ensure(e->total_bytes + 64));
      HIPCHK(fill_u32(&sc->n_left, 0, 1, st)); /* the list is made anew */
    }
    if (emitted) {
      e->sort_passes = sort_packed_passes(e->scalars.sort, !e->sort_all_bits);
      if (!e->sort_all_bits && !sort_packed_in_one_launch(N)) e->sort_info[0] = e->scalars.sort.low_bits;
    }
    else if (e->scalars.error & ~(KTJ_DEVERR_CAREFUL | KTJ_DEVERR_DISTINCT_DEVICES | KTJ_DEVERR_DISTINCT_RESOURCES)) {
      e->last_error = limit_text(e->scalars.error);
      return KTJ_ERR_LIMIT;
    } else {
      e->stepwise = true;
      HIPCHK(clear_error_bits(sc, KTJ_DEVERR_CAREFUL, st));
    }
  }
  if (!emitted) { /* the stepwise rest */
  e->rows_with_sort = false;
  HIPCHK(publish(sc, nullptr, nullptr, 0, &e->h_ctl_dev->scalars, nullptr, nullptr, st));
  HIPCHK(hipStreamSynchronize(st));
  e->scalars = e->h_ctl->scalars;
  const unsigned distinct_overflow = e->scalars.error & (KTJ_DEVERR_DISTINCT_DEVICES | KTJ_DEVERR_DISTINCT_RESOURCES);
  if (e->scalars.error & ~distinct_overflow) {
    e->last_error = limit_text(e->scalars.error);
    return KTJ_ERR_LIMIT;
  }
  uint32_t ts_bits = 0, res_bits = 0, key_bits = 0, rank_bits = 0;
  if (e->scalars.n_valid) {
    ts_bits = (uint32_t)bits_for(e->scalars.ts_max_biased - e->scalars.ts_min_biased);
    res_bits = (uint32_t)bits_for(e->scalars.n_res_ranks ? e->scalars.n_res_ranks - 1 : 0);
    const uint32_t dev_bits = (uint32_t)bits_for(e->scalars.n_dev_ranks ? e->scalars.n_dev_ranks - 1 : 0);
    key_bits = ts_bits + res_bits + dev_bits;
    rank_bits = res_bits + dev_bits;
  }
  {
    uint64_t* ka = e->keys_a.as<uint64_t>(); uint32_t* va = e->vals_a.as<uint32_t>();
    uint64_t* kb = e->keys_b.as<uint64_t>(); uint32_t* vb = e->vals_b.as<uint32_t>();
    uint32_t* hist = e->hist.as<uint32_t>(); uint64_t* scan_tmp = e->scan_tmp.as<uint64_t>();
    /* one more stable sort on top of the order so far: keys made from the rows in that order,
     * into the pair of buffers that does not hold it */
    auto sort_again = [&](auto make, uint32_t bits) -> int {
      const uint32_t* order = e->perm;
      if (order == va) { HIPCHK(make(order, kb, vb)); HIPCHK(radix_sort(kb, vb, ka, va, N, bits, hist, scan_tmp, &e->sorted_keys, &e->perm, st)); }
      else { HIPCHK(make(order, ka, va)); HIPCHK(radix_sort(ka, va, kb, vb, N, bits, hist, scan_tmp, &e->sorted_keys, &e->perm, st)); }
      return KTJ_OK;
    };
    if (distinct_overflow) {
      /* too many distinct deviceId or resourceId values for ranks: timestamp, then resourceId, then
       * deviceId, each on the raw values, then dropped rows to the back */
      HIPCHK(clear_error_bits(sc, distinct_overflow, st));
      HIPCHK(make_ts_keys(c, N, sc, ka, va, st));
      HIPCHK(radix_sort(ka, va, kb, vb, N, ts_bits, hist, scan_tmp, &e->sorted_keys, &e->perm, st));
      int rc = sort_again([&](const uint32_t* o, uint64_t* k, uint32_t* v) { return make_column_keys(c.res, c.meta, o, N, 0, k, v, st); }, 64);
      if (rc == KTJ_OK) rc = sort_again([&](const uint32_t* o, uint64_t* k, uint32_t* v) { return make_column_keys(c.dev, c.meta, o, N, 0, k, v, st); }, 64);
      if (rc == KTJ_OK) rc = sort_again([&](const uint32_t* o, uint64_t* k, uint32_t* v) { return make_column_keys(c.dev, c.meta, o, N, 1, k, v, st); }, 1);
      if (rc != KTJ_OK) return rc;
    } else if (e->sort_mode != 1 && sort_packed_fits(N, e->scalars.sort)) {
      HIPCHK(sort_packed(c, N, sets, sc, sort_packed_passes(e->scalars.sort, false), false, ka, kb, va, hist, e->offs.as<uint32_t>(), nullptr, st));
      e->perm = va;
      e->sorted_keys = nullptr;
    } else if (key_bits <= 62) {
      HIPCHK(make_keys(c, N, sets, sc, ts_bits, res_bits, key_bits, ka, va, st));
      HIPCHK(radix_sort(ka, va, kb, vb, N, key_bits + 1, hist, scan_tmp, &e->sorted_keys, &e->perm, st));
    } else {
      /* timestamp span too wide for one composite key: stable sort by timestamp, then by ranks
       * (at most 2 x 12 bits) */
      HIPCHK(make_ts_keys(c, N, sc, ka, va, st));
      HIPCHK(radix_sort(ka, va, kb, vb, N, ts_bits, hist, scan_tmp, &e->sorted_keys, &e->perm, st));
      const int rc = sort_again([&](const uint32_t* o, uint64_t* k, uint32_t* v) { return make_rank_keys(c, o, N, sets, res_bits, rank_bits, k, v, st); },
                                rank_bits + 1);
      if (rc != KTJ_OK) return rc;
    }
  }

  /* ---- stage 4a: joined rows + lengths ---- */
  const uint32_t* sync_first = nullptr;
  if (e->scalars.n_sync_typed != 0) { /* known since the read-back before the sort */
    NEED(e->sync_keys, (KTJ_SYNC_CAP + 1ull) * 8); NEED(e->sync_pos, (KTJ_SYNC_CAP + 1ull) * 4);
    NEED(e->sync_first, ng * 4 + 16);
    HIPCHK(stream_sync_first(e->perm, e->scalars.n_valid, g_recs, ng, c.dev, ctx.dict, e->sync_keys.as<uint64_t>(),
                             e->sync_pos.as<uint32_t>(), e->sync_first.as<uint32_t>(), sc, st));
    sync_first = e->sync_first.as<uint32_t>();
  }
  HIPCHK(mat_rows(g_recs, ng, 0, sync_first, d_recs, nd, c, ng + nr, links_in(e->dev_link.p, nd), clock_of(e), ctx, rows, e->len.as<uint32_t>(), sc, st));
  HIPCHK(mat_rows(e->synth_recs.as<ktj_generic_rec>(), e->n_spans, ng + nr + nd, nullptr, nullptr, 0, c, 0, Links{}, clock_of(e), ctx, rows,
                  e->len.as<uint32_t>(), sc, st));
  if (n_coll) HIPCHK(collective_first(mat, e->perm, e->scalars.n_valid, n_coll, e->d_coll_first.as<uint32_t>(), st));

  /* ---- scan ---- */
  if (straight) HIPCHK(fill_u32(&sc->n_left, 0, 1, st));
  HIPCHK(gather_offsets(e->perm, e->len.as<uint32_t>(), N, e->len_sorted.as<uint32_t>(), e->kind_sorted.as<uint8_t>(),
                        e->scan_tmp.as<uint64_t>(), e->offs.as<uint64_t>(), left(), sc, DocText{}, st));
  uint64_t act_bytes = 0;
  e->coll_first.assign(2ull * n_coll, 0xFFFFFFFFu);
  const bool list_fits = 2ull * n_coll * 4 <= e->pinned_small_cap; /* through the engine's pinned buffer when it fits */
  if (n_coll && !list_fits && e->noalloc) {
    e->last_error = "ktj_process_noalloc: too many collective entries for the pinned staging buffer";
    return KTJ_ERR_LIMIT;
  }
  HIPCHK(publish(sc, e->offs.as<uint64_t>() + N, e->d_coll_first.as<uint32_t>(), list_fits ? 2u * n_coll : 0u, &e->h_ctl_dev->scalars,
                 &e->h_ctl_dev->act_bytes, reinterpret_cast<uint32_t*>(e->pinned_small_dev), st));
  if (n_coll && !list_fits) HIPCHK(hipMemcpyAsync(e->coll_first.data(), e->d_coll_first.p, 2ull * n_coll * 4, hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  if (n_coll && list_fits) memcpy(e->coll_first.data(), e->pinned_small, 2ull * n_coll * 4);
  act_bytes = e->h_ctl->act_bytes;
  e->scalars = e->h_ctl->scalars;
  if (e->scalars.error) {
    e->last_error = limit_text(e->scalars.error);
    return KTJ_ERR_LIMIT;
  }
  std::string distributed_info;
  if (n_coll) { /* the uses in emission order: one per entry and backend is enough, later ones repeat it */
    std::vector<std::pair<uint32_t, uint32_t>> firsts; /* (position, 2 * index + hccl) */
    for (uint32_t k = 0; k < 2u * n_coll; ++k)
      if (e->coll_first[k] != 0xFFFFFFFFu) firsts.emplace_back(e->coll_first[k], k);
    std::sort(firsts.begin(), firsts.end());
    std::vector<CollectiveUse> uses;
    for (const auto& f : firsts) uses.push_back(CollectiveUse{f.second >> 1, (f.second & 1u) != 0});
    distributed_info = distributed_info_text(e->collectives, uses);
  }

  /* ---- emit ---- */
  std::string prefix = e->txt_header + e->txt_before;
  std::string suffix = e->txt_after;
  append_trace_end(suffix, end_time_ns, e->base_time_ns, e->out_path, distributed_info);
  e->prefix_len = prefix.size();
  e->act_bytes = act_bytes;
  e->total_bytes = prefix.size() + act_bytes + suffix.size();
  if (out_device) { /* the caller's buffer: whole 16-byte blocks are stored, so a little room past the end is needed */
    if (e->total_bytes + 64 > out_cap) return short_output(e);
    e->out.borrow(out_device, out_cap);
  } else HIPCHK(e->out.ensure(e->total_bytes + 64)); /* never a piece of the pool, which the next pass deals out anew */
  const size_t small = prefix.size() + suffix.size() + 64; /* each piece starts where its place in the document does, modulo 16 */
  { const int rc = ensure_text(e, small); if (rc != KTJ_OK) return rc; }
  {
    char* dst_a = e->out.as<char>();
    char* dst_b = dst_a + prefix.size() + act_bytes;
    const size_t at_a = (size_t)(((uintptr_t)dst_a - (uintptr_t)e->pinned_small_dev) & 15u);
    const size_t after_a = (at_a + prefix.size() + 15u) & ~(size_t)15u;
    const size_t at_b = after_a + (size_t)(((uintptr_t)dst_b - (uintptr_t)(e->pinned_small_dev + after_a)) & 15u);
    memcpy(static_cast<char*>(e->pinned_small) + at_a, prefix.data(), prefix.size());
    memcpy(static_cast<char*>(e->pinned_small) + at_b, suffix.data(), suffix.size());
    HIPCHK(put_text(e->pinned_small_dev + at_a, dst_a, prefix.size(), e->pinned_small_dev + at_b, dst_b, suffix.size(), st));
  }
  const uint32_t tile = emit_tile_bytes(act_bytes, e->scalars.n_valid);
  NEED(e->tile_start, (emit_tile_count(e->prefix_len, act_bytes, tile) + 2) * 4);
  {
    if (e->flags & KTJ_CREATE_TILE_EMIT)
      HIPCHK(emit(mat, e->perm, e->offs.as<uint64_t>(), N, ctx, e->out.as<char>(), e->prefix_len, act_bytes, tile,
                  e->tile_start.as<uint32_t>(), st));
    else
    {
      const int rc = put_activities(e->scalars.n_valid, was_woven(), e->prefix_len);
      if (rc != KTJ_OK) return rc;
    }
  }
  HIPCHK(hipEventRecord(e->ev[EV_EMIT], st));
  HIPCHK(hipStreamSynchronize(st));
  } /* the stepwise rest */
  e->stage_small_used = 0; /* the stream has passed every upload: ring and slots are free from their beginning */
  e->stage_big_used = 0;
  if (!out_device) e->most_needed = std::max(e->most_needed, pass_bytes + (size_t)e->total_bytes);

  /* ---- statistics ---- */
  count_stats(e, N);
  ktj_stats& s = e->stats;
  /* A stage begins with its first kernel's first workgroup, by the device's clock (an event between two
   * kernels leaves the GPU idle for 5 us, on a trace of some thousand records a tenth of the pass); a
   * stage that launched nothing has no time.  Where the host looks at the plan of the sort its wait is part
   * of the sort.  The whole pass is taken by events; emit, the last stage, is what the others leave of it. */
  {
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e->ev[EV_START], e->ev[EV_EMIT]));
    s.stage_ms[KTJ_STAGE_TOTAL_GPU] = ms;
  }
  if (stage_times) {
    HIPCHK(know_wall_clock(e));
    const unsigned long long* ck = e->scalars.clock;
    const int stages[] = {KTJ_STAGE_DICT, KTJ_STAGE_DECODE, KTJ_STAGE_JOIN, KTJ_STAGE_SORT, KTJ_STAGE_SIZE, KTJ_STAGE_SCAN};
    static_assert(sizeof stages / sizeof stages[0] == KTJ_CLOCK_COUNT - 1, "a stage between every two of the clock's points");
    unsigned long long end = ck[KTJ_CLOCK_EMIT];
    for (int k = KTJ_CLOCK_COUNT - 2; k >= 0; --k)
      if (ck[k]) { s.stage_ms[stages[k]] = clock_ms(e, ck[k], end); end = ck[k]; }
    s.stage_ms[KTJ_STAGE_EMIT] = std::max(0.0f, s.stage_ms[KTJ_STAGE_TOTAL_GPU] - clock_ms(e, ck[KTJ_CLOCK_BEGIN], ck[KTJ_CLOCK_EMIT]));
  }
  e->processed = true;
  return KTJ_OK;
}

/* A pass that ends early leaves nothing behind on the device: neither launches that still read the caller's records
 * or use the scratch array, which are theirs and another engine's again when the call returns, nor small tables on
 * their way into that array. */
static int run_pass(ktj_engine* e, int64_t end_time_ns, void* out_device, uint64_t out_cap) {
  const bool failed_before = e->hip_failed;
  auto pass = [&]() {
    e->hip_error = hipSuccess;
    const int rc = process_pass(e, end_time_ns, out_device, out_cap);
    if (rc != KTJ_OK) {
      (void)put_pending_pieces(e);
      (void)hipStreamSynchronize(e->stream);
    }
    return rc;
  };
  int rc = pass();
  if (rc != KTJ_OK && e->hip_error == hipErrorOutOfMemory && e->rows_are_text) { /* as many records as without text rows */
    (void)hipGetLastError();
    e->pool.release();
    e->hip_failed = failed_before;
    e->no_room_for_text = true; /* until other records are submitted: the next pass begins with what has fitted */
    rc = pass();
    if (rc != KTJ_OK) e->no_room_for_text = false;
  }
  return rc;
}

int ktj_process(ktj_engine* e, int64_t end_time_ns) {
  if (!e) return KTJ_ERR_ARG;
  if (e->bad_sink) return KTJ_OK;
  const int flushed = flush_sdk_api_rows(e);
  if (flushed != KTJ_OK) return flushed;
  e->noalloc = false;
  return run_pass(e, end_time_ns, nullptr, 0);
}

/* The pass with no allocation in it: working memory is this GPU's copy of the static scratch
 * array, the document goes to the caller's buffer, small tables and read-backs go through the
 * pinned buffers that ktj_create allocated. */
int ktj_process_noalloc(ktj_engine* e, int64_t end_time_ns, void* out_device, uint64_t out_capacity, uint64_t* n_bytes) {
  if (n_bytes) *n_bytes = 0;
  if (!e || !out_device || ((uintptr_t)out_device & 15u) != 0) return KTJ_ERR_ARG;
  if (e->bad_sink) return KTJ_OK;
  if (!e->arena) { e->last_error = "ktj_process_noalloc: no scratch array on this device"; return KTJ_ERR_STATE; }
  if (!e->sdk_api_rows.empty() || !e->sdk_api_ext.empty() || !e->sdk_api_user.empty()) {
    e->last_error = "ktj_process_noalloc: rows of ktj_submit_sdk_api_record are still buffered on the host (call ktj_flush first: it may allocate)";
    return KTJ_ERR_STATE;
  }
  if (e->usercorr.n != 0) {
    e->last_error = "ktj_process_noalloc: user-domain correlation records (GPU user annotations) are not supported here";
    return KTJ_ERR_LIMIT;
  }
  e->noalloc = true;
  const int rc = run_pass(e, end_time_ns, out_device, out_capacity);
  e->noalloc = false;
  /* The small tables of this pass sit in the scratch array, which every engine on this GPU shares:
   * whatever the pass returned, the next allocating pass must upload them into its own buffers again. */
  e->schemas_dirty = e->api_dirty = e->coll_dirty = true;
  for (DevBuf* b : {&e->d_fields, &e->d_schemas, &e->d_cid_names, &e->d_flow_bits, &e->d_coll_blob, &e->d_coll_off}) b->unborrow();
  if (n_bytes) *n_bytes = e->total_bytes; /* on KTJ_ERR_LIMIT for a short output buffer: the size that is needed */
  return rc;
}

int ktj_output_device(ktj_engine* e, const void** device_ptr, uint64_t* n_bytes) {
  if (!e || !device_ptr || !n_bytes) return KTJ_ERR_ARG;
  if (!e->processed) return KTJ_ERR_STATE;
  *device_ptr = e->out.p;
  *n_bytes = e->total_bytes;
  return KTJ_OK;
}

int ktj_output_host(ktj_engine* e, const char** host_ptr, uint64_t* n_bytes) {
  if (!e || !host_ptr || !n_bytes) return KTJ_ERR_ARG;
  if (!e->processed) return KTJ_ERR_STATE;
  HIPCHK(hipSetDevice(e->device));
  if (!e->host_copy_valid) {
    if (e->total_bytes > e->pinned_out_cap) {
      if (e->pinned_out) HIPCHK(hipHostFree(e->pinned_out));
      e->pinned_out = nullptr; e->pinned_out_cap = 0;
      void* p = nullptr;
      HIPCHK(hipHostMalloc(&p, e->total_bytes + 4096, hipHostMallocDefault));
      e->pinned_out = static_cast<char*>(p);
      e->pinned_out_cap = e->total_bytes + 4096;
    }
    HIPCHK(hipEventRecord(e->ev_d2h[0], e->stream));
    HIPCHK(hipMemcpyAsync(e->pinned_out, e->out.p, e->total_bytes, hipMemcpyDeviceToHost, e->stream));
    HIPCHK(hipEventRecord(e->ev_d2h[1], e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e->ev_d2h[0], e->ev_d2h[1]));
    e->stats.stage_ms[KTJ_STAGE_D2H] = ms;
    e->stats.stage_bytes[KTJ_STAGE_D2H] = e->total_bytes;
    e->host_copy_valid = true;
  }
  *host_ptr = e->pinned_out;
  *n_bytes = e->total_bytes;
  return KTJ_OK;
}

/* A document on its way to the host goes through the pinned slots, never through a pinned buffer of its
 * own size: pinning and unpinning such a buffer, and the faults of its pages, cost more than the copy
 * (60 MB: 15 ms of the 15.7 ms that a session took). */

/* The parts of a document crossing the link: copy_parts is launched for half of the slots at a time,
 * whenever the half's previous parts have been taken. */
struct DocumentParts {
  ktj_engine* e;
  uint64_t n, part, n_parts, seq, launched = 0;
  uint32_t slots;
  explicit DocumentParts(ktj_engine* e_) : e(e_), n(e_->total_bytes) {
    /* short documents in short parts: the first is there sooner, and the last is soon taken */
    part = n < (2ull << 20) ? 128u << 10 : n < (8ull << 20) ? 256u << 10 : 512u << 10;
    slots = (uint32_t)std::min<uint64_t>(KTJ_PART_SLOTS, KTJ_STAGE_SLOTS * KTJ_STAGE_SLOT / part);
    n_parts = (n + part - 1) / part;
    seq = e->part_seq;
    e->part_seq += n_parts;
  }
  size_t len(uint64_t c) const { return (size_t)std::min<uint64_t>(part, n - c * part); }
  const char* data(uint64_t c) const { return e->stage_big + (c % slots) * part; }
  bool here(uint64_t c) const { return __atomic_load_n(&e->h_ctl->part_flag[c % slots], __ATOMIC_ACQUIRE) == seq + c; }
  /* may the next parts be launched once `taken` parts have left their slots? */
  bool room(uint64_t taken) const { return launched < n_parts && launched + slots / 2 <= taken + slots; }
  hipError_t launch() {
    const uint64_t last = std::min<uint64_t>(launched + slots / 2, n_parts);
    const hipError_t err = copy_parts(e->out.as<char>(), n, launched, last, part, slots, e->stage_big_dev, e->h_ctl_dev->part_flag, seq,
                                      e->d_scalars.as<Scalars>()->part_done, e->stream);
    launched = last;
    return err;
  }
  /* part c is waited for: a launch that failed must not be waited for forever */
  hipError_t wait(uint64_t c) const {
    Patience patience;
    for (unsigned naps = 0; !here(c);)
      if (patience.pause() && ++naps % 8 == 0) {
        const hipError_t q = hipStreamQuery(e->stream);
        if (q != hipErrorNotReady && !here(c)) return q == hipSuccess ? hipErrorUnknown : q;
      }
    return hipSuccess;
  }
};

/* into a caller's memory: this thread has the parts sent and sees them arrive, the others copy them out of
 * their slots (one thread's copy is slower than the link, and the destination's pages are often new:
 * the threads share its faults) */
#define KTJ_COPY_OUT_PER_THREAD (3ull << 20) /* a thread costs some 10 us to start: not worth it for less */
#define KTJ_COPY_OUT_THREADS 6
#define KTJ_COPY_OUT_ONE (512u << 10)
static int copy_document_out(ktj_engine* e, char* dst) {
  int rc = drain_stage(e);
  if (rc == KTJ_OK) rc = ensure_stage(e, KTJ_STAGE_SLOTS * KTJ_STAGE_SLOT);
  if (rc != KTJ_OK) return rc;
  if (e->total_bytes <= KTJ_COPY_OUT_ONE) { /* one transfer and one copy: 8 us for 64 KiB, 20 us in parts */
    HIPCHK(hipMemcpyAsync(e->stage_big, e->out.p, e->total_bytes, hipMemcpyDeviceToHost, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    memcpy(dst, e->stage_big, e->total_bytes);
    return KTJ_OK;
  }
  DocumentParts doc(e);
  hipError_t err = hipSuccess;
  while (doc.room(0) && err == hipSuccess) err = doc.launch();
  HIPCHK(err);
  const unsigned n_threads = copy_threads(doc.n, KTJ_COPY_OUT_PER_THREAD, KTJ_COPY_OUT_THREADS);
  PartQueue queue(doc.n_parts);
  std::atomic<uint64_t> left[KTJ_PART_SLOTS]; /* 1 + the last part that was copied out of the slot */
  for (auto& x : left) x.store(0, std::memory_order_relaxed);
  auto copy_one = [&](uint64_t c) {
    memcpy(dst + c * doc.part, doc.data(c), doc.len(c));
    left[c % doc.slots].store(c + 1, std::memory_order_release);
  };
  run_workers(n_threads, [&](unsigned t) {
    uint64_t k;
    if (t != 0) {
      while (queue.take(&k)) copy_one(k);
      return;
    }
    uint64_t taken = 0; /* parts 0 .. taken - 1 have left their slots */
    Patience patience;
    for (uint64_t c = 0; err == hipSuccess;) {
      while (taken < c && left[taken % doc.slots].load(std::memory_order_acquire) > taken) { ++taken; patience = Patience(); }
      if (doc.room(taken)) err = doc.launch();
      else if (c < doc.launched && doc.here(c)) { ++c; queue.arrive(); }
      else if (queue.try_help(&k)) copy_one(k); /* nothing new: help with what is here */
      else if (c < doc.launched) err = doc.wait(c);
      else if (c == doc.n_parts) break; /* all have been there: the others are at the last of them, and are waited for below */
      else patience.pause(); /* the others are at the parts that hold the slots */
    }
    if (err != hipSuccess) queue.give_up();
  });
  const hipError_t done = hipStreamSynchronize(e->stream);
  HIPCHK(err);
  HIPCHK(done);
  return KTJ_OK;
}

int ktj_output_copy(ktj_engine* e, void* dst, uint64_t capacity, uint64_t* n_bytes) {
  if (!e || !n_bytes) return KTJ_ERR_ARG;
  if (!e->processed) return KTJ_ERR_STATE;
  *n_bytes = e->total_bytes;
  if (!dst || capacity < e->total_bytes) return KTJ_ERR_ARG;
  HIPCHK(hipSetDevice(e->device));
  if (e->host_copy_valid) { memcpy(dst, e->pinned_out, e->total_bytes); return KTJ_OK; }
  struct timespec t0, t1;
  clock_gettime(CLOCK_MONOTONIC, &t0);
  const int rc = copy_document_out(e, static_cast<char*>(dst));
  if (rc != KTJ_OK) return rc;
  clock_gettime(CLOCK_MONOTONIC, &t1);
  e->stats.stage_ms[KTJ_STAGE_D2H] = (float)((t1.tv_sec - t0.tv_sec) * 1e3 + (t1.tv_nsec - t0.tv_nsec) * 1e-6);
  e->stats.stage_bytes[KTJ_STAGE_D2H] = e->total_bytes;
  return KTJ_OK;
}

/* into the file: one writer (writers of one file wait for each other on its inode), the next parts
 * crossing meanwhile */
static int stream_document_to_file(ktj_engine* e, int fd, float* copy_wait_ms) {
  int rc = drain_stage(e);
  if (rc == KTJ_OK) rc = ensure_stage(e, KTJ_STAGE_SLOTS * KTJ_STAGE_SLOT);
  if (rc != KTJ_OK) return rc;
  DocumentParts doc(e);
  double waited = 0;
  for (uint64_t c = 0; c < doc.n_parts; ++c) {
    while (doc.room(c)) HIPCHK(doc.launch());
    struct timespec t0, t1;
    clock_gettime(CLOCK_MONOTONIC, &t0);
    HIPCHK(doc.wait(c));
    clock_gettime(CLOCK_MONOTONIC, &t1);
    waited += (t1.tv_sec - t0.tv_sec) * 1e3 + (t1.tv_nsec - t0.tv_nsec) * 1e-6;
    const char* src = doc.data(c);
    size_t left = doc.len(c);
    while (left) {
      const ssize_t w = write(fd, src, left);
      if (w < 0 && errno == EINTR) continue;
      if (w <= 0) { (void)hipStreamSynchronize(e->stream); return KTJ_ERR_IO; }
      src += w; left -= (size_t)w;
    }
  }
  HIPCHK(hipStreamSynchronize(e->stream));
  if (copy_wait_ms) *copy_wait_ms = (float)waited;
  return KTJ_OK;
}

int ktj_finalize(ktj_engine* e, int64_t end_time_ns, uint64_t* bytes_written) {
  if (!e) return KTJ_ERR_ARG;
  if (bytes_written) *bytes_written = 0;
  if (e->bad_sink) { /* output_json.cpp:1067-1070 */
    e->last_error = "Failed to write to log file!";
    return KTJ_ERR_IO;
  }
  int rc = ktj_process(e, end_time_ns);
  if (rc != KTJ_OK) return rc;
  if (e->flags & KTJ_CREATE_NO_FILE) {
    if (bytes_written) *bytes_written = e->total_bytes;
    return KTJ_OK;
  }
  HIPCHK(hipSetDevice(e->device));
  const uint64_t n = e->total_bytes;
  struct timespec t0, t1;
  clock_gettime(CLOCK_MONOTONIC, &t0);
  if (!e->sink) return KTJ_ERR_STATE;
  float copy_wait_ms = 0;
  rc = fflush(e->sink) == 0 ? stream_document_to_file(e, fileno(e->sink), &copy_wait_ms) : KTJ_ERR_IO;
  const int crc = fclose(e->sink);
  e->sink = nullptr;
  if (rc == KTJ_ERR_IO || (rc == KTJ_OK && crc != 0)) { e->last_error = "short write to " + e->tmp_path; return KTJ_ERR_IO; }
  if (rc != KTJ_OK) return rc;
  e->stats.stage_ms[KTJ_STAGE_D2H] = copy_wait_ms; /* time the writer waited for copies */
  e->stats.stage_bytes[KTJ_STAGE_D2H] = n;
  remove(e->out_path.c_str()); /* output_json.cpp:1100-1107 */
  if (rename(e->tmp_path.c_str(), e->out_path.c_str()) != 0) {
    e->last_error = "Failed to rename " + e->tmp_path + " to " + e->out_path + ": " + strerror(errno);
    return KTJ_ERR_IO;
  }
  clock_gettime(CLOCK_MONOTONIC, &t1);
  e->stats.stage_ms[KTJ_STAGE_FILE] = (float)((t1.tv_sec - t0.tv_sec) * 1e3 + (t1.tv_nsec - t0.tv_nsec) * 1e-6);
  e->stats.stage_bytes[KTJ_STAGE_FILE] = n;
  if (bytes_written) *bytes_written = n;
  return KTJ_OK;
}

int ktj_get_stats(ktj_engine* e, ktj_stats* out) {
  if (!e || !out) return KTJ_ERR_ARG;
  *out = e->stats;
  return KTJ_OK;
}

void ktj_debug_force_sort_passes(int on) { sort_packed_force_passes(on != 0); }

int ktj_debug_fail_allocations(int n) { return std::max(g_failing_allocations.exchange(n), 0); }

int ktj_debug_copy_reference(ktj_engine* e, uint64_t n_bytes, float* ms) {
  if (!e || !ms) return KTJ_ERR_ARG;
  HIPCHK(hipSetDevice(e->device));
  DevBuf a, b;
  HIPCHK(a.ensure(n_bytes));
  HIPCHK(b.ensure(n_bytes));
  HIPCHK(hipMemsetAsync(a.p, 1, n_bytes, e->stream));
  HIPCHK(copy_reference(a.p, b.p, n_bytes, e->stream)); /* warm-up */
  HIPCHK(hipEventRecord(e->ev_d2h[0], e->stream));
  HIPCHK(copy_reference(a.p, b.p, n_bytes, e->stream));
  HIPCHK(hipEventRecord(e->ev_d2h[1], e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  HIPCHK(hipEventElapsedTime(ms, e->ev_d2h[0], e->ev_d2h[1]));
  a.release();
  b.release();
  return KTJ_OK;
}

int ktj_debug_fetch(ktj_engine* e, int what, void* dst, uint64_t cap, uint64_t* n_bytes) {
  if (!e || !n_bytes) return KTJ_ERR_ARG;
  if (!e->processed) return KTJ_ERR_STATE;
  if (what == KTJ_DBG_PASS || what == KTJ_DBG_SORT) { /* (say what the last pass did: make none) */
    const void* info = what == KTJ_DBG_PASS ? e->pass_info : e->sort_info;
    *n_bytes = what == KTJ_DBG_PASS ? sizeof e->pass_info : sizeof e->sort_info;
    if (dst) memcpy(dst, info, std::min<uint64_t>(*n_bytes, cap));
    return KTJ_OK;
  }
  const bool as_text = what == KTJ_DBG_MAT && e->rows_are_text;
  const bool not_kept = (what == KTJ_DBG_COL_DUR || what == KTJ_DBG_COL_EXT) && !e->columns_are_all;
  if (e->small_last || as_text || not_kept) { /* a small pass keeps none of these: the launches of a large trace make them (and the same document) */
    e->no_small = true;
    e->no_weave = what == KTJ_DBG_MAT;
    e->all_columns = true;
    const int rc = ktj_process(e, e->last_end_time);
    e->no_small = e->no_weave = e->all_columns = false;
    if (rc != KTJ_OK) return rc;
  }
  const void* src = nullptr;
  uint64_t n = 0;
  const uint64_t N = e->N;
  switch (what) {
    case KTJ_DBG_COL_TS: src = e->c_ts.p; n = N * 8; break;
    case KTJ_DBG_COL_DUR: src = e->c_dur.p; n = N * 8; break;
    case KTJ_DBG_COL_DEV: src = e->c_dev.p; n = N * 8; break;
    case KTJ_DBG_COL_RES: src = e->c_res.p; n = N * 8; break;
    case KTJ_DBG_COL_META: src = e->c_meta.p; n = N * 4; break;
    case KTJ_DBG_COL_EXT: src = e->c_ext.p; n = N * 4; break;
    case KTJ_DBG_PERM: src = e->perm; n = N * 4; break;
    case KTJ_DBG_LEN: src = e->len_sorted.p; n = N * 4; break;
    case KTJ_DBG_OFFS: src = e->offs.p; n = (N + 1) * 8; break;
    case KTJ_DBG_MAT: src = e->mat.p; n = N * sizeof(MatRow); break;
    case KTJ_DBG_SORT_KEYS:
      if (!e->sorted_keys) { e->last_error = "the sorted keys exist only in an engine created with KTJ_CREATE_PAIR_SORT"; return KTJ_ERR_STATE; }
      src = e->sorted_keys; n = N * 8; break;
    case KTJ_DBG_NAME_VIEW: case KTJ_DBG_NAME_OFF: case KTJ_DBG_ARG_VIEW: case KTJ_DBG_ARG_OFF: {
      /* the views of all strings, one behind the other, and where each begins */
      const bool names = what == KTJ_DBG_NAME_VIEW || what == KTJ_DBG_NAME_OFF;
      std::vector<DictEntry> d(e->n_strings);
      std::vector<char> blob((names ? 2 : 1) * e->blob_bytes + KTJ_DICT_ROOM * (e->n_strings + 1));
      HIPCHK(hipSetDevice(e->device));
      if (!d.empty()) HIPCHK(hipMemcpy(d.data(), e->d_entries.p, d.size() * sizeof(DictEntry), hipMemcpyDeviceToHost));
      if (!d.empty()) HIPCHK(hipMemcpy(blob.data(), names ? e->d_name_blob.p : e->d_arg_blob.p, blob.size(), hipMemcpyDeviceToHost));
      std::string view;
      std::vector<uint64_t> off(1, 0);
      for (const DictEntry& x : d) { view.append(blob.data() + (names ? x.name_off : x.arg_off), names ? x.name_len : x.arg_len); off.push_back(view.size()); }
      const bool text = what == KTJ_DBG_NAME_VIEW || what == KTJ_DBG_ARG_VIEW;
      *n_bytes = text ? view.size() : off.size() * 8;
      if (dst) memcpy(dst, text ? static_cast<const void*>(view.data()) : off.data(), std::min<uint64_t>(*n_bytes, cap));
      return KTJ_OK;
    }
    default: return KTJ_ERR_ARG;
  }
  *n_bytes = n;
  if (dst && src && n) {
    HIPCHK(hipSetDevice(e->device));
    HIPCHK(hipMemcpy(dst, src, n < cap ? n : cap, hipMemcpyDeviceToHost));
  }
  return KTJ_OK;
}

}  // extern "C"
