/*
 * gpu_stages.h — launch interface between the host side of the engine (engine.cpp) and the HIP
 * kernels (kernels.hip).  Every function only enqueues work on the given stream and returns the
 * HIP status of the launch; none of them synchronises or allocates.
 */
#ifndef KTJ_GPU_STAGES_H_
#define KTJ_GPU_STAGES_H_

#include <hip/hip_runtime_api.h>

#include "mat_core.h"
#include "weave_core.h"

namespace ktj {
namespace gpu {

/* Join tables in device memory.  A table maps a 64-bit key to a slot index; what is stored per
 * slot lives in separate arrays indexed by it: compact 4-byte arrays for the "winner" indices that
 * are updated with atomics (atomics on neighbouring addresses coalesce; on 48-byte strides they
 * were measured 20 times slower), and payload arrays that the winners fill with plain stores.
 * A table is either direct-addressed (slot = key - base, chosen on the GPU when the keys that
 * will be inserted span less than the capacity: correlation ids are dense counters in practice,
 * so rows that arrive in id order touch consecutive slots and nothing is probed) or an
 * open-addressing hash table over `keys` (any other key set).  A hash slot is free while its key
 * is KTJ_EMPTY_KEY; slot `cap` (one past the power-of-two range) is reserved for the key whose
 * value equals KTJ_EMPTY_KEY.  The mode lives in device memory (TableCtl) so that no host round
 * trip is needed to choose it.  In direct mode a table with keyed_direct == 0 does not touch
 * `keys` at all: an id inside the range that was never inserted simply has empty per-slot
 * values. */
#define KTJ_EMPTY_KEY 0xFFFFFFFFFFFFFFFFULL
struct KeyRange {          /* over the keys that will be inserted; empty while lo > hi */
  unsigned long long lo, hi;
};
struct TableCtl {
  uint64_t base;           /* direct mode: smallest key */
  uint64_t span;           /* direct mode: largest key - base */
  uint32_t direct;
  uint32_t no_heads;       /* narrow table: NarrowCols::head is not used */
};
struct Table {
  uint64_t* keys;          /* cap + 1 */
  uint32_t mask;           /* cap - 1, cap a power of two >= 16: slots that direct mode can have; the one behind them is the reserved key's */
  uint32_t runs;           /* hash mode: runs of sixteen slots that are used, a power of two or a prime, all below cap */
  uint32_t keyed_direct;   /* 1: a plain set, membership is told by the stored key in both modes */
  const TableCtl* ctl;
};
/* per slot of the table keyed by the full correlation id */
struct FullPay {           /* published by the winning runtime row, read by device rows */
  int64_t first_ts;        /* timestamp of the first runtime row with this id                   */
  uint64_t stream;         /* stream of row stream_src[slot]; 0 = no row carries one            */
};                         /* 16 bytes */
struct FullCols {
  uint32_t* has_runtime;   /* one bit per slot: some runtime row has this id.  Runtime rows arrive
                              before device rows, so where the bit is set the first row of the id is
                              a runtime row and its timestamp is in the payload; the bitmap is small
                              enough to stay in cache, unlike the array of first rows              */
  uint32_t* first;         /* smallest arrival index seen with this id, 0xFFFFFFFF = none (atomicMin);
                              filled for runtime rows only where they share ids, and for device rows
                              whose id no runtime row has                                          */
  uint32_t* stream_src;    /* last runtime row (index + 1) that carries a stream (atomicMax)    */
  FullPay* pay;
};
/* per slot of the table keyed by the int-narrowed correlation id (and by the external-correlation
 * records' full id) */
struct NarrowPay {         /* two writers (external-correlation records, runtime rows), in different passes */
  int32_t ext_val;         /* external id if a CPU op with that id exists, else 0               */
  uint32_t info;           /* bits 0-1: KTJ_DL_HAS_SIZE / KTJ_DL_HAS_GRID, what pay[] holds;
                              bit 2: ext_val names an existing CPU op; bits 3-31: 1 + index of the
                              collective metadata of the linked CPU op, 0 = none                  */
  uint64_t pay[3];         /* bytes of the winning copy / malloc row in pay[0], or packed grid /
                              workgroup of the winning kernel-launch row (see pack_grid)        */
};                         /* 32 bytes: a slot never straddles a line */
/* What the external-correlation records leave, by itself: a row that reads it has 16 slots to a line instead of four, and only these
 * have to be cleared.  Every runtime row writes all of its slot's NarrowPay, these two words as well, and a device row believes that where
 * FullCols::has_runtime has its id and reads the head otherwise.  This takes that the narrow slot is the full id's: with ids beyond
 * 31 bits (and where there is no room for the heads) NarrowPay is cleared, and has the records' two words from the start (TableCtl::no_heads).
 * 22 million records: k_plan_clear 91 -> 42 us, k_build_extcorr 151 -> 72, k_join_runtime 1098 -> 1124 (it no longer has
 * in the cache what it writes to); 3 million: 15 -> 9, 13 -> 9, 94 -> 81, and 77 -> 69 where no launch hands anything over, whose rows write
 * 32 bytes here that they did not write before. */
struct NarrowHead { int32_t ext_val; uint32_t info; };
#define KTJ_NP_KIND_MASK 3u
#define KTJ_NP_LINKED 4u
#define KTJ_NP_COLL_SHIFT 3
#define KTJ_MAX_COLLECTIVES ((1u << 29) - 2u)
struct NarrowCols {
  uint32_t* ext_src;       /* last external-correlation record (index + 1), 0 = none            */
  uint32_t* kern_src;      /* last in-window kernel-launch row (index + 1)                     */
  uint32_t* copy_src;      /* last in-window copy / malloc row (index + 1)                     */
  NarrowPay* pay;
  NarrowHead* head;        /* or none */
};
#define KTJ_TBL_FULL 0
#define KTJ_TBL_NARROW 1
#define KTJ_TBL_CPU 2
struct JoinPlan {
  KeyRange range[3];
  TableCtl ctl[3];
};
/* what a device row takes over from the runtime row(s) with its correlation id */
struct DevLink {
  uint64_t p[3];           /* size in p[0], or packed grid / workgroup */
  uint32_t flags;          /* KTJ_DL_* */
  uint32_t coll;           /* 1 + index of the collective metadata of the linked CPU op (kernels) */
};                         /* 32 bytes */
#define KTJ_DL_HAS_SIZE 1u
#define KTJ_DL_HAS_GRID 2u
/* The same for many rows, each value by itself: most rows of graph launches take nothing over, and the values that a wavefront's rows
 * have none of are neither stored nor loaded (11 million kernels of graphs: k_link_device 227 -> 167 us, k_mat_rows 558 -> 505; where all rows
 * have a grid 4 bytes a row less). */
struct Links {
  uint64_t* p[3];          /* [0] where KTJ_DL_HAS_SIZE or KTJ_DL_HAS_GRID, the others where KTJ_DL_HAS_GRID */
  uint32_t* info;          /* KTJ_DL_* | coll << KTJ_NP_COLL_SHIFT */
};
inline Links links_in(void* memory /* n DevLinks */, uint64_t n) {
  uint64_t* const w = static_cast<uint64_t*>(memory);
  return Links{{w, w + n, w + 2 * n}, reinterpret_cast<uint32_t*>(w + 3 * n)};
}

/* Columns in arrival order: generic rows, then runtime rows, then device rows.  Where a row's record is read again anyway, for its
 * joined row, duration and correlation id come from there, and nothing reads the "External id" of rows that are no device rows
 * here: 12 to 20 bytes a row that are neither written nor read (22 million records 7995 -> 7850 us, 11 million 3695 -> 3655, 5 million with long strings 3680 -> 3655). */
struct Columns {
  int64_t* ts;    /* raw begin, after convert: timestamp()          */
  int64_t* dur;   /* raw end, after convert: duration(); only with all */
  uint64_t* corr; /* correlation id; of others than device rows only with all */
  int64_t* dev;   /* deviceId()                                      */
  int64_t* res;   /* resourceId(); device rows: stream before and after back-fill */
  uint32_t* meta; /* KTJ_M_VALID | class                              */
  int32_t* ext;   /* "External id" value; of others than device rows only with all */
  bool all;       /* user annotations and ktj_debug_fetch read these */
};

/* small block of scalars the kernels update and the host reads back */
#ifndef KTJ_COUNTER_SHARDS
#define KTJ_COUNTER_SHARDS 64u
#endif
#define KTJ_PART_SLOTS 32u
struct SortPlan { /* of the composite key */
  unsigned int ts_bits, res_bits, key_bits, low_bits; /* .., of all of it, of what the passes may leave to sort_finish */
  unsigned int n_dev;                                 /* dropped rows have this device's rank */
};
/* wall clock (wall_clock64) at the points of a pass: its start and the start of each stage; the runs of
 * small.hip name their own */
enum { KTJ_CLOCK_BEGIN = 0, KTJ_CLOCK_DECODE, KTJ_CLOCK_JOIN, KTJ_CLOCK_SORT, KTJ_CLOCK_SIZE, KTJ_CLOCK_SCAN, KTJ_CLOCK_EMIT, KTJ_CLOCK_COUNT };
#define KTJ_RANGE_TS 4 /* place of the timestamps' range (biased) behind those of the join tables in Scalars::range_shard */
enum { KTJ_DONE_DENSE = 0, KTJ_DONE_COLLECT, KTJ_DONE_COUNT };
struct Scalars {
  unsigned long long ts_min_biased;   /* min over valid rows of ts ^ 2^63 */
  unsigned long long ts_max_biased;
  unsigned long long out_of_range;
  unsigned long long out_of_order;
  unsigned long long n_flow;
  unsigned long long n_linked;
  unsigned long long n_blank_names;
  unsigned long long n_valid;
  unsigned long long n_unresolved;    /* device rows still without a stream after the correlation pass */
  unsigned long long n_sync_typed;    /* generic rows of type CUDA_SYNC */
  unsigned long long n_device_orphans; /* in-window device rows whose id no runtime row has */
  unsigned int error;                 /* KTJ_DEVERR_* bits */
  unsigned int have_stream_src;       /* some runtime row carries a stream */
  unsigned int n_dev_ranks;           /* distinct deviceId values */
  unsigned int n_res_ranks;           /* distinct resourceId values */
  unsigned int n_dense;               /* distinct (device, stream key) pairs */
  unsigned int runtime_ids_repeat;    /* two runtime rows share a slot of the full table */
  unsigned int n_queues;              /* distinct hardware queues entered into the queue -> stream table */
  unsigned int n_sync_rows;           /* distinct (device, row) pairs of Stream Sync activities */
  unsigned int n_plain;               /* small traces: activities that small_emit leaves to small_plain */
  unsigned int n_left;                /* activities that weave leaves to emit_direct */
  unsigned int no_text;               /* it leaves them all (too_many_left); n_left is 0 then */
  unsigned int ext_ids_repeat;        /* two external-correlation records share a correlation id */
  unsigned long long emit_rows;       /* activities to format: n_valid, or none where the pass cannot end so */
  unsigned long long clock[KTJ_CLOCK_COUNT];
  SortPlan sort;
  unsigned int done[KTJ_DONE_COUNT];  /* workgroups of a launch that have finished (last_workgroup) */
  unsigned int part_done[KTJ_PART_SLOTS]; /* copy_parts: workgroups that have finished the part in a slot */
  alignas(256) JoinPlan plan;         /* key ranges and modes of the join tables: read by every row of the join
                                         kernels, so kept off the cache lines that take the counters' atomics */
  /* The counters that most workgroups add to (KTJ_CNT_*) are kept in KTJ_COUNTER_SHARDS copies, one
   * 128-byte line each; a workgroup adds to the copy of its index.  Atomics on one address are carried
   * out one after the other, and tens of thousands of workgroups adding to the same few words cost the
   * join more than its table lookups.  publish_scalars sums the copies into the fields above, of which the
   * device reads emit_rows only, and hands the host everything in front of this array. */
  alignas(128) unsigned long long shard[KTJ_COUNTER_SHARDS][16];
  alignas(128) unsigned long long range_shard[KTJ_COUNTER_SHARDS][16]; /* likewise the key ranges of the join tables: [2t] smallest,
                                                                           [2t + 1] largest key of table t */
};
enum { KTJ_CNT_OUT_OF_RANGE = 0, KTJ_CNT_OUT_OF_ORDER, KTJ_CNT_FLOW, KTJ_CNT_LINKED, KTJ_CNT_BLANK_NAMES, KTJ_CNT_VALID,
       KTJ_CNT_SYNC_TYPED, KTJ_CNT_COUNT,
       KTJ_CNT_NOT_TEXT = KTJ_CNT_COUNT }; /* (not the host's) printed rows that can be no text rows (left_generic and the following) */
#define KTJ_DEVERR_TABLE_FULL 1u         /* a join table sized from the record counts filled up (a defect) */
#define KTJ_DEVERR_DISTINCT_DEVICES 2u   /* more distinct deviceId values than the rank set holds: the sort
                                            takes its slower path without ranks, no error reaches the caller */
#define KTJ_DEVERR_HASH_COLLISION 4u
#define KTJ_DEVERR_RECORD_TOO_LONG 8u
#define KTJ_DEVERR_DISTINCT_RESOURCES 16u /* as DISTINCT_DEVICES, for resourceId values */
#define KTJ_DEVERR_STREAMS 32u            /* more than KTJ_MAX_STREAM_PAIRS (device, stream) pairs */
#define KTJ_DEVERR_QUEUES 64u             /* more than KTJ_MAX_QUEUES hardware queues */
#define KTJ_DEVERR_SYNC_ROWS 128u         /* more than KTJ_MAX_SYNC_ROWS (device, row) pairs of Stream Sync events */

#define KTJ_DEVERR_UNSORTED 1024u         /* the sort's passes have to take all bits; no error reaches the caller */
#define KTJ_DEVERR_CAREFUL 512u           /* the pass went by assumptions that do not hold; no error reaches the caller */
#define KTJ_DEVERR_SMALL_UNFIT 256u       /* a small trace that needs the launches of a large one; no error reaches the caller */

#define KTJ_SET_CAP 16384u     /* slots of the distinct-value sets; KTJ_SET_MAX values get a rank */
#define KTJ_SET_MAX 4096u
#define KTJ_DENSE_CAP (2u * KTJ_MAX_STREAM_PAIRS) /* slots of the (device, stream) table */
#define KTJ_QUEUE_CAP (2u * KTJ_MAX_QUEUES)       /* slots of the queue -> stream table */
#define KTJ_SYNC_CAP (2u * KTJ_MAX_SYNC_ROWS)     /* slots of the Stream Sync (device, row) table */
#define KTJ_TABLE_PROBES 256u  /* linear probing of these small tables gives up after this many slots: a backstop,
                                  the documented limits are enforced by counting the distinct keys */

struct ApiTable {
  const uint32_t* cid_name_ids;
  uint32_t n_cids;
  const uint32_t* flow_start_bits; /* bitmap over cids */
  uint32_t malloc_cid;
};

/* read-backs and text of a pass without the copy engine: sc, *total (may be null) and list[0..n_list)
 * into pinned host memory (device-visible addresses); two pieces of host text to their places in the
 * document (source and destination of a piece must agree modulo 16) */
hipError_t publish(Scalars* sc, const uint64_t* total, const uint32_t* list, uint32_t n_list, Scalars* h_sc,
                   uint64_t* h_total, uint32_t* h_list, hipStream_t st);
hipError_t put_text(const char* src_a, char* dst_a, uint64_t n_a, const char* src_b, char* dst_b, uint64_t n_b, hipStream_t st);
/* pieces of page-locked host memory to their places in device memory, in one launch */
#define KTJ_MAX_PIECES 16u
struct PieceJobs {
  const char* src[KTJ_MAX_PIECES];
  char* dst[KTJ_MAX_PIECES];
  uint64_t n[KTJ_MAX_PIECES];
  uint32_t count;
};
hipError_t put_pieces(const PieceJobs& jobs, hipStream_t st);
/* Parts first .. last - 1 of n bytes of device memory into page-locked slots, part c (part_bytes long, the
 * last one what is left) into slot c % n_slots at `slots + slot * part_bytes`; as soon as a part is there
 * flag[slot] becomes seq + c.  src and slots 16-byte aligned, up to 15 bytes behind n are read; n_slots
 * <= KTJ_PART_SLOTS; done: Scalars::part_done. */
hipError_t copy_parts(const char* src, uint64_t n, uint64_t first, uint64_t last, uint64_t part_bytes, uint32_t n_slots, char* slots,
                      uint64_t* flag, uint64_t seq, unsigned int* done, hipStream_t st);
/* ---- utilities ---- */
hipError_t fill_u64(uint64_t* p, uint64_t v, uint64_t n, hipStream_t st);
hipError_t fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t st);
struct FillJobs {          /* up to 12 fills in one launch */
  void* p[12];
  uint64_t value[12];
  uint64_t n[12];
  uint32_t bytes_each[12]; /* 4 or 8 */
  uint32_t count;
  void add(void* ptr, uint64_t v, uint64_t elems, uint32_t width) { p[count] = ptr; value[count] = v; n[count] = elems; bytes_each[count] = width; ++count; }
};
hipError_t copy_reference(const void* src, void* dst, uint64_t bytes, hipStream_t st);

/* Working memory for callers that cannot allocate: a static array in device memory, one copy per
 * GPU, KTJ_NOALLOC_SCRATCH_BYTES long.  Returns the address of the copy on `device` (which must be
 * the current device); the address is looked up once per device and kept. */
hipError_t scratch_address(int device, void** ptr, size_t* bytes);

/* exclusive scan in place; tmp must hold scan_tmp_elems(n) uint64 values */
uint64_t scan_tmp_elems(uint64_t n);
hipError_t scan_u32_inplace(uint32_t* data, uint64_t n, uint64_t* tmp, hipStream_t st);

/* ---- start of a pass: scalars, fills, and stage 0, the dictionary's views ----
 * entries: n_strings; name_blob: 2 * blob bytes + KTJ_DICT_ROOM * (n + 1), arg_blob: blob bytes + KTJ_DICT_ROOM * (n + 1) */
hipError_t begin_pass(Scalars* s, const FillJobs& jobs, const char* blob, const uint64_t* off, uint32_t n_strings, DictEntry* entries,
                      char* name_blob, char* arg_blob, hipStream_t st);

/* ---- stage 1: decode, with the clock conversion and the capture window (stage 2a) ---- */
struct DecodeJob {
  const ktj_generic_rec* g; const ktj_runtime_rec* r; const ktj_device_rec* d; const ktj_extcorr_rec* x;
  uint64_t ng, nr, nd, nx;   /* x: only their correlation ids' range */
  uint64_t first;            /* arrival index of the first generic record; runtime and device rows follow ng records */
  bool whole_pass;           /* false: generic records made during the pass, which are in no table */
  bool text;                 /* a pass that makes text rows: those that will be none are counted, as far as their records say so */
  uint32_t schemas_not_taken, n_cids;
  uint64_t* queue;           /* of the device rows: what they have instead of a stream, and hardly ever read */
  ClockDev clk;
  int64_t win_start, win_end;
  uint32_t gb, rb, db;       /* set by decode() */
};
hipError_t decode(DecodeJob job, Columns c, EmitCtx ctx, Scalars* sc, hipStream_t st);

/* ---- stage 2b: joins ---- */
/* the tables' modes (direct unless force_hash or the span of their keys is too wide), and all of them cleared */
/* n_rows: of all classes, in a pass that makes text rows (0: it makes none); h_weave: page-locked, what k_decode has counted for the
 * weaver (KTJ_WEAVE_*) */
enum { KTJ_WEAVE_UNKNOWN = 0, KTJ_WEAVE_ALL, KTJ_WEAVE_MOST, KTJ_WEAVE_NONE };
hipError_t plan_tables(Table tf, FullCols fc, Table tn, NarrowCols nc, Table cpu, bool force_hash, uint64_t n_rows, uint32_t* h_weave, Scalars* sc, hipStream_t st);
/* Whether the weaver prints nothing where it would leave n_left of n activities.  Each that it leaves ends what it
 * has begun (a fifth of 120 000 CPU ops instant events: k_weave 43 us instead of 25), and the launch for these is never shorter
 * than 30 us, however few.  Passes of 100 000 / 260 000 / 733 000 / 3 million records with one of them left: woven 266 / 315 / 587 /
 * 1280 us, not woven 254 / 302 / 590 / 1565. */
#define KTJ_FEW_ACTIVITIES 262144u
static inline __host__ __device__ bool too_many_left(uint64_t n_left, uint64_t n) { return n_left != 0 && (n <= KTJ_FEW_ACTIVITIES || n_left * 32u > n); }
hipError_t build_cpu_ids(const ktj_generic_rec* g, uint64_t n, Table cpu, uint32_t* cpu_row, Scalars* sc, hipStream_t st);
/* after build_cpu_ids: enters the external-correlation records and resolves their external ids */
hipError_t build_extcorr(const ktj_extcorr_rec* e, uint64_t n, Table tn, NarrowCols nc, Table cpu, const uint32_t* cpu_row,
                         const ktj_generic_rec* g, EmitCtx ctx, Scalars* sc, hipStream_t st);
hipError_t collective_first(const MatRow* mat, const uint32_t* perm, uint64_t n_rows, uint32_t n_coll, uint32_t* first,
                            hipStream_t st);
/* per device row: "External id", timestamp-order check, stream of the launching row, and the
 * size / grid hand-over (into link[]) */
hipError_t link_device_rows(uint64_t n, Columns c, uint64_t first_device, Table tf, FullCols fc, Table tn, NarrowCols nc,
                            Links link, unsigned long long* orphans /* a bit per row */, Scalars* sc, hipStream_t st);
/* stream back-fill: queue table (keys/vals/ambiguous) and dense table are caller-provided, zeroed */
struct StreamTables {
  uint64_t* q_keys;   /* KTJ_QUEUE_CAP + 1, filled with KTJ_EMPTY_KEY */
  uint64_t* q_stream; /* 0 = unset */
  uint32_t* q_amb;
  uint64_t* d_hash;   /* KTJ_DENSE_CAP + 1, filled with KTJ_EMPTY_KEY */
  uint32_t* d_first;  /* min arrival index, filled with 0xFFFFFFFF */
  int32_t* d_dev;
  uint64_t* d_key;
  uint32_t* d_rank;
  uint32_t* d_list;   /* KTJ_MAX_STREAM_PAIRS: slots of the pairs */
};
/* also checks the device rows whose id no runtime row has (tf, fc, link) */
hipError_t backfill_streams(const uint64_t* queue, uint64_t n, bool assign, Columns c, uint64_t first_device, Table tf, FullCols fc, const unsigned long long* orphans,
                            StreamTables t, Scalars* sc, hipStream_t st);

/* ---- GPU user annotations (GenericActivityProfiler.cpp:277-327, 423-433): one span per
 * (device, resource, annotation id) over the device rows that the user-domain correlation
 * records lead to.  Tables are caller-provided: u_keys (cap_user + 1, KTJ_EMPTY_KEY), u_src (0),
 * and the span table of cap_span + 1 slots: hash (KTJ_EMPTY_KEY), first (0xFFFFFFFF), lo/hi
 * (biased timestamps: lo ~0, hi 0), zero (0). ---- */
struct SpanTables {
  uint64_t* u_keys; uint32_t* u_src; uint32_t u_mask;   /* correlation id -> last user record (index + 1) */
  uint64_t* hash; uint32_t* first; uint64_t* lo; uint64_t* hi; uint32_t* zero; uint32_t mask;
  int32_t* dev; int64_t* res; uint64_t* ext; uint32_t* name;  /* written by the first row of a span */
};
struct SpanOut {            /* one finished span, read back by the host */
  int64_t res;
  uint64_t ext;             /* the annotation's id (key of the CPU-op table) */
  int64_t start, end;       /* min timestamp, max end over the span's rows */
  int32_t dev;
  uint32_t name;            /* string id of the annotation's name */
  uint32_t first;           /* index of the first device row of the span: insertion order */
  uint32_t zero;            /* some row starts at time 0: the start needs the sequential rule */
};                          /* 48 bytes */
struct SpanMember { uint32_t slot, row; int64_t ts; };  /* rows of spans with `zero` set */
hipError_t build_usercorr(const ktj_extcorr_rec* u, uint64_t n, SpanTables t, Scalars* sc, hipStream_t st);
hipError_t group_spans(const ktj_extcorr_rec* u, const ktj_generic_rec* g, uint64_t n_device, Columns c, uint64_t first_device,
                       Table cpu, const uint32_t* cpu_row, SpanTables t, SpanOut* out, uint32_t* n_out, Scalars* sc,
                       hipStream_t st);
hipError_t span_members(const ktj_extcorr_rec* u, uint64_t n_device, Columns c, uint64_t first_device, Table cpu,
                        SpanTables t, SpanMember* out, uint32_t cap_out, uint32_t* n_out, hipStream_t st);

/* ---- stage 3: canonical order ---- */
/* The device rows whose resourceId the sort still has to make of their streams and queues (k_dense_assign has, where n is 0) */
struct Backfill { const uint64_t* queue; uint64_t first_device, n; StreamTables t; };
struct SortSets {
  uint64_t* dev_keys;  /* KTJ_SET_CAP + 1, KTJ_EMPTY_KEY filled */
  uint32_t* dev_rank;
  uint64_t* res_keys;
  uint32_t* res_rank;
  uint32_t* dev_list;  /* KTJ_SET_MAX: slots of the values */
  uint32_t* res_list;
};
/* distinct values and their ranks, and Scalars::sort; straight: the host will not look at anything before
 * the end of the pass, so what needs that is flagged (KTJ_DEVERR_CAREFUL).  book, if not null: what text_row and
 * weave_activities need to know of the schemas, from the dictionary views */
hipError_t collect_distinct(Columns c, uint64_t n, uint64_t n_device, const Backfill& fill, SortSets s, Scalars* sc, bool straight, const EmitCtx& ctx, weave::SchemaBook* book, hipStream_t st);
/* key = ((rank(dev) << res_bits | rank(res)) << ts_bits) | (ts - ts_min); dropped rows get 1 << key_bits */
hipError_t make_keys(Columns c, uint64_t n, SortSets s, const Scalars* sc, uint32_t ts_bits, uint32_t res_bits,
                     uint32_t key_bits, uint64_t* keys, uint32_t* vals, hipStream_t st);
/* for timestamp spans too wide for one composite key: keys = ts - ts_min with vals = arrival
 * index, then keys = composite rank of row order[p] with vals = order[p] (dropped rows get
 * 1 << rank_bits) */
hipError_t make_ts_keys(Columns c, uint64_t n, const Scalars* sc, uint64_t* keys, uint32_t* vals, hipStream_t st);
/* keys[p] = sign-biased column value of row order[p] (validity != 0: 0 for kept rows, 1 for dropped ones) */
hipError_t make_column_keys(const int64_t* column, const uint32_t* meta, const uint32_t* order, uint64_t n, int validity,
                            uint64_t* keys, uint32_t* vals, hipStream_t st);
hipError_t clear_error_bits(Scalars* sc, unsigned int bits, hipStream_t st);
/* With schemas set the rows are TextRows (those that the weaver does not print MatRows in the same places, marked:
 * KTJ_ROW_LEFT, and tail kind KTJ_KIND_LEFT beside their lengths but where Scalars::no_text leaves all); otherwise all are MatRows. */
struct Rows {
  void* p;
  const weave::SchemaBook* schemas;
  weave::WideText* wide; /* of the generic records */
};
/* What mat_rows takes, for the sort: the rows are made in its last launch where it has one that they may come with (made). */
struct RowsJob {
  const ktj_generic_rec* g;
  uint64_t ng;
  const ktj_device_rec* d;
  uint64_t nd;
  Columns c;
  uint64_t first_device;
  Links link;
  ClockDev clk;
  EmitCtx ctx;
  Rows rows;
  uint32_t* len;
  bool made;
};
/* The composite-key sort on single 64-bit words (key above the arrival index); perm receives the
 * arrival index per sorted position.  Usable when sort_packed_fits(n, plan). */
bool sort_packed_fits(uint64_t n, const SortPlan& plan);
bool sort_packed_passes_forced();
bool sort_packed_in_one_launch(uint64_t n); /* which has no use for finish */
void sort_packed_force_passes(bool on); /* tests: no one-launch sort of a single tile */
uint32_t sort_packed_passes(const SortPlan& plan, bool finish); /* finish: the lowest bits are left to a launch behind the passes */
/* key widths come from Scalars::sort; `passes` is how many are launched: those beyond the plan end at once, and
 * a plan that needs more (or does not fit a word) sets KTJ_DEVERR_CAREFUL in Scalars::error */
hipError_t sort_packed(Columns c, uint64_t n, SortSets s, Scalars* sc, uint32_t passes, bool finish, uint64_t* buf_a, uint64_t* buf_b, uint32_t* perm,
                       uint32_t* hist, uint32_t* chain_hist /* 8 bytes per row */, RowsJob* job /* or none */, hipStream_t st);
hipError_t make_rank_keys(Columns c, const uint32_t* order, uint64_t n, SortSets s, uint32_t res_bits, uint32_t rank_bits,
                          uint64_t* keys, uint32_t* vals, hipStream_t st);
/* stable LSD radix sort of (key, val) pairs on the low `bits` bits; result ends in keys_out/vals_out
 * pointers returned through *res_keys / *res_vals (one of the two buffer pairs) */
uint64_t radix_tmp_elems(uint64_t n);
hipError_t radix_sort(uint64_t* keys_a, uint32_t* vals_a, uint64_t* keys_b, uint32_t* vals_b, uint64_t n,
                      uint32_t bits, uint32_t* hist /* radix_tmp_elems(n) */, uint64_t* scan_tmp,
                      uint64_t** res_keys, uint32_t** res_vals, hipStream_t st);

/* ---- stage 4a: joined rows + exact byte length (arrival order) ---- */
#define KTJ_KIND_LEFT 3u
/* keys: KTJ_SYNC_CAP + 1, first_pos: KTJ_SYNC_CAP + 1, is_first: n_generic (all caller-provided);
 * dev: the deviceId column */
hipError_t stream_sync_first(const uint32_t* perm, uint64_t n_sorted, const ktj_generic_rec* g, uint64_t n_generic,
                             const int64_t* dev, DictViews d, uint64_t* keys, uint32_t* first_pos, uint32_t* is_first, Scalars* sc,
                             hipStream_t st);
/* joined rows and lengths of generic records (arrival index first_generic on; sync_first: per record, from
 * stream_sync_first, or null when there are no such rows) and of device records */
hipError_t mat_rows(const ktj_generic_rec* g, uint64_t ng, uint64_t first_generic, const uint32_t* sync_first, const ktj_device_rec* d, uint64_t nd,
                    Columns c, uint64_t first_device, Links link, const ClockDev& clk, EmitCtx ctx, Rows rows, uint32_t* len, Scalars* sc, hipStream_t st);
/* the pass over the runtime rows: publishes what device rows take over (first timestamp, stream, grid,
 * size) into the tables, reads the "External id", makes the joined rows and their lengths; runs
 * after build_extcorr and before link_device_rows */
hipError_t join_runtime_rows(const ktj_runtime_rec* r, uint64_t n, Columns c, uint64_t first, ApiTable api, Table tf, FullCols fc,
                             Table tn, NarrowCols nc, uint32_t* slot_f, uint32_t* slot_n, const ClockDev& clk, EmitCtx ctx, Rows rows,
                             uint32_t* len, Scalars* sc, hipStream_t st);
/* winners write the payload again and repeated ids are checked; returns at once where no two
 * runtime rows share a slot */
hipError_t republish_runtime_rows(const ktj_runtime_rec* r, uint64_t n, Columns c, uint64_t first, FullCols fc, NarrowCols nc,
                                  const uint32_t* slot_f, const uint32_t* slot_n, Scalars* sc, hipStream_t st);
/* lengths and tail kinds in emission order, and the activities' offsets (n + 1).  With text.out set the
 * document's header and footer text go to their places and scalars and total to the host: the emit kernels
 * may follow without the host having seen anything. */
struct DocText {
  const char* prefix; uint64_t n_prefix;   /* page-locked, 16-byte aligned, readable up to the next multiple of 16 */
  const char* suffix; uint64_t n_suffix;
  char* out; uint64_t out_cap;             /* what does not fit with 64 bytes to spare is not written */
  Scalars* h_sc; uint64_t* h_total;        /* page-locked: the scalars in front of the shards, the activities' bytes */
  uint64_t* h_end;                         /* small traces: the wall clock when the last activities were written */
};
uint64_t offsets_tmp_elems(uint64_t n);
/* left: where the places of the rows that are left to emit_direct go (Scalars::n_left of them, at most n) */
hipError_t gather_offsets(const uint32_t* perm, const uint32_t* len, uint64_t n, uint32_t* len_sorted, uint8_t* kind_sorted, uint64_t* sums,
                          uint64_t* offs, uint32_t* left, Scalars* sc, const DocText& text, hipStream_t st);

/* ---- stage 4b: emit ---- */
/* tile size (bytes of output per workgroup) for a document whose activity section has act_bytes
 * bytes in n_rows activities, and the number of tiles / entries of tile_start (tiles + 1) */
uint32_t emit_tile_bytes(uint64_t act_bytes, uint64_t n_rows);
uint64_t emit_tile_count(uint64_t prefix_len, uint64_t act_bytes, uint32_t tile);
hipError_t emit(const MatRow* mat, const uint32_t* perm, const uint64_t* offs /* n+1 */, uint64_t n,
                EmitCtx ctx, char* out, uint64_t prefix_len, uint64_t act_bytes, uint32_t tile,
                uint32_t* tile_start /* tiles + 1 */, hipStream_t st);

/* direct variant: one lane per activity; kind_sorted holds the tail kind of every activity in emission order;
 * Scalars::emit_rows of them, at most n_most.  left: only the Scalars::n_left activities on this list, rows are sizeof(TextRow) apart;
 * all of them, in order, where Scalars::no_text says so */
hipError_t emit_direct(const void* rows, const uint32_t* perm, const uint64_t* offs, const uint8_t* kind_sorted, uint64_t n_most, EmitCtx ctx,
                       char* out, uint64_t prefix_len, const Scalars* sc, const uint32_t* left, hipStream_t st);

/* The activities of rows that are text (TextRow), one lane per segment (weave.hip).  The others, if any, are on the list
 * that gather_offsets made: emit_direct's. */
hipError_t weave_activities(const weave::TextRow* rows, const uint32_t* perm, const uint64_t* offs, const uint8_t* kind_sorted, uint64_t n_most, EmitCtx ctx, char* out,
                 uint64_t prefix_len, const Scalars* sc, const weave::SchemaBook* schemas, const weave::WideText* wide, hipStream_t st);

/* ---- small traces: the whole pass in three launches (small.hip) ---- */
#define SMALL_ROWS 2048u       /* records of the three classes together: what LDS holds the join tables for */
#define SMALL_EXT 2048u        /* external-correlation records */
struct SmallArgs {
  const ktj_generic_rec* g; const ktj_runtime_rec* r; const ktj_device_rec* d; const ktj_extcorr_rec* x;
  uint32_t ng, nr, nd, nx;
  uint32_t slots;              /* small_slots() */
  Columns c;
  DevLink* link;               /* nd */
  ClockDev clk;
  int64_t win_start, win_end;
  EmitCtx ctx;
  DictEntry* entries;
  ApiTable api;
  MatRow* mat; uint32_t* len;  /* per arrival index, as for a large trace */
  uint32_t* perm;
  Scalars* sc;
};
bool small_fits(uint64_t n_generic, uint64_t n_runtime, uint64_t n_device, uint64_t n_ext);
uint32_t small_slots(uint64_t n_generic, uint64_t n_runtime, uint64_t n_device, uint64_t n_ext);
/* decode to order and lengths; then the document.  Scalars::error holds KTJ_DEVERR_SMALL_UNFIT afterwards
 * where the trace needs the launches of a large one: nothing is written then. */
hipError_t small_pass(const SmallArgs& a, uint32_t n_strings, hipStream_t st);
hipError_t small_emit(const SmallArgs& a, const DocText& t, hipStream_t st);
/* behind small_emit where Scalars::n_plain is not zero: the activities that it left out */
hipError_t small_plain(const SmallArgs& a, const DocText& t, hipStream_t st);

}  // namespace gpu
}  // namespace ktj
#endif
