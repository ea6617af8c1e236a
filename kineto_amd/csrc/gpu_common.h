/*
 * gpu_common.h — device helpers shared by the kernels of large traces (kernels.hip) and of small ones
 * (small.hip): hashing, wavefront primitives, and the per-record steps that both take.
 */
#ifndef KTJ_GPU_COMMON_H_
#define KTJ_GPU_COMMON_H_

#include <hip/hip_runtime.h>

#include "gpu_stages.h"

namespace ktj {
namespace gpu {

#define KTJ_NOSLOT 0xFFFFFFFFu
#define KTJ_BLOCK 256

/* ------------------------------------------------------------------------------------------ */
/* helpers                                                                                      */
/* ------------------------------------------------------------------------------------------ */
__device__ __forceinline__ uint64_t hash64(uint64_t x) {
  x ^= x >> 33; x *= 0xff51afd7ed558ccdULL; x ^= x >> 33; x *= 0xc4ceb9fe1a85ec53ULL; x ^= x >> 33;
  return x;
}
__device__ __forceinline__ uint32_t lane_id() { return threadIdx.x & 63u; }
/* Values that a pass streams through once — a row's own columns and records, the rows it writes —
 * are loaded and stored past the L2's usual replacement: what the cache is for in these passes are
 * the table lines that rows reach at random. */
template <typename T> __device__ __forceinline__ T load_once(const T* p) { return __builtin_nontemporal_load(p); }
template <typename T> __device__ __forceinline__ void store_once(T* p, T v) { __builtin_nontemporal_store(v, p); }
__device__ __forceinline__ uint64_t lanemask_lt() { return (1ULL << lane_id()) - 1ULL; }

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ void stage_clock(Scalars* sc, int k) { sc->clock[k] = wall_clock64(); }
__device__ __forceinline__ void flag_error(Scalars* sc, unsigned bit) { atomicOr(&sc->error, bit); }

/* grid-stride kernels: enough workgroups to fill 256 CUs several times over */
#define KTJ_MAX_GRID 4096u
static inline unsigned grid_for(uint64_t n, unsigned per_block) { return (unsigned)((n + per_block - 1) / per_block); }
static inline unsigned grid_stride_for(uint64_t n, unsigned per_block) {
  const uint64_t g = (n + per_block - 1) / per_block;
  return (unsigned)(g < KTJ_MAX_GRID ? g : KTJ_MAX_GRID);
}
#define KTJ_LAUNCH_CHECK() hipGetLastError()


/* Eight bytes of a string at once: a string of a kilobyte (a templated kernel name) is two loads per lane instead of
 * sixteen, one after the other, and its views two stores (2084 strings of 1 KB: k_begin 27 -> 16 us). */
#define BYTES_01 0x0101010101010101ULL
#define BYTES_7F 0x7F7F7F7F7F7F7F7FULL
/* the top bit of every byte of v that is c */
__device__ __forceinline__ uint64_t bytes_equal(uint64_t v, char c) {
  const uint64_t x = v ^ (uint64_t)(unsigned char)c * BYTES_01;
  return ~(((x & BYTES_7F) + BYTES_7F) | x | BYTES_7F);
}
/* the bytes [k, k + 8) of a string of eight bytes or more, zeros behind its end; in: the top bit of those inside */
__device__ __forceinline__ uint64_t string_word(const char* p, uint64_t len, uint64_t k, uint64_t* in) {
  const uint64_t at = k + 8 <= len ? k : len - 8; /* never a byte outside the string */
  uint64_t v;
  __builtin_memcpy(&v, p + at, 8);
  const uint32_t past = (uint32_t)(k - at) * 8u;
  *in = (~BYTES_7F) >> past;
  return v >> past;
}

/* ---- stage 0, one string: both views, by one wavefront ---- */
__device__ __forceinline__ void dict_string(const char* blob, const uint64_t* off, uint32_t id, DictEntry* entries, char* name_blob, char* arg_blob) {
  const uint64_t start = off[id], len = off[id + 1] - start;
  const char* p = blob + start;
  uint32_t nl = 0, q = 0, bad = 0, nonblank = 0;
  const bool wide = len >= 8;
  if (wide) {
    for (uint64_t k = 8ull * lane_id(); k < len; k += 512) {
      uint64_t in; /* the top bit of every byte that is the string's */
      const uint64_t v = string_word(p, len, k, &in);
      const uint64_t nls = bytes_equal(v, '\n') & in, lo = v & BYTES_7F;
      nl += (uint32_t)__popcll(nls);
      q += (uint32_t)__popcll(bytes_equal(v, '"') & in);
      bad += (uint32_t)__popcll((v | (lo + BYTES_01) | ~(lo + 0x60u * BYTES_01)) & in & ~nls); /* > 0x7e or < 0x20 */
      nonblank += (uint32_t)__popcll(~(bytes_equal(v, ' ') | bytes_equal(v, '\t') | bytes_equal(v, '\v') | bytes_equal(v, '\f') |
                                       bytes_equal(v, '\r')) & in & ~nls);
    }
  } else
  for (uint64_t k = lane_id(); k < len; k += 64) {
    const unsigned char c = (unsigned char)p[k];
    if (c == '\n') { ++nl; continue; }
    if (c == '"') ++q;
    if (c < 0x20 || c > 0x7e) ++bad;
    if (!(c == ' ' || c == '\t' || c == '\v' || c == '\f' || c == '\r')) ++nonblank;
  }
  nl = wave_sum_u32(nl); q = wave_sum_u32(q); bad = wave_sum_u32(bad); nonblank = wave_sum_u32(nonblank);
  const bool is_kernel = len == 6 && p[0] == 'k' && p[1] == 'e' && p[2] == 'r' && p[3] == 'n' && p[4] == 'e' && p[5] == 'l';
  DictEntry d;
  d.flags = is_kernel ? KTJ_SF_NAME_KERNEL : bad ? KTJ_SF_NAME_UNKNOWN : 0u;
  d.name_len = is_kernel ? 6u : bad ? 7u : (uint32_t)len - nl + q;
  d.arg_len = (uint32_t)len - nl;
  /* behind the room of the strings before it, whatever their views' lengths are */
  d.name_off = (2 * start + KTJ_DICT_ROOM * (uint64_t)id) & ~15ULL;
  d.arg_off = (start + KTJ_DICT_ROOM * (uint64_t)id) & ~15ULL;
  d.pad = 0;
  if (nonblank == 0) d.flags |= KTJ_SF_ARG_BLANK;
  if (len == 11) {
    const char* want = "Stream Sync";
    bool same = true;
    for (int k = 0; k < 11; ++k) same = same && p[k] == want[k];
    if (same) d.flags |= KTJ_SF_STREAM_SYNC;
  }
  if (lane_id() == 0) entries[id] = d;
  char* an = arg_blob + d.arg_off;
  char* nn = name_blob + d.name_off;
  /* zeros up to the next 16-byte boundary: a view is read in whole blocks */
  auto pad = [&](char* view, uint32_t n) { if (lane_id() < 16u && lane_id() >= (n & 15u) && (n & 15u)) view[(n & ~15u) + lane_id()] = 0; };
  pad(an, d.arg_len);
  pad(nn, d.name_len);
  const bool literal_name = (d.flags & (KTJ_SF_NAME_KERNEL | KTJ_SF_NAME_UNKNOWN)) != 0;
  if (literal_name) {
    const char* lit = is_kernel ? "Kernel" : "unknown";
    if (lane_id() < d.name_len) nn[lane_id()] = lit[lane_id()];
  }
  if (wide && nl == 0 && q == 0) { /* nothing goes and nothing comes: both views are the string but for its backslashes */
    for (uint64_t k = 8ull * lane_id(); k < len; k += 512) {
      uint64_t in;
      uint64_t v = string_word(p, len, k, &in);
      const uint64_t slash = (bytes_equal(v, '\\') >> 7) * 0xFFu;
      v = (v & ~slash) | (slash & (uint64_t)'/' * BYTES_01);
      /* (the last word may reach up to seven bytes past the view, into its room) */
      *reinterpret_cast<uint64_t*>(an + k) = v;
      if (!literal_name) *reinterpret_cast<uint64_t*>(nn + k) = v;
    }
    return;
  }
  uint64_t aw = 0, nw = 0; /* bytes written so far (wave-uniform) */
  const uint64_t lt = lanemask_lt();
  for (uint64_t base = 0; base < len; base += 64) {
    const uint64_t k = base + lane_id();
    const bool in = k < len;
    unsigned char c = in ? (unsigned char)p[k] : 0;
    const bool keep = in && c != '\n';
    if (c == '\\') c = '/';
    const bool isq = keep && c == '"';
    const uint64_t km = __ballot(keep ? 1 : 0);
    const uint64_t qm = __ballot(isq ? 1 : 0);
    const uint32_t kpos = (uint32_t)__popcll(km & lt);
    if (keep) {
      an[aw + kpos] = (char)c;
      if (!literal_name) {
        const uint64_t np = nw + kpos + (uint32_t)__popcll(qm & lt);
        if (isq) { nn[np] = '\\'; nn[np + 1] = '"'; }
        else nn[np] = (char)c;
      }
    }
    aw += (uint32_t)__popcll(km);
    nw += (uint32_t)__popcll(km) + (uint32_t)__popcll(qm);
  }
}

/* ---- stage 1, one row: what the decode kernels put into the columns ---- */
struct RowCols { int64_t ts, dur, dev, res; uint64_t corr; uint32_t meta; };
__device__ __forceinline__ RowCols cols_generic(const ktj_generic_rec& g, const EmitCtx& ctx) {
  RowCols r;
  r.ts = g.start_ns;
  r.dur = g.end_ns - g.start_ns;                  /* GenericTraceActivity.h:65-67 */
  r.corr = (uint64_t)(int64_t)g.id;
  r.dev = generic_device(g, ctx.args, ctx.n_args);
  r.res = g.resource;
  r.meta = (generic_record_prints(g, ctx) ? KTJ_M_VALID : 0u) | (KTJ_CLASS_GENERIC << KTJ_M_CLASS_SHIFT);
  return r;
}
/* runtime and device rows: the clock is converted and the capture window applied (stage 2a:
 * RocprofActivityApi.cpp:166-175, ApproximateClock.cpp:83-90, RocprofActivity.h:42-47 and 122-127,
 * GenericActivityProfiler.cpp:329-340), so that timestamp and duration are written once */
__device__ __forceinline__ RowCols cols_runtime(const ktj_runtime_rec& rec, const ClockDev& clk, int64_t win_start, int64_t win_end) {
  RowCols r;
  uint64_t b = rec.begin, e = rec.end;
  convert_range(clk, clk.runtime_mode, &b, &e);
  r.ts = (int64_t)b;
  r.dur = (int64_t)(e - b);                       /* RocprofActivity.h:42-47 */
  r.corr = rec.id;
  r.dev = (int64_t)rec.pid;
  r.res = (int64_t)rec.tid;
  const uint32_t kind = rec.kind <= KTJ_RT_MALLOC ? rec.kind : KTJ_RT_DEFAULT;
  const uint64_t stream = kind == KTJ_RT_KERNEL ? rec.u.kernel.stream : (kind == KTJ_RT_COPY ? rec.u.copy.stream : 0);
  r.meta = (KTJ_CLASS_RUNTIME << KTJ_M_CLASS_SHIFT) | (kind << KTJ_M_KIND_SHIFT) | (stream != 0 ? KTJ_M_HAS_STREAM : 0u) |
           (out_of_range(r.ts, r.dur, win_start, win_end) ? 0u : KTJ_M_VALID);
  return r;
}
__device__ __forceinline__ RowCols cols_device(const ktj_device_rec& d, const ClockDev& clk, int64_t win_start, int64_t win_end) {
  RowCols r;
  const uint32_t dom = device_row_domain(d.domain);
  uint64_t b = d.begin, e = d.end;
  convert_range(clk, clk.device_mode, &b, &e);
  device_times(dom, b, e, &r.ts, &r.dur);
  r.corr = d.id;
  r.dev = (int64_t)d.device;
  r.res = device_row_stream(dom, d.stream);
  r.meta = (KTJ_CLASS_DEVICE << KTJ_M_CLASS_SHIFT) | (dom << KTJ_M_KIND_SHIFT) |
           (out_of_range(r.ts, r.dur, win_start, win_end) ? 0u : KTJ_M_VALID);
  return r;
}
__device__ __forceinline__ void store_cols(const Columns& c, uint64_t a, const RowCols& r) {
  c.ts[a] = r.ts; c.dur[a] = r.dur; c.corr[a] = r.corr; c.dev[a] = r.dev; c.res[a] = r.res; c.meta[a] = r.meta; c.ext[a] = 0;
}
/* what the launches behind read; linked: device rows, which are joined without their records */
__device__ __forceinline__ void store_cols(const Columns& c, uint64_t a, const RowCols& r, bool linked) {
  c.ts[a] = r.ts; c.dev[a] = r.dev; c.res[a] = r.res; c.meta[a] = r.meta;
  if (linked || c.all) c.corr[a] = r.corr;
  if (c.all) { c.dur[a] = r.dur; c.ext[a] = 0; }
}

__device__ __forceinline__ uint32_t row_domain(uint32_t meta) { return (meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT; }
__device__ __forceinline__ bool is_async_op(uint32_t domain) { return domain != KTJ_DOM_MEMSET; }

__device__ __forceinline__ bool dense_key(uint32_t domain, uint64_t stream, uint64_t queue, uint64_t* key) {
  if (!is_async_op(domain)) return false;
  if (stream != 0) *key = stream;
  else if (queue != 0) *key = queue | (1ULL << 63);
  else return false;
  return true;
}

/* exact byte length in the low 30 bits, tail kind (see tail_kind) in the top two */
__device__ __forceinline__ uint32_t row_length(const MatRow& m, const EmitCtx& ctx, Scalars* sc) {
  if (!(m.meta & KTJ_M_VALID)) return 0;
  CountWriter cw;
  format_activity(cw, m, ctx);
  if (cw.n >= (1ull << 30)) { flag_error(sc, KTJ_DEVERR_RECORD_TOO_LONG); return 0; }
  return (uint32_t)cw.n | (tail_kind(m, has_args(m, ctx)) << 30);
}

/* the tail kind of the activity at a place of the emission order */
__device__ __forceinline__ uint32_t tail_kind_at(const uint8_t* kind_sorted, const weave::TextRow* rows, const uint32_t* perm, uint64_t i, const EmitCtx& ctx) {
  const uint32_t k = kind_sorted[i];
  if (k != KTJ_KIND_LEFT) return k;
  const MatRow m = *reinterpret_cast<const MatRow*>(&rows[perm[i]]);
  return tail_kind(m, has_args(m, ctx));
}

/* ---- bytes to any address of the document ---- */
typedef uint64_t u64_any __attribute__((aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));
typedef uint16_t u16_any __attribute__((aligned(1)));
typedef __attribute__((address_space(1))) char* doc_ptr; /* global memory: no flat accesses */
typedef const __attribute__((address_space(1))) char* text_ptr;
__device__ __forceinline__ void put8(doc_ptr p, uint64_t v) { *reinterpret_cast<__attribute__((address_space(1))) u64_any*>(p) = v; }
__device__ __forceinline__ uint64_t get8(text_ptr p) { return *reinterpret_cast<const __attribute__((address_space(1))) u64_any*>(p); }
/* the n (0..7) low bytes of v */
__device__ __forceinline__ void put_low(doc_ptr p, uint64_t v, uint32_t n) {
  if (n & 4u) { *reinterpret_cast<__attribute__((address_space(1))) u32_any*>(p) = (uint32_t)v; p += 4; v >>= 32; }
  if (n & 2u) { *reinterpret_cast<__attribute__((address_space(1))) u16_any*>(p) = (uint16_t)v; p += 2; v >>= 16; }
  if (n & 1u) *p = (char)v;
}

/* n bytes of header or footer text, by the whole workgroup */
__device__ __forceinline__ void put_text_block(const char* src, char* dst, uint64_t n) { /* src 16-byte aligned */
  const doc_ptr d = reinterpret_cast<doc_ptr>((uintptr_t)dst);
  const uint4* s = reinterpret_cast<const uint4*>(src);
  for (uint64_t k = threadIdx.x; k < (n + 15u) / 16u; k += blockDim.x) {
    const uint4 v = s[k];
    const uint64_t lo = v.x | ((uint64_t)v.y << 32), hi = v.z | ((uint64_t)v.w << 32);
    const uint64_t left = n - k * 16u;
    if (left >= 16u) { put8(d + k * 16u, lo); put8(d + k * 16u + 8u, hi); }
    else if (left >= 8u) { put8(d + k * 16u, lo); put_low(d + k * 16u + 8u, hi, (uint32_t)left - 8u); }
    else put_low(d + k * 16u, lo, (uint32_t)left);
  }
}


}  // namespace gpu
}  // namespace ktj
#endif
