/*
 * weave.hip — stage 4b: the activities' text into the document, one lane per segment (weave_core.h).
 *
 * A lane per activity (k_emit_direct) walks its text piece by piece: 4420 vector instructions for 64 activities with
 * the lanes of a wavefront at different pieces, 168 registers for three wavefronts per SIMD, and no pass shorter than 38 us
 * as every wavefront runs through all of the formatter's code.  Here the text of 16 activities is laid out by the four
 * lanes that load each row, as a list of parts; then 64 segments at a time are fetched (a descriptor, up to 64 bytes of
 * text from LDS, a number of the row's), a prefix sum of their lengths gives their places, and they are written into a
 * piece of the document in LDS (put_segment), whose whole lines leave with lane-consecutive stores.  Numbers were made
 * into text in the size pass, which needs their lengths anyway; the texts with process and thread are made once per
 * track.
 *
 * What bounds it: latency, the LDS pipe and the vector units before memory (22 million records 2.97 ms when it came to five wavefronts
 * per SIMD, 2.83 now, 13.4 GB, of which 2.6 ms are what a copy of two parts read and seven written takes; without its stores the kernel takes some 2.5, without words written
 * to LDS either 2.0), so it is the wavefronts in flight that count: five per SIMD, which five workgroups of
 * four make (of five or of ten wavefronts three and one fit into a CU: 4.2 and 4.5 ms).  That takes 96 registers and
 * 32000 bytes of LDS per workgroup: texts that begin alike are there once, and names and the piece of the document share their room
 * (2944 bytes of document and 1280 of names would not fit; 2304 and 768 are short of most groups of 64 segments: 11 million
 * kernels 1.88 ms).  Four -> five wavefronts: 733 000 records 136 -> 121 us, 3 million 443 -> 402, 22 million 3.30 -> 2.97 ms,
 * 5 million operators with long strings 2.64 -> 2.45, 11 million kernels, at the memory's rate, 1.65 -> 1.62; three: 2.48, two 2.83.
 *
 * Measured against k_emit_direct (lane per activity): 10 000 x 3 records 38.7 -> 15 us, 4000 operators with long strings
 * 71 -> 23 us, 733 000 records 176 -> 105 us, 3 million 795 -> 367 us, 11 million kernels 2.06 -> 1.52 ms, 22 million
 * records 4.59 -> 2.83 ms, 5 million operators with long strings (1.4 KB each: strings beyond 128 bytes are fetched from
 * memory piece by piece) 3.20 -> 2.44 ms; the size pass has become up to 18 % longer for the numbers' text.
 * (Long strings' whole lines from the dictionary to the document past the tile, the loads of four strings at a time in
 * front of any store: no gain.  Strings waited for in front of the last lines' stores, with these lines read from LDS a second time: passes 0.6 to
 * 1.5 % longer.)
 */
#include "gpu_common.h"
#include "weave_core.h"

namespace ktj {
namespace gpu {

using namespace weave;

#define WV_ROWS 16u                                   /* activities at a time, four lanes to each */
#define WV_WAVES 4u                                   /* wavefronts per workgroup, at most */
#define WV_PARTS (WV_ROWS * 7u)
#define WV_VAL_BYTES (S_RUN * 16u)                    /* S_A and the following; an odd number of sixteens: the same slot of neighbours lies in other banks */
#define WV_VAL(slot) (((slot) - 1u) * 16u)
#define WV_NAMES 1280u                                /* bytes of strings that wait in LDS, at most */
#define WV_NAME_MOST 128u
/* of a wavefront: */
#define WV_TRACK_AT (WV_ROWS * WV_VAL_BYTES)
#define WV_PARTS_AT (WV_TRACK_AT + T_COUNT * KTJ_WEAVE_LIT)
#define WV_TILE_AT (WV_PARTS_AT + WV_PARTS * 4u + 32u)
/* the bytes of the document that wait in LDS, from the front on, and the strings, from the end on: between them what texts write beyond
 * their end, behind the former at least a line */
#define WV_SPACE 3600u
#define WV_GAP 32u
#define WV_TILE_MOST 3072u                            /* whole lines leave in three turns at most */
#define WV_WAVE_BYTES (WV_TILE_AT + WV_SPACE)
/* of the workgroup, in front of them: the texts, the book's and the schemas'; where the parts are: the book's, those of the schemas' args and
 * an empty one, those of their args2 and an empty one; descriptors */
#define WV_BOOK_REF ((LDS_BOOK.n_text + SCHEMA_TEXT) * 16u)
#define WV_REF_SCHEMA R_COUNT
#define WV_REF_SCHEMA2 (WV_REF_SCHEMA + MAX_SCHEMAS + 1u)
#define WV_REF_EMPTY (WV_REF_SCHEMA + MAX_SCHEMAS)
#define WV_REFS (WV_REF_SCHEMA2 + MAX_SCHEMAS + 1u)
#define WV_BOOK_DESC (WV_BOOK_REF + (WV_REFS + 1u) / 2u * 4u)
#define WV_BOOK_BYTES ((WV_BOOK_DESC + (MAX_DESC + SCHEMA_DESC) * 4u + 15u) / 16u * 16u)

/* a part: first segment | kind << 15 (text, or one of the strings of S_RUN) | first descriptor << 17 | activity << 26 */
#define WV_PART_START(x) ((x) & 0x7FFFu)
#define WV_PART_KIND(x) (((x) >> 15) & 3u)
#define WV_PART_DESC(x) (((x) >> 17) & 0x1FFu)
#define WV_PART_ACT(x) ((x) >> 26)

/* The book as it lies in LDS.  A text's first 32 bytes and the others are at places of their own (in 27 heads of events the former are
 * the same), a part is named by sixteen bits. */
#define WV_WD_LEN(x) ((x) & 0x7Fu)
#define WV_WD_TRACK (1u << 7)
#define WV_WD_SLOT(x) (((x) >> 8) & 0xFu)
#define WV_WD_UNIT(x) (((x) >> 12) & 0x1FFu)
#define WV_WD_UNIT2(x) (((x) >> 21) & 0x1FFu)       /* (bits 30 and 31: WV_FAR) */
#define WV_WD(len, slot, unit, unit2) ((len) | ((slot) << 8) | ((unit) << 12) | ((unit2) << 21))
#define WV_REF(base, count) ((base) | ((count) << 9))
#define WV_REF_BASE(r) ((r) & 0x1FFu)
#define WV_REF_COUNT(r) ((r) >> 9)
struct LdsBook {
  uint32_t text[MAX_TEXT * 4], desc[MAX_DESC], n_text;
  uint16_t ref[R_COUNT];
};
constexpr LdsBook make_lds_book() {
  LdsBook l{};
  auto place = [&](const uint32_t* w, uint32_t units) { /* the same bytes somewhere already? */
    uint32_t at = 0;
    for (; at + units <= l.n_text; ++at) {
      bool same = true;
      for (uint32_t i = 0; i < units * 4; ++i) same = same && l.text[at * 4 + i] == w[i];
      if (same) break;
    }
    if (at + units > l.n_text) {
      at = l.n_text;
      for (uint32_t i = 0; i < units * 4; ++i) l.text[at * 4 + i] = w[i];
      l.n_text += units;
    }
    return at;
  };
  for (uint32_t k = 0; k < BOOK.n_desc; ++k) {
    const uint32_t d = BOOK.desc[k], len = KTJ_WD_LEN(d), unit = KTJ_WD_UNIT(d), units = (len + 15) / 16;
    if (d & KTJ_WD_TRACK) l.desc[k] = WV_WD(len, KTJ_WD_SLOT(d), unit, unit + 2) | WV_WD_TRACK;
    else l.desc[k] = WV_WD(len, KTJ_WD_SLOT(d), place(BOOK.text + unit * 4, units < 2 ? units : 2), units > 2 ? place(BOOK.text + (unit + 2) * 4, units - 2) : 0);
  }
  for (uint32_t r = 0; r < R_COUNT; ++r) l.ref[r] = (uint16_t)WV_REF(KTJ_WREF_BASE(BOOK.ref[r]), KTJ_WREF_COUNT(BOOK.ref[r]));
  return l;
}
constexpr LdsBook LDS_BOOK = make_lds_book();
static_assert(MAX_DESC + SCHEMA_DESC <= 512u && SCHEMA_DESC < 128u && LDS_BOOK.n_text + SCHEMA_TEXT + 2u <= 512u, "nine bits each, seven for a count");
static __device__ constexpr LdsBook g_book = LDS_BOOK;

__device__ __forceinline__ uint32_t dpp_add(uint32_t v) { /* inclusive sum over the wavefront */
#define WV_DPP(ctrl, rows) v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xF, false)
  WV_DPP(0x111, 0xF); WV_DPP(0x112, 0xF); WV_DPP(0x114, 0xF); WV_DPP(0x118, 0xF);
  WV_DPP(0x142, 0xA); WV_DPP(0x143, 0xC);
#undef WV_DPP
  return v;
}
/* inclusive sum over the activities, four lanes to each that have the same */
__device__ __forceinline__ uint32_t quad_add(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);
  return v;
}
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ void or_word(char* p, uint32_t v) {
  __hip_atomic_fetch_or(reinterpret_cast<uint32_t*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
typedef unsigned long long v2u64 __attribute__((ext_vector_type(2)));
typedef uint32_t v4u32 __attribute__((ext_vector_type(4)));

#define WV_WORD(hi, lo) __builtin_amdgcn_alignbyte(hi, lo, sh)
/* a segment of up to 32 bytes of text (zeros behind its text and its number) to byte p of a zero-filled buffer */
__device__ __forceinline__ void or_segment(char* buf, uint32_t p, uint32_t len, const v4u32& a, const v4u32& b, uint32_t n_num, const v4u32& num) {
  {
    const uint32_t sh = 0u - p;                                   /* bits 0 and 1 count */
    char* q = buf + (int32_t)(((int32_t)p - 1) & ~3);             /* the word of the byte before */
    or_word(q, WV_WORD(a.x, 0u)); or_word(q + 4, WV_WORD(a.y, a.x)); or_word(q + 8, WV_WORD(a.z, a.y)); or_word(q + 12, WV_WORD(a.w, a.z));
    or_word(q + 16, WV_WORD(b.x, a.w)); or_word(q + 20, WV_WORD(b.y, b.x)); or_word(q + 24, WV_WORD(b.z, b.y)); or_word(q + 28, WV_WORD(b.w, b.z));
    or_word(q + 32, WV_WORD(0u, b.w));
  }
  if (n_num) {
    const uint32_t p2 = p + len, sh = 0u - p2;
    char* q = buf + (int32_t)(((int32_t)p2 - 1) & ~3);
    or_word(q, WV_WORD(num.x, 0u)); or_word(q + 4, WV_WORD(num.y, num.x)); or_word(q + 8, WV_WORD(num.z, num.y));
    or_word(q + 12, WV_WORD(num.w, num.z)); or_word(q + 16, WV_WORD(0u, num.w));
  }
}
typedef volatile __attribute__((address_space(3))) uint32_t* lds_word; /* (volatile: these accesses stay in their order) */
__device__ __forceinline__ void put_word(char* p, uint32_t v) { *(lds_word)p = v; }
__device__ __forceinline__ void or_shared_word(char* p, uint32_t v) { __hip_atomic_fetch_or((lds_word)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT); }
/* Segments one behind the other, a lane's behind that of the lane before it, to byte p and the following of a buffer that holds
 * anything.  A word belongs to the segment that has its first byte, is written whole and OR-ed by whoever has the others.  A text's words are
 * written up to the end of its sixteen bytes, whatever it has of them: the words too many are zeros in words of lanes behind, and these lanes
 * write there later, as the last word of a text goes first, everybody's, and a word of a lane behind is an earlier one of its text.  Then come
 * the numbers, which write their own words only, then the words that are shared.  A wavefront's LDS accesses are carried out in
 * their order.  (All of them OR-ed to a buffer of zeros, whole lines cleared when they left: a 64-lane store of 16 bytes each takes
 * the LDS pipe 14 cycles, three of them of the 290 that 64 segments take.  22 million records 3.42 -> 3.30 ms, 11 million kernels
 * 1.68 -> 1.65, 733 000 records 141 -> 136 us.) */
__device__ __forceinline__ void put_segment(char* buf, uint32_t p, uint32_t len, const v4u32& a, const v4u32& b, const v4u32& c, const v4u32& d,
                                            uint32_t n_num, const v4u32& num) {
  char* const q = buf + (int32_t)(((int32_t)p - 1) & ~3);       /* the word of the byte before: shared, if anything of the text is in it */
  const uint32_t sh = 0u - p;                                   /* bits 0 and 1 count */
  if (len + n_num + ((p - 1u) & 3u) > 3u) {                     /* (all in the first word: the lane behind has the same words) */
    if (len > 16u) {
      if (len > 32u) {
        if (len > 48u) { put_word(q + 64, WV_WORD(0u, d.w)); put_word(q + 60, WV_WORD(d.w, d.z)); put_word(q + 56, WV_WORD(d.z, d.y)); put_word(q + 52, WV_WORD(d.y, d.x)); }
        put_word(q + 48, WV_WORD(len > 48u ? d.x : 0u, c.w)); put_word(q + 44, WV_WORD(c.w, c.z)); put_word(q + 40, WV_WORD(c.z, c.y)); put_word(q + 36, WV_WORD(c.y, c.x));
      }
      put_word(q + 32, WV_WORD(len > 32u ? c.x : 0u, b.w)); put_word(q + 28, WV_WORD(b.w, b.z)); put_word(q + 24, WV_WORD(b.z, b.y)); put_word(q + 20, WV_WORD(b.y, b.x));
    }
    put_word(q + 16, WV_WORD(len > 16u ? b.x : 0u, a.w)); put_word(q + 12, WV_WORD(a.w, a.z)); put_word(q + 8, WV_WORD(a.z, a.y)); put_word(q + 4, WV_WORD(a.y, a.x));
  }
  if (n_num) {
    const uint32_t p2 = p + len, sh = 0u - p2, upto = n_num + ((p2 - 1u) & 3u) + 1u; /* bytes from q2 on */
    char* const q2 = buf + (int32_t)(((int32_t)p2 - 1) & ~3);
    if (upto > 4u) {
      put_word(q2 + 4, WV_WORD(num.y, num.x));
      if (upto > 8u) {
        put_word(q2 + 8, WV_WORD(num.z, num.y));
        if (upto > 12u) {
          put_word(q2 + 12, WV_WORD(num.w, num.z));
          if (upto > 16u) put_word(q2 + 16, WV_WORD(0u, num.w));
        }
      }
    }
    or_shared_word(q2, WV_WORD(num.x, 0u));
  }
  or_shared_word(q, WV_WORD(a.x, 0u));
}
/* (of a fixed size, also where a workgroup has fewer wavefronts: its address is then a constant that the compiler folds) */
#define WV_LDS_BYTES (WV_BOOK_BYTES + WV_WAVES * WV_WAVE_BYTES)
/* the track's texts, with the lead of its times; their lengths, a byte each */
__device__ __forceinline__ uint64_t make_track(char* lds, uint32_t mine, uint64_t dev, uint64_t thread, uint32_t lead) {
  const uint32_t lane = lane_id();
  char* const track = lds + mine + WV_TRACK_AT;
  if (lane < T_COUNT * 4u) *reinterpret_cast<uint4*>(track + lane * 16u) = make_uint4(0, 0, 0, 0);
  const Text pid = text_of(dev), tid = text_of(thread);
  Text time = text_of(lead);
  if (lead == 0) { time.lo = 0; time.n = 0; }
  const uint32_t desc = lane < N_PIECES ? *reinterpret_cast<const uint32_t*>(lds + WV_BOOK_DESC + (WV_REF_BASE(LDS_BOOK.ref[R_PIECES]) + lane) * 4u) : 0u;
  const uint32_t len = WV_WD_LEN(desc), slot = WV_WD_SLOT(desc), n_num = slot == S_PID ? pid.n : slot == S_TID ? tid.n : slot == S_LEAD ? time.n : 0u;
  const v4u32 zero = {0, 0, 0, 0};
  v4u32 a = zero, b = zero, num = zero;
  const v4u32* t = reinterpret_cast<const v4u32*>(lds) + WV_WD_UNIT(desc);
  if (len) a = t[0];
  if (len > 16u) b = t[1];
  if (slot == S_PID) { num.x = (uint32_t)pid.lo; num.y = (uint32_t)(pid.lo >> 32); num.z = (uint32_t)pid.hi; num.w = (uint32_t)(pid.hi >> 32); }
  if (slot == S_TID) { num.x = (uint32_t)tid.lo; num.y = (uint32_t)(tid.lo >> 32); num.z = (uint32_t)tid.hi; num.w = (uint32_t)(tid.hi >> 32); }
  if (slot == S_LEAD) num.x = (uint32_t)time.lo, num.y = (uint32_t)(time.lo >> 32);
  const uint32_t end = dpp_add(len + n_num);
  /* pieces 0-2, 3-5, 6-8, 9-10, 11-12 are a text each */
  const uint32_t which = lane < 9u ? lane / 3u : lane < 11u ? 3u : 4u;
  const uint32_t e2 = __builtin_amdgcn_readlane(end, 2), e5 = __builtin_amdgcn_readlane(end, 5), e8 = __builtin_amdgcn_readlane(end, 8),
                 e10 = __builtin_amdgcn_readlane(end, 10), e12 = __builtin_amdgcn_readlane(end, 12);
  const uint32_t start = which == 0 ? 0u : which == 1 ? e2 : which == 2 ? e5 : which == 3 ? e8 : e10;
  wave_lds_order();
  if (lane < N_PIECES) or_segment(track, which * KTJ_WEAVE_LIT + (end - len - n_num - start), len, a, b, n_num, num);
  return (uint64_t)(e2 | ((e5 - e2) << 8) | ((e8 - e5) << 16) | ((e10 - e8) << 24)) | ((uint64_t)(e12 - e10) << 32);
}

/* A document that does not stay in the 256 MB last-level cache leaves it and the L2s, when stored in the ordinary way, full of lines that are
 * written back while the next kernels run: whole passes of
 * 733 000 records 485 -> 465 us, of 3 million 1150 -> 1125 (k_decode of the next pass 94 -> 69 us), of 11 million 3590 -> 3560.  A small one
 * is read back from there: sessions of 4000 operators with long strings (6 MB) 470 us with ordinary stores, 508 past the caches, files
 * of 90 000 records (37 MB) 6430 and 6750.  The host knows the activities at this point and not their bytes, so the line is at as many as make 250 MB
 * of 480 bytes each.  On either side of it, passes with ordinary stores and past the caches, us, sessions to the host's memory with both the same within
 * their spread of 3 %: above, 600 000 plain operators (167 MB) 239 and 226, 555 000 records (224 MB) 302 and 291; below, 286 000 records (127 MB) 257 and 256,
 * 440 000 (196 MB) 299 and 293, 504 000 kernels of graphs (229 MB) 318 and 314, operators with strings of a kilobyte 264 and 255 (200 000, 276 MB), 393 and 372
 * (400 000, 552 MB): short activities lose nothing by it, and long ones leave some unused. */
#define WV_PAST_FROM (1u << 19)
/* PAST: the document's whole lines are stored past the caches' replacement */
template <bool PAST>
__global__ void __launch_bounds__(WV_WAVES * 64u) __attribute__((amdgpu_waves_per_eu(5)))
k_weave(const TextRow* rows, const uint32_t* perm, const uint64_t* offs, const uint8_t* kind_sorted, EmitCtx ctx, char* out, uint64_t prefix_len,
        const Scalars* sc, uint32_t rounds, const SchemaBook* schemas, const WideText* wide) {
  __shared__ __attribute__((aligned(16))) char wv_lds[WV_LDS_BYTES];
  if (sc->no_text) return;
  const uint32_t lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (uint32_t k = threadIdx.x; k < LDS_BOOK.n_text + SCHEMA_TEXT; k += blockDim.x)
    reinterpret_cast<uint4*>(wv_lds)[k] = k < LDS_BOOK.n_text ? reinterpret_cast<const uint4*>(g_book.text)[k] : reinterpret_cast<const uint4*>(schemas->text)[k - LDS_BOOK.n_text];
  uint16_t* const refs = reinterpret_cast<uint16_t*>(wv_lds + WV_BOOK_REF);
  for (uint32_t k = threadIdx.x; k < R_COUNT; k += blockDim.x) refs[k] = g_book.ref[k];
  if (threadIdx.x <= MAX_SCHEMAS) {
    const SchemaPlan* const p = schemas->plan + threadIdx.x;
    const uint32_t a = threadIdx.x < MAX_SCHEMAS ? p->args : 0u, b = threadIdx.x < MAX_SCHEMAS ? p->args2 : 0u;
    refs[WV_REF_SCHEMA + threadIdx.x] = (uint16_t)WV_REF(KTJ_WREF_BASE(a), KTJ_WREF_COUNT(a));
    refs[WV_REF_SCHEMA2 + threadIdx.x] = (uint16_t)WV_REF(KTJ_WREF_BASE(b), KTJ_WREF_COUNT(b));
  }
  for (uint32_t k = threadIdx.x; k < MAX_DESC + SCHEMA_DESC; k += blockDim.x) {
    uint32_t d;
    if (k < MAX_DESC) d = g_book.desc[k];
    else {
      const uint32_t x = schemas->desc[k - MAX_DESC], unit = (KTJ_WD_UNIT(x) - SCHEMA_UNIT + LDS_BOOK.n_text) & 0x1FFu;
      d = WV_WD(KTJ_WD_LEN(x), KTJ_WD_SLOT(x), unit, (unit + 2u) & 0x1FFu);
    }
    reinterpret_cast<uint32_t*>(wv_lds + WV_BOOK_DESC)[k] = d;
  }
  const uint32_t mine = WV_BOOK_BYTES + wave * WV_WAVE_BYTES; /* this wavefront's LDS */
  uint32_t* const parts = reinterpret_cast<uint32_t*>(wv_lds + mine + WV_PARTS_AT);
  char* const tile = wv_lds + mine + WV_TILE_AT;
  __syncthreads();
  const uint64_t n_rows = sc->emit_rows;
  typedef __attribute__((address_space(1))) v2u64* gptr;
  typedef const __attribute__((address_space(1))) v4u32* gsrc;

  const uint32_t h = lane & 3u, act = lane >> 2;
  /* which of an activity's parts the lane names, and where the plan says which they are: head, name, body and args, then the string between
   * them, args2 and tail */
  const uint32_t shift_a = h == 0u ? 0u : h == 1u ? 5u : h == 2u ? 12u : 14u, width_a = h == 0u ? 5u : h == 2u ? 2u : 7u;
  const uint32_t base_a = h == 0u ? (uint32_t)R_HEAD : h == 1u ? 0u : h == 2u ? (uint32_t)R_BODY_NONE : (uint32_t)R_ARGS;
  const uint32_t shift_b = h == 1u ? 14u : 21u, width_b = h == 1u ? 7u : h == 2u ? 4u : 0u;
  const uint32_t base_b = h == 1u ? (uint32_t)R_ARGS2 : h == 2u ? (uint32_t)R_TAIL : (uint32_t)WV_REF_EMPTY;
  v2u64* const vals = reinterpret_cast<v2u64*>(wv_lds + mine + act * WV_VAL_BYTES);
  uint64_t track_made = ~0ull; /* what the track's texts are made of */
  uint32_t track_made_high = ~0u;
  uint64_t track_lens = 0;
  const uint64_t i_begin = ((uint64_t)blockIdx.x * (blockDim.x >> 6) + wave) * rounds * WV_ROWS;
  if (i_begin >= n_rows) return;
  const uint64_t i_end = i_begin + rounds * WV_ROWS < n_rows ? i_begin + rounds * WV_ROWS : n_rows;
  /* A row's four lanes load it together, two blocks each.  The rows of the next turn are on their way while this one's are
   * put together. */
  v4u32 q0, q1;
  auto load_row = [&](uint32_t row) {
    const gsrc r = reinterpret_cast<gsrc>((uint64_t)(uintptr_t)rows + (uint64_t)row * sizeof(TextRow));
    q0 = r[h];                           /* S_Z, S_EXT, S_FLOW, S_DUR and plan, name, lens, more */
    q1 = r[4u + h];                      /* S_A and the track, S_TS, S_X, S_Y */
  };
  auto row_at = [&](uint64_t i) { return perm[i < i_end ? i : i_end - 1]; }; /* (with a condition on the load the next turn's rows were waited for as
   * soon as they were asked for, where a register that the other way leaves as it is meets the one that is loaded: 22 million records 2.99 ms,
   * then 2.85, 11 million kernels 1.62 and 1.52) */
  uint32_t row = row_at(i_begin + act);
  load_row(row);
  row = row_at(i_begin + WV_ROWS + act);

  uint32_t part = 0, pend = 0, own = 0;
  char* doc = nullptr;
  bool open = false;
  /* the document's bytes end here for this wavefront: the block shared with what follows */
  auto close_document = [&](uint64_t i_next) {
    open = false;
    const uint32_t fill = pend & 15u, at = pend & ~15u;
    if (lane == 0 && fill) {
      uint64_t* t = reinterpret_cast<uint64_t*>(tile + at);
      uint64_t* w = reinterpret_cast<uint64_t*>(doc + at);
      if (i_next == n_rows) {
        if (fill < 8) { const uint64_t k = (1ull << (8 * fill)) - 1ull; t[0] = (t[0] & k) | (w[0] & ~k); t[1] = w[1]; }
        else { const uint64_t k = (1ull << (8 * (fill - 8))) - 1ull; t[1] = (t[1] & k) | (w[1] & ~k); }
      } else if (fill >= 8) { /* the successor's first bytes complete it */
        const uint32_t s = 8 * (fill - 8);
        t[1] = (t[1] & ((1ull << s) - 1ull)) | (BlockWriter::head_bytes() << s);
      }
    }
    wave_lds_order();
    const uint32_t blocks = (pend >> 4) + (fill >= 8 || (fill && i_next == n_rows) ? 1u : 0u);
    if (lane <= 8u) {
      const v2u64 x = reinterpret_cast<v2u64*>(tile)[lane];
      if (lane >= own && lane < blocks) reinterpret_cast<gptr>((uintptr_t)doc)[lane] = x;
    }
    wave_lds_order();
  };

  for (uint64_t i0 = i_begin; i0 < i_end; i0 += WV_ROWS) {
    const bool active = i0 + act < i_end;
    /* rows that format_activity prints are another kernel's */
    const uint64_t left_of = __builtin_amdgcn_ballot_w64(!active || (h == 3u && (q1.w >> 24) == KTJ_ROW_LEFT));
    const uint64_t ok_mask = ~(left_of | (left_of >> 3)) & 0x1111111111111111ull; /* a bit at the first lane of each of the others */
    const bool mine_ok = (ok_mask >> (lane & ~3u)) & 1u;
#define WV_QUAD(x, k) ((uint32_t)__builtin_amdgcn_mov_dpp((int)(x), (k) * 0x55, 0xF, 0xF, true)) /* the k-th lane's, for all four */
    const uint32_t plan = WV_QUAD(q0.w, KTJ_TR_PLAN), name_off = WV_QUAD(q0.w, KTJ_TR_NAME), lens = WV_QUAD(q0.w, KTJ_TR_LENS), more = WV_QUAD(q0.w, KTJ_TR_MORE);
    const uint32_t track_low = WV_QUAD(q1.z, 0), track_mid = WV_QUAD(q1.w, 0);
    /* the times' lead and the thread's upper bits */
    uint32_t track_high = KTJ_TR_TID_HIGH(plan);
    if (__builtin_amdgcn_ballot_w64((lens & KTJ_TR_HAS_LEAD) != 0)) {
      uint32_t lead = KTJ_TR_LEAD_NIBBLE(q0.z) << (4u * h);
      lead |= (uint32_t)__builtin_amdgcn_mov_dpp((int)lead, 0xB1, 0xF, 0xF, true); /* the quad's: its lanes 1 0 3 2, then 2 3 0 1 */
      lead |= (uint32_t)__builtin_amdgcn_mov_dpp((int)lead, 0x4E, 0xF, 0xF, true);
      if (lens & KTJ_TR_HAS_LEAD) track_high |= lead << 5;
    }
    /* activities whose track or lead is not that of the one before: a bit at the first lane of each */
    uint64_t new_track;
    {
      /* the lane four before: the last of the row before for the first lanes of a row of sixteen, the wavefront's last activity's for the first of all */
#define WV_BEFORE(x, first) ((uint32_t)__builtin_amdgcn_update_dpp(__builtin_amdgcn_update_dpp((int)(first), (int)(x), 0x142, 0xE, 0xF, false), (int)(x), 0x114, 0xF, 0xF, false))
      const uint32_t low = WV_BEFORE(track_low, (uint32_t)track_made), mid = WV_BEFORE(track_mid, (uint32_t)(track_made >> 32)), high = WV_BEFORE(track_high, track_made_high);
#undef WV_BEFORE
      new_track = __builtin_amdgcn_ballot_w64(((track_low ^ low) | (track_mid ^ mid) | (track_high ^ high)) != 0u) & 0x1111111111111111ull;
    }
    const v4u32 z = {q0.x, q0.y, q0.z & 0xFFFFFFu, q0.z & 0xF000000u};
    vals[S_Z - 1u + h] = __builtin_bit_cast(v2u64, z);
    {
      const uint32_t on = (q1.y >> 24) > KTJ_TR_A_NEAR ? more : 0u; /* (of the first lane) */
      const v4u32 a = {q1.x, (q1.y & 0xFFFFFFu) | (on << 24), on >> 8, q1.y & 0xFF000000u}, x = h == 0u ? a : q1;
      vals[S_A - 1u + h] = __builtin_bit_cast(v2u64, x);
    }
    const uint32_t len0 = lens & 0xFFFFu, len1 = KTJ_TR_LEN1(lens), between = KTJ_TR_BETWEEN(plan);
    /* The parts: four lanes name an activity's, two each.  Sums over its lanes in front (segments and parts of the first four, of the others),
     * then over the activities.  (By one lane of the four, one part after the other, each behind its own access to LDS, and a dozen
     * instructions more per 64 segments: 22 million records 2.86 ms, now 2.82, 11 million kernels 1.53 and 1.49.) */
    uint32_t before, upto;
    {
      uint32_t ref_a = __builtin_amdgcn_ubfe(plan, shift_a, width_a) + base_a, ref_b = __builtin_amdgcn_ubfe(plan, shift_b, width_b) + base_b;
      const uint32_t args = KTJ_TR_ARGS(plan), schema = args - KTJ_TR_SCHEMA < MAX_SCHEMAS ? args - KTJ_TR_SCHEMA : MAX_SCHEMAS;
      if (args >= KTJ_TR_SCHEMA && h == 3u) ref_a = WV_REF_SCHEMA + schema;
      if (args >= KTJ_TR_SCHEMA && h == 1u) ref_b = WV_REF_SCHEMA2 + schema;
      const uint32_t a = refs[ref_a], b = refs[ref_b];
      uint32_t n_a = WV_REF_COUNT(a), n_b = WV_REF_COUNT(b), part_a = (WV_REF_BASE(a) << 17) | (act << 26), part_b = (WV_REF_BASE(b) << 17) | (act << 26);
      if (h == 1u && KTJ_TR_NAMED(plan) == KTJ_TR_NAME_RUN) { n_a = (len0 + KTJ_WEAVE_LIT - 1u) / KTJ_WEAVE_LIT; part_a = (1u << 15) | (act << 26); }
      if (h == 0u) { n_b = (len1 + KTJ_WEAVE_LIT - 1u) / KTJ_WEAVE_LIT; part_b = (2u << 15) | (act << 26); }
      n_a = mine_ok ? n_a : 0u; n_b = mine_ok ? n_b : 0u;
      static_assert((KTJ_WEAVE_MAX_RUN + KTJ_WEAVE_LIT - 1u) / KTJ_WEAVE_LIT + 127u * 2u < 1024u, "ten bits for an activity's segments on either side");
      const uint32_t c = n_a | ((n_a ? 1u : 0u) << 10) | (n_b << 13) | ((n_b ? 1u : 0u) << 23);
      uint32_t in_front = (uint32_t)__builtin_amdgcn_mov_dpp((int)c, 0x90, 0xF, 0xF, true);              /* lanes 0 0 1 2 */
      in_front = h >= 1u ? in_front : 0u;
      const uint32_t two = in_front + (uint32_t)__builtin_amdgcn_mov_dpp((int)in_front, 0x90, 0xF, 0xF, true);
      in_front += (uint32_t)__builtin_amdgcn_mov_dpp((int)two, 0x90, 0xF, 0xF, true);                  /* of the lanes before: none, one, two, three */
      const uint32_t all = WV_QUAD(in_front + c, 3);
      const uint32_t first_segs = all & 0x3FFu, first_parts = (all >> 10) & 7u;
      const uint32_t total = (first_segs + ((all >> 13) & 0x3FFu)) | ((first_parts + (all >> 23)) << 16);
      upto = quad_add(total);
      before = upto - total;
      const uint32_t segs = before & 0xFFFFu, n_parts = before >> 16;
      if (n_a) parts[n_parts + ((in_front >> 10) & 7u)] = part_a | (segs + (in_front & 0x3FFu)); /* (segments stay below their 15 bits) */
      if (n_b) parts[n_parts + first_parts + (in_front >> 23)] = part_b | (segs + first_segs + ((in_front >> 13) & 0x3FFu));
    }
    /* the strings in LDS: wide texts, two units each, and names as far as there is room */
    static_assert(WV_ROWS * sizeof(WideText) <= WV_NAMES && sizeof(WideText) == 32, "the wide texts have room");
    const bool is_wide = mine_ok && between == 3u;
    const uint32_t name_units = mine_ok && len0 <= WV_NAME_MOST ? (len0 + 15u) / 16u : 0u;
    const uint32_t units_upto = quad_add(name_units | (is_wide ? 2u << 16 : 0u));
    const uint32_t wide_units = __builtin_amdgcn_readlane(units_upto, 63) >> 16, name_upto = (units_upto & 0xFFFFu) + wide_units;
    const bool near = name_units != 0 && name_upto <= WV_NAMES / 16u;
    const uint32_t double_at = WV_WAVE_BYTES - (units_upto >> 16) * 16u, name_at = WV_WAVE_BYTES - name_upto * 16u;
    /* what they leave of the space (the last of the names that are there says it) */
    const uint64_t near_ones = __builtin_amdgcn_ballot_w64(near);
    const uint32_t taken = (near_ones ? __builtin_amdgcn_readlane(name_upto, 63u - (uint32_t)__builtin_clzll(near_ones)) : wide_units) * 16u + WV_GAP;
    const uint32_t room = WV_SPACE - taken < WV_TILE_MOST ? WV_SPACE - taken : WV_TILE_MOST;
    v4u32 nx, ny, wx;
    const bool load_wide = is_wide && h < 2u, load_x = near && h < name_units, load_y = near && h + 4u < name_units;
    if (load_wide) wx = reinterpret_cast<gsrc>((uint64_t)(uintptr_t)wide + (uint64_t)more * sizeof(WideText))[h];
    {
      const gsrc src = reinterpret_cast<gsrc>((uint64_t)(uintptr_t)ctx.dict.name_blob + (uint64_t)name_off * 16u);
      if (load_x) { nx = src[h]; if (load_y) ny = src[h + 4u]; }
    }
#undef WV_QUAD
    if (h == 0u && mine_ok) {
      const uint32_t at = between < 2u ? 0u : between == 2u ? act * WV_VAL_BYTES + WV_VAL(S_Y) : double_at;
      v4u32 runs;
      runs.x = more; runs.y = len1 | (at << 16);
      if (KTJ_TR_ARGS(plan) == A_COPY) runs.y = ((32u - (uint32_t)__clz((int)more) + 7u) >> 3) << 24; /* of the kind's characters, up to four */
      runs.z = name_off; runs.w = len0 | ((near ? name_at : 0u) << 16);
      vals[S_RUN - 1u] = __builtin_bit_cast(v2u64, runs);
    }
    const uint32_t n_parts = __builtin_amdgcn_readlane(upto, 63) >> 16;
    if (load_wide) *reinterpret_cast<v4u32*>(wv_lds + mine + double_at + h * 16u) = wx;
    if (load_x) {
      *reinterpret_cast<v4u32*>(wv_lds + mine + name_at + h * 16u) = nx;
      if (load_y) *reinterpret_cast<v4u32*>(wv_lds + mine + name_at + (h + 4u) * 16u) = ny;
    }
    /* the next turn's rows */
    load_row(row);
    row = row_at(i0 + 2u * WV_ROWS + act);

    /* ---- neighbouring activities of a track ---- */
    if (open && !(ok_mask & 1u)) close_document(i0);
    uint64_t todo = ok_mask, track_seen = 0; /* ..: activities whose change of track the texts have followed */
    while (todo) {
      const uint32_t first = (uint32_t)__ffsll((unsigned long long)todo) - 1u; /* lanes: four to an activity */
      const uint64_t later = first >= 60u ? 0ull : ~0ull << (first + 4u);
      const uint64_t gap = ((~todo & 0x1111111111111111ull) | new_track) & later;
      const uint32_t next_lane = gap ? (uint32_t)__ffsll((unsigned long long)gap) - 1u : 64u, last = next_lane - 4u;
      todo &= next_lane == 64u ? 0ull : ~0ull << next_lane;
      uint32_t g = __builtin_amdgcn_readlane(before, first) & 0x7FFFu;
      const uint32_t g_end = __builtin_amdgcn_readlane(upto, last) & 0x7FFFu;
      part = __builtin_amdgcn_readlane(before, first) >> 16;
      const uint64_t upto_first = first >= 60u ? ~0ull : (1ull << (first + 4u)) - 1ull;
      if (new_track & upto_first & ~track_seen) {
        const uint32_t low = __builtin_amdgcn_readlane(track_low, first), high = __builtin_amdgcn_readlane(track_mid, first);
        track_made_high = (uint32_t)__builtin_amdgcn_readlane(track_high, first);
        track_made = (uint64_t)low | ((uint64_t)high << 32);
        track_lens = make_track(wv_lds, mine, low & ((1u << KTJ_TR_DEV_BITS) - 1u), (track_made >> KTJ_TR_DEV_BITS) | ((uint64_t)(track_made_high & 31u) << 42), track_made_high >> 5);
        track_seen = upto_first;
      }
      if (!open) {
        open = true;
        const uint64_t i_first = i0 + (first >> 2), pos = prefix_len + offs[i_first];
        doc = out + (pos & ~127ull);
        pend = (uint32_t)(pos & 127u);   /* bytes of the tile in use */
        own = pend >> 4;                 /* first block of the tile that this wavefront stores */
        const uint32_t fill = pend & 15u;
        if (fill) {
          if (i_first == 0) { /* what precedes the first activity is in the document already */
            if (lane == 0) {
              uint64_t* w = reinterpret_cast<uint64_t*>(doc + (pend & ~15u));
              uint64_t lo = w[0], hi = w[1];
              if (fill < 8) { lo &= (1ull << (8 * fill)) - 1ull; hi = 0; } else if (fill > 8) hi &= (1ull << (8 * (fill - 8))) - 1ull; else hi = 0;
              uint64_t* t = reinterpret_cast<uint64_t*>(tile + (pend & ~15u));
              t[0] = lo; t[1] = hi;
            }
          } else if (fill < 8) {
            if (lane == 0) *reinterpret_cast<uint64_t*>(tile + (pend & ~15u)) = tail_bytes(tail_kind_at(kind_sorted, rows, perm, i_first - 1, ctx), fill);
          } else ++own; /* the predecessor writes this block */
        }
      }
      wave_lds_order();
      /* 64 segments at a time: what the next ones are made of is read before these are put together */
      struct Piece { v4u32 a, num; uint32_t desc, at, at2, part; }; /* at: in LDS; WV_FAR: place in the string's blob, in units of sixteen bytes */
#define WV_FAR (1u << 30)
#define WV_FAR_ARG (1u << 31)
      uint32_t part_after = 0;
      auto fetch = [&]() {
        Piece x;
        /* which part each segment belongs to: the first segments of the parts behind this one are marked, the marks counted (one that
         * is 64 behind marks the first, which does not count, like the sixty-fifth it is) */
        const uint32_t rel = WV_PART_START(parts[part + 1u + lane]) - g;
        const bool follows = lane < n_parts - 1u - part && rel <= 64u;
        const uint64_t marks = __builtin_amdgcn_ballot_w64(__builtin_amdgcn_ds_permute((int)(follows ? rel * 4u : 0u), 1) != 0);
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(marks >> 33), __builtin_amdgcn_mbcnt_lo((uint32_t)(marks >> 1), 0u));
        x.part = part + rank;
        uint32_t pr = parts[x.part];
        part_after = part + (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(follows));
        const bool valid = lane < g_end - g;
        const uint32_t seg = g + lane - WV_PART_START(pr);
        if (!valid) pr = 0;
        const uint32_t kind = WV_PART_KIND(pr), vrow = mine + WV_PART_ACT(pr) * WV_VAL_BYTES;
        const uint32_t idx = kind == 0 && valid ? WV_PART_DESC(pr) + seg : 0u;
        x.desc = *reinterpret_cast<const uint32_t*>(wv_lds + WV_BOOK_DESC + idx * 4u);
        x.at = WV_WD_UNIT(x.desc) * 16u;
        x.at2 = WV_WD_UNIT2(x.desc) * 16u;
        if (x.desc & WV_WD_TRACK) {
          x.desc |= (uint32_t)(track_lens >> (WV_WD_UNIT(x.desc) * 2u)) & 0x7Fu; /* (four units to a text) */
          x.at += mine + WV_TRACK_AT;
          x.at2 += mine + WV_TRACK_AT;
        }
        if (kind != 0) {
          const uint64_t r = *reinterpret_cast<const uint64_t*>(wv_lds + vrow + WV_VAL(S_RUN) + (2u - kind) * 8u);
          const uint32_t rest = ((uint32_t)(r >> 32) & 0xFFFFu) - seg * KTJ_WEAVE_LIT, near = (uint32_t)(r >> 48);
          x.at = (near ? mine + near : (uint32_t)r) + (seg << (near ? 6u : 2u));
          x.at2 = x.at + 32u;
          x.desc = WV_WD(rest < KTJ_WEAVE_LIT ? rest : KTJ_WEAVE_LIT, S_NONE, 0u, 0u) | (near ? 0u : kind == 1u ? WV_FAR : WV_FAR | WV_FAR_ARG);
        }
        x.a = *reinterpret_cast<const v4u32*>(wv_lds + (x.desc & WV_FAR ? 0u : x.at));
        const uint32_t slot = WV_WD_SLOT(x.desc);
        x.num = *reinterpret_cast<const v4u32*>(wv_lds + vrow + slot * 16u - 16u); /* (S_NONE: what lies there, which does not count) */
        if (__builtin_amdgcn_ballot_w64(slot == S_K) && slot == S_K) { /* in the place of S_RUN */
          x.num = *reinterpret_cast<const v4u32*>(wv_lds + vrow + WV_VAL(S_RUN));
          x.num.w = x.num.y; x.num.y = 0; x.num.z = 0;
        }
        if (slot == S_NONE) x.num.w = 0;
        return x;
      };
      uint32_t nb = 0;
      v2u64 y0, y1, y2, rest;
      /* The tile's whole lines are taken out of it and leave.  Between the two the next segments are fetched, so that neither
       * waits for the other's LDS accesses (the segments after next fetched instead, twelve registers more: the same). */
      auto take_lines = [&]() {
        nb = (pend >> 7) * 8u;
        if (nb) {
          v2u64* tb = reinterpret_cast<v2u64*>(tile);
          /* (three turns reach the end of the tile) */
          if (lane < nb) y0 = tb[lane];
          if (lane + 64u < nb) y1 = tb[lane + 64u];
          if (lane + 128u < nb) y2 = tb[lane + 128u];
          if (lane < 8u) rest = tb[nb + lane];
        }
      };
      auto put_line = [](gptr p, v2u64 x) { if constexpr (PAST) __builtin_nontemporal_store(x, p); else *p = x; };
      auto store_lines = [&]() {
        if (nb) {
          const gptr dst = reinterpret_cast<gptr>((uintptr_t)doc);
          if (lane < 8u) reinterpret_cast<v2u64*>(tile)[lane] = rest;
          if (lane < nb && lane >= own) put_line(dst + lane, y0);
          if (lane + 64u < nb) put_line(dst + lane + 64u, y1);
          if (lane + 128u < nb) put_line(dst + lane + 128u, y2);
          wave_lds_order();
          doc += (uint64_t)nb * 16u;
          pend &= 127u;
          own = 0;
          nb = 0;
        }
      };
      /* As many of them as the tile has room for; the others are fetched again.  (All of them, in two turns over the tile:
       * 5 % more for 11 million kernels.) */
      auto put = [&](Piece& x) {
        const uint32_t len = WV_WD_LEN(x.desc);
        const bool far = (x.desc & WV_FAR) != 0;
        v4u32 b, c, d; /* (what a text does not reach does not count) */
        if (len > 16u && !far) {
          b = *reinterpret_cast<const v4u32*>(wv_lds + x.at + 16u);
          if (len > 32u) {
            c = *reinterpret_cast<const v4u32*>(wv_lds + x.at2);
            if (len > 48u) d = *reinterpret_cast<const v4u32*>(wv_lds + x.at2 + 16u);
          }
        }
        if (__builtin_amdgcn_ballot_w64(far)) {
          if (far) {
            const gsrc src = reinterpret_cast<gsrc>((uint64_t)(uintptr_t)(x.desc & WV_FAR_ARG ? ctx.dict.arg_blob : ctx.dict.name_blob)) + x.at;
            x.a = src[0];
            if (len > 16u) { b = src[1]; if (len > 32u) { c = src[2]; if (len > 48u) d = src[3]; } }
          }
          /* waited for here, once for the four of them and only where there are any: this wait is also for the lines that
           * store_lines has just stored, as loads and stores are counted together and in order */
          asm volatile("" : "+v"(x.a), "+v"(b), "+v"(c), "+v"(d));
        }
        const uint32_t n_num = x.num.w >> 24;
        x.num.w &= 0xFFFFFFu;
        const bool valid = lane < g_end - g;
        const uint32_t mine_len = valid ? len + n_num : 0u;
        const uint32_t end = dpp_add(mine_len);
        const bool now = valid && end + pend <= room;
        const uint32_t n = (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(now)); /* (never 0: a segment is shorter than the tile) */
        if (now) put_segment(tile, pend + (end - mine_len), len, x.a, b, c, d, n_num, x.num);
        pend += __builtin_amdgcn_readlane(end, n - 1u);
        wave_lds_order();
        take_lines();
        part = n == 64u ? part_after : __builtin_amdgcn_readlane(x.part, n);
        g += n;
      };
      while (g < g_end) {
        Piece x = fetch();
        store_lines();
        put(x);
      }
      asm volatile("" : "+v"(q0), "+v"(q1), "+v"(row)); /* the next turn's rows are waited for here, and not behind these lines' stores */
      store_lines();
      if (next_lane != 64u && !(todo & (1ull << next_lane))) close_document(i0 + (next_lane >> 2));
    }
  }
  if (open) close_document(i_end);
}

hipError_t weave_activities(const TextRow* rows, const uint32_t* perm, const uint64_t* offs, const uint8_t* kind_sorted, uint64_t n_most, EmitCtx ctx, char* out,
                 uint64_t prefix_len, const Scalars* sc, const SchemaBook* schemas, const WideText* wide, hipStream_t st) {
  if (n_most == 0) return hipSuccess;
  static_assert(WV_TILE_MOST / 16u <= 3u * 64u && WV_TILE_MOST + 128u <= WV_SPACE, "three turns, and a line behind them");
  static_assert(WV_LDS_BYTES <= 32000u, "five workgroups per CU: 160 KB in pieces of 1280 bytes");
  const uint64_t turns = (n_most + WV_ROWS - 1) / WV_ROWS;
  const uint32_t waves = turns >= 256u * WV_WAVES ? WV_WAVES : turns <= 256u ? 1u : (uint32_t)((turns + 255u) / 256u);
  /* Turns of a wavefront: those of a pass that all wavefronts at once can take with up to forty each are dealt out to them (3 million
   * records 37 each 400 us, 19 and twice as many wavefronts 407).  Of longer passes each takes about twelve: the fewer, the closer
   * together lie the pieces of the document that are written at a time, but each copies the book (22 million records with 8, 12, 16,
   * 24, 40: 3.09, 2.97, 3.00, 3.04, 3.04 ms; 5 million operators with long strings 2.45, 2.44, 2.52, 2.50, 2.51).  Around the line, which is at 3.28 million rows,
   * whole passes dealt out and with about twelve turns each: 2.55 million records 855 and 863 us, 3.33 million 1070 and 1077, 3.9 million 1212 and 1220, 3.16 million
   * kernels 1020 and 1016, operators with long strings 3 million 2050 and 2026, 3.5 million 2382 and 2360. */
  const uint64_t at_once = 256u * 20u, times = turns <= at_once * 40u ? 1u : (turns + at_once * 12u - 1u) / (at_once * 12u);
  const uint32_t rounds = (uint32_t)((turns + at_once * times - 1u) / (at_once * times));
  const auto kernel = n_most >= WV_PAST_FROM ? k_weave<true> : k_weave<false>;
  hipLaunchKernelGGL(kernel, dim3(grid_for(turns, waves * rounds)), dim3(waves * 64u), 0, st, rows, perm, offs,
                     kind_sorted, ctx, out, prefix_len, sc, rounds, schemas, wide);
  return KTJ_LAUNCH_CHECK();
}

}  // namespace gpu
}  // namespace ktj
