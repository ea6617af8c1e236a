/*
 * weave_core.h — an activity's text as a list of segments: what the emit kernel of weave.hip writes with one
 * lane per segment, and the tables it takes the fixed text from.
 *
 * A segment is up to 64 bytes of text followed by at most one number.  An activity is a few parts, each a run
 * of consecutive descriptors of the table below (the head of the event by its category, the body up to the
 * args, the args by kind, the end with its flow event) or a dictionary string in pieces of 64 bytes.  text_row()
 * names the parts of a joined row; it answers false for the rows that only format_activity (fmt_core.h) prints.
 * The text here is that of fmt_core.h; the CPU tests hold the two against each other for every kind of row.
 */
#ifndef KTJ_WEAVE_CORE_H_
#define KTJ_WEAVE_CORE_H_

#include "fmt_core.h"
#include "mat_core.h"

namespace ktj {
namespace weave {

#define KTJ_WEAVE_LIT 64u          /* bytes of text per segment */
#define KTJ_WEAVE_MAX_RUN 12800u   /* longer strings are left to format_activity */

/* The numbers of one activity, printed: sixteen bytes each, up to fifteen characters (zeros behind them) and their count
 * in the last byte.  Activities with longer ones are left to format_activity. */
enum : uint32_t {
  S_NONE = 0,
  S_A,                             /* cid, or queue, or context, or the fourth of a schema's numbers */
  S_TS,
  S_X, S_Y,                        /* grid and block ("a, b, c"), addresses, or bytes; a double of up to 24 characters: S_Y and S_Z */
  S_Z,                             /* shared memory or bytes */
  S_EXT,                           /* with the comma behind it where something follows */
  S_FLOW, S_DUR,
  S_RUN,                           /* the strings between the args and of the name, eight bytes each: place in the blob in units of sixteen bytes,
                                      length, place in LDS (0: it stays in the blob) */
  S_K,                             /* copy kind, in place of the first of them */
  S_PID = S_TS, S_TID = S_DUR, S_LEAD = S_X /* in the pieces of the track's texts */
};

/* A joined row as the size pass leaves it for the weaver: a line of eight blocks of sixteen bytes.  Most numbers are
 * short: S_Z, S_EXT, S_FLOW and S_DUR have twelve bytes (eleven characters) of the first four blocks, whose last words are
 * plan, name, lens and more; S_A has eight of the fifth (seven characters), in front of the track, and where there is nothing else
 * for it four more in the word for more (the sequence number of an operator is the fourth number of its schema, and a long job
 * has more than 10 million of them); the others a block each.
 *
 * A time has eighteen characters and more where the base lies months behind (libkineto floors it to 91 days) or at 0, more than
 * S_TS has.  What is above 10^11 us (28 hours) is the same for nearly all rows: that number, the time's lead, is printed once
 * for many, with the track's texts, and S_TS then has the eleven digits behind it with their zeros.  Where a row has a lead, its
 * sixteen bits stand in the count bytes of the first four blocks, whose counts take four bits each.  (In every row, without
 * the bit that says so: size pass of 22 million records 27 us longer.)
 *
 * (Sixteen bytes
 * for each number, 160 for a row: the size pass, whose rows wait in LDS, ran three instead of four wavefronts per SIMD,
 * 22 million records 1.32 + 0.70 + 0.15 ms instead of 1.15 + 0.57 + 0.13.) */
struct alignas(16) TextRow { uint32_t w[8][4]; };
/* The text of a double that has no room in its row, for generic records whose schemas have one among too many numbers.  (Printed
 * by the weaver, with a quarter of the lanes, it took two thirds of its time for 5 million such records.) */
struct alignas(16) WideText { uint64_t w[4]; };
#define KTJ_TR_BLOCK(slot) (((slot) + 3u) & 7u)
#define KTJ_TR_PLAN 0u             /* KTJ_TR_*, the thread's bits from 42 on */
#define KTJ_TR_NAME 1u             /* place of the name in its blob, in units of sixteen bytes */
#define KTJ_TR_LENS 2u             /* its length; << 16: that of the string or double between the args' parts; KTJ_TR_HAS_LEAD */
#define KTJ_TR_MORE 3u             /* the string's place in its blob; the WideText's number; a copy's kind as text; S_A's eighth character and the following */
#define KTJ_TR_A_NEAR 7u           /* characters of S_A in its block */
static_assert(KTJ_WEAVE_MAX_RUN < 0x8000u, "a length and a bit");
static_assert(sizeof(TextRow) == 128 && sizeof(TextRow) >= sizeof(MatRow), "a row that is left to format_activity is a MatRow in the same place");
/* a row of the other kind: the last byte, S_Y's count of characters otherwise */
#define KTJ_ROW_LEFT 0xFFu
#define KTJ_TR_TYPE(x) ((x) & 31u)
#define KTJ_TR_NAMED(x) (((x) >> 5) & 127u)    /* a part, or KTJ_TR_NAME_RUN */
#define KTJ_TR_NAME_RUN 127u
#define KTJ_TR_BODY(x) (((x) >> 12) & 3u)      /* R_BODY_NONE and the following */
#define KTJ_TR_ARGS(x) (((x) >> 14) & 127u)    /* A_*, or KTJ_TR_SCHEMA + schema, or KTJ_TR_NO_ARGS */
#define KTJ_TR_SCHEMA 64u
#define KTJ_TR_NO_ARGS 127u
#define KTJ_TR_TAIL(x) (((x) >> 21) & 15u)     /* R_TAIL and the following */
#define KTJ_TR_BETWEEN(x) (((x) >> 25) & 3u)   /* 1 string, 2 double in S_Y and S_Z, 3 double beside the row (WideText) */
#define KTJ_TR_TID_HIGH(x) ((x) >> 27)
#define KTJ_LEAD_UNIT 100000000000ull          /* us */
#define KTJ_TR_HAS_LEAD (1u << 31)
#define KTJ_TR_LEN1(lens) (((lens) >> 16) & 0x7FFFu)
#define KTJ_TR_LEAD_NIBBLE(w) ((w) >> 28)      /* of the third word of a block: the first block has the lead's lowest */
#define KTJ_TR_COUNT(w) (((w) >> 24) & 15u)    /* of the same word */
#define KTJ_TR_DEV_BITS 22u                    /* a track's process or device, and 42 of the thread's or stream's 47 bits */

/* Neighbouring activities share their track, so process and thread (device and stream), and the lead of the time behind
 * them, are printed once for many: these texts are made where the track or the lead changes, and are the text of one segment each. */
enum : uint32_t { T_BODY = 0, T_FLOW, T_DEVICE, T_MEMSET, T_STREAM, T_COUNT };

/* descriptor of a segment: length of its text, number behind it, place of the text in units of sixteen bytes (in the
 * book, or among the track's texts) */
#define KTJ_WD(len, slot, unit) ((len) | ((slot) << 8) | ((unit) << 12))
#define KTJ_WD_LEN(x) ((x) & 0x7Fu)
#define KTJ_WD_SLOT(x) (((x) >> 8) & 0xFu)
#define KTJ_WD_UNIT(x) (((x) >> 12) & 0xFFFu)
#define KTJ_WD_TRACK (1u << 24)    /* (the length is the wavefront's) */

/* An activity is: head by its category, name, body up to the args, the args (one part, or two around a string or a
 * double), and the end with its flow event. */
enum : uint32_t {
  R_HEAD = 0,                                    /* + type */
  R_COPY_NAME = 32,                              /* + direction */
  R_MEMSET_NAME = 37,                            /* + memory kind, 8 = any other */
  R_BODY_NONE = 46, R_BODY_ARGS, R_BODY_EXT,
  R_ARGS,                                        /* + A_* */
  R_ARGS2 = R_ARGS + 32,                         /* the same, behind the string */
  R_TAIL = R_ARGS2 + 32,                         /* + 5 where an args object closes, + 10 where an array does before it;
                                                    + flow: none, start, end, the same of fwdbwd */
  R_PIECES = R_TAIL + 15,
  R_COUNT
};
enum : uint32_t {
  A_DEFAULT = 0, A_LAUNCH, A_LAUNCH_NAMED, A_COPY, A_MALLOC, A_MALLOC_BYTES,
  A_KERNEL, A_KERNEL_SIZE, A_KERNEL_GRID, A_MEMSET, A_MEMSET_BANDWIDTH,
  A_COPIED,                                      /* + 3 * direction, + 1 with bytes, + 2 with a grid */
  /* Bytes without a bandwidth, as copies of no duration have: + 0 a kernel's, + 1 + direction a copy's.  (Left to k_emit_direct, 50 of
   * them among 3 million records cost a launch of 33 us: a pass of 1251 us, 1217 now.) */
  A_BYTES_ONLY = A_COPIED + 15,
  A_COUNT = A_BYTES_ONLY + 6
};
static_assert(A_COUNT <= R_ARGS2 - R_ARGS && A_COUNT <= KTJ_TR_SCHEMA, "the args' parts");
/* a part: first descriptor, their number */
#define KTJ_WREF(base, count) ((base) | ((count) << 16))
#define KTJ_WREF_BASE(r) ((r) & 0xFFFFu)
#define KTJ_WREF_COUNT(r) ((r) >> 16)

/* The args of generic records follow their schema: descriptors and texts for the first schemas of a trace are made on the
 * device (render_schemas), behind the fixed ones.  A schema takes up to four numbers (two of them may be arrays of up to
 * three), and one string or one double. */
constexpr uint32_t MAX_DESC = 208, MAX_TEXT = 232, N_PIECES = 13;
constexpr uint32_t MAX_SCHEMAS = 16, SCHEMA_DESC = 56, SCHEMA_TEXT = 60;
enum : uint32_t { I_NONE = 0, I_I64, I_U64, I_BOOL, I_ARRAY }; /* I_ARRAY + number of elements */
struct SchemaPlan {
  uint32_t args, args2;            /* parts (0: the schema is none of these) */
  uint32_t what;                   /* 1: taken, 2: prints something, 4: one string and nothing else, which may be blank; << 8: argument
                                      slots; << 16: KTJ_TR_BETWEEN; << 24: its slot */
  uint32_t item[4];                /* of item_slot(0..3): I_* | slot << 8 */
  uint32_t chars;                  /* of the parts' texts */
};
struct SchemaBook {
  uint32_t text[SCHEMA_TEXT * 4];
  SchemaPlan plan[MAX_SCHEMAS];
  uint32_t desc[SCHEMA_DESC];
};

struct Book {
  uint32_t text[MAX_TEXT * 4];
  uint32_t ref[R_COUNT];
  uint32_t desc[MAX_DESC];
  uint32_t n_desc, n_text;
};

/* In the weaver's LDS the schemas' texts lie behind the book's texts: unit of the first of them. */
constexpr uint32_t SCHEMA_UNIT = MAX_TEXT;

/* In the texts byte 1 and a letter is a number, which ends a segment; byte 2 and a letter is a text of the track's. */
#define WN(c) "\x01" c
#define WT(c) "\x02" c
struct Builder {
  Book b{};
  char cur[KTJ_WEAVE_LIT] = {};
  uint32_t n = 0, at = 0, track = T_COUNT;
  constexpr void begin() { at = b.n_desc; n = 0; track = T_COUNT; }
  constexpr void segment(uint32_t slot) {
    if (track != T_COUNT) { /* its text is put in by the wavefront */
      b.desc[b.n_desc++] = KTJ_WD(0u, slot, track * (KTJ_WEAVE_LIT / 16u)) | KTJ_WD_TRACK;
      track = T_COUNT;
      return;
    }
    uint32_t w[KTJ_WEAVE_LIT / 4] = {}, unit = 0;
    for (uint32_t i = 0; i < n; ++i) w[i / 4] |= (uint32_t)(unsigned char)cur[i] << (8 * (i % 4));
    const uint32_t units = (n + 15) / 16;
    for (; unit + units <= b.n_text; ++unit) { /* the same bytes somewhere already? */
      bool same = true;
      for (uint32_t i = 0; i < units * 4; ++i) same = same && b.text[unit * 4 + i] == w[i];
      if (same) break;
    }
    if (unit + units > b.n_text) {
      unit = b.n_text;
      for (uint32_t i = 0; i < units * 4; ++i) b.text[unit * 4 + i] = w[i];
      b.n_text += units;
    }
    b.desc[b.n_desc++] = KTJ_WD(n, slot, unit);
    n = 0;
  }
  constexpr void flush() { if (n) segment(S_NONE); }
  constexpr void number(char c) {
    const char* const codes = "auxyzefrk"; /* S_A and the following */
    for (uint32_t k = 0; codes[k]; ++k) if (codes[k] == c) segment(c == 'k' ? S_K : S_A + k);
  }
  constexpr void add(const char* s) {
    for (; *s; ++s) {
      if (*s == 1) { number(*++s); continue; }
      if (*s == 2) { flush(); track = (uint32_t)(*++s - '0'); continue; }
      if (n == KTJ_WEAVE_LIT) flush();
      cur[n++] = *s;
    }
  }
  constexpr void end(uint32_t ref) { flush(); b.ref[ref] = KTJ_WREF(at, b.n_desc - at); }
  constexpr void part(uint32_t ref, const char* s, const char* s2 = "", const char* s3 = "", const char* s4 = "") { begin(); add(s); add(s2); add(s3); add(s4); end(ref); }
};
constexpr Book make_book() {
  Builder b;
  const char* const cat[29] = {
      "cpu_op", "user_annotation", "gpu_user_annotation", "gpu_memcpy", "gpu_memset", "kernel", "external_correlation", "cuda_runtime", "cuda_driver",
      nullptr, "python_function", "overhead", "mtia_runtime", "mtia_ccp_events", "mtia_insight", "cuda_sync", "cuda_event", nullptr, "glow_runtime",
      "cuda_profiler_range", "hpu_op", "xpu_runtime", "xpu_driver", "collective_comm", "privateuse1_runtime", "privateuse1_driver", nullptr,
      "xpu_sync", nullptr};
  for (uint32_t t = 0; t < 29; ++t) /* (instant and counter events have none) */
    if (cat[t]) b.part(R_HEAD + t, "\n  {\n    \"ph\": \"X\",\n    \"cat\": \"", cat[t], "\",\n    \"name\": \"");
  b.part(R_COPY_NAME + 0, "Memcpy <unknown> (? -> ?)");
  b.part(R_COPY_NAME + KTJ_COPY_H2H, "Memcpy HtoH (Host -> Host)");
  b.part(R_COPY_NAME + KTJ_COPY_H2D, "Memcpy HtoD (Host -> Device)");
  b.part(R_COPY_NAME + KTJ_COPY_D2H, "Memcpy DtoH (Device -> Host)");
  b.part(R_COPY_NAME + KTJ_COPY_D2D, "Memcpy DtoD (Device -> Device)");
  b.part(R_MEMSET_NAME + KTJ_MEMKIND_UNKNOWN, "Memset (Unknown)");
  b.part(R_MEMSET_NAME + KTJ_MEMKIND_PAGEABLE, "Memset (Pageable)");
  b.part(R_MEMSET_NAME + KTJ_MEMKIND_PINNED, "Memset (Pinned)");
  b.part(R_MEMSET_NAME + KTJ_MEMKIND_DEVICE, "Memset (Device)");
  b.part(R_MEMSET_NAME + KTJ_MEMKIND_ARRAY, "Memset (Array)");
  b.part(R_MEMSET_NAME + KTJ_MEMKIND_MANAGED, "Memset (Managed)");
  b.part(R_MEMSET_NAME + KTJ_MEMKIND_DEVICE_STATIC, "Memset (Device Static)");
  b.part(R_MEMSET_NAME + KTJ_MEMKIND_MANAGED_STATIC, "Memset (Managed Static)");
  b.part(R_MEMSET_NAME + 8, "Memset (Unrecognized)");
#define KTJ_WEAVE_BODY WT("0") WN("u") ",\n    \"dur\": " WN("r")
  b.part(R_BODY_NONE, KTJ_WEAVE_BODY "\n    \n  },");
  b.part(R_BODY_ARGS, KTJ_WEAVE_BODY "\n    ,\n    \"args\": {\n      ");
  b.part(R_BODY_EXT, KTJ_WEAVE_BODY "\n    ,\n    \"args\": {\n      \"External id\": " WN("e"));
#define KTJ_WEAVE_CID "\"cid\": " WN("a") ", \"correlation\": " WN("f")
#define KTJ_WEAVE_LAUNCH ", \"grid\": [" WN("x") "], \"block\": [" WN("y") "], \"shared memory\": " WN("z")
#define KTJ_WEAVE_SIZE ", \"bytes\": " WN("x") ", \"memory bandwidth (GB/s)\": "
#define KTJ_WEAVE_GRID ", \"grid\": [" WN("x") "], \"block\": [" WN("y")
#define KTJ_WEAVE_DEVICE WT("2") WN("a") ", \"correlation\": " WN("f") ", \"kind\": \""
#define KTJ_WEAVE_MEMSET WT("3") WN("a") WT("4") WN("f") ", \"bytes\": " WN("x")
  b.part(R_ARGS + A_DEFAULT, KTJ_WEAVE_CID);
  b.part(R_ARGS + A_LAUNCH, KTJ_WEAVE_CID KTJ_WEAVE_LAUNCH);
  b.part(R_ARGS + A_LAUNCH_NAMED, "\"kernel\": \"");
  b.part(R_ARGS2 + A_LAUNCH_NAMED, "\", " KTJ_WEAVE_CID KTJ_WEAVE_LAUNCH);
  b.part(R_ARGS + A_COPY, KTJ_WEAVE_CID ", \"src\": \"0x" WN("x") "\", \"dst\": \"0x" WN("y") "\", \"bytes\": " WN("z") ", \"kind\": \"" WN("k") "\"");
  b.part(R_ARGS + A_MALLOC, KTJ_WEAVE_CID ", \"ptr\": \"0x" WN("x") "\"");
  b.part(R_ARGS + A_MALLOC_BYTES, "\"bytes\": " WN("z") ", " KTJ_WEAVE_CID ", \"ptr\": \"0x" WN("x") "\"");
  b.part(R_ARGS + A_KERNEL, KTJ_WEAVE_DEVICE "Dispatch Kernel\"");
  b.part(R_ARGS + A_KERNEL_SIZE, KTJ_WEAVE_DEVICE "Dispatch Kernel\"" KTJ_WEAVE_SIZE);
  b.part(R_ARGS + A_KERNEL_GRID, KTJ_WEAVE_DEVICE "Dispatch Kernel\"" KTJ_WEAVE_GRID);
  b.part(R_ARGS + A_MEMSET, KTJ_WEAVE_MEMSET);
  b.part(R_ARGS + A_MEMSET_BANDWIDTH, KTJ_WEAVE_MEMSET ", \"memory bandwidth (GB/s)\": ");
  const char* const direction[5] = {"<unknown>", "HtoH", "HtoD", "DtoH", "DtoD"}; /* KTJ_COPY_H2H = 1 and so on */
  for (uint32_t d = 0; d < 5; ++d) {
    b.part(R_ARGS + A_COPIED + 3 * d, KTJ_WEAVE_DEVICE, direction[d], "\"");
    b.part(R_ARGS + A_COPIED + 3 * d + 1, KTJ_WEAVE_DEVICE, direction[d], "\"" KTJ_WEAVE_SIZE);
    b.part(R_ARGS + A_COPIED + 3 * d + 2, KTJ_WEAVE_DEVICE, direction[d], "\"" KTJ_WEAVE_GRID);
  }
  for (uint32_t k = 0; k < 6; ++k) { /* as with a bandwidth, but for the text in front of it, which is the last segment */
    const uint32_t with = b.b.ref[R_ARGS + (k ? A_COPIED + 3 * (k - 1) + 1 : (uint32_t)A_KERNEL_SIZE)];
    b.b.ref[R_ARGS + A_BYTES_ONLY + k] = KTJ_WREF(KTJ_WREF_BASE(with), KTJ_WREF_COUNT(with) - 1);
  }
  const char* const close[3] = {"", "\n    }\n  },", "]\n    }\n  },"};
  const char* const flow[5] = {
      "", "\n  {\n    \"ph\": \"s\",\n    \"id\": " WN("f") WT("1") WN("u"), "\n  {\n    \"ph\": \"f\",\n    \"id\": " WN("f") WT("1") WN("u"),
      "\n  {\n    \"ph\": \"s\",\n    \"id\": " WN("f") WT("1") WN("u"), "\n  {\n    \"ph\": \"f\",\n    \"id\": " WN("f") WT("1") WN("u")};
  const char* const last[5] = {
      "", ",\n    \"cat\": \"ac2g\",\n    \"name\": \"ac2g\"\n    \n  },", ",\n    \"cat\": \"ac2g\",\n    \"name\": \"ac2g\"\n    , \"bp\": \"e\"\n  },",
      ",\n    \"cat\": \"fwdbwd\",\n    \"name\": \"fwdbwd\"\n    \n  },",
      ",\n    \"cat\": \"fwdbwd\",\n    \"name\": \"fwdbwd\"\n    , \"bp\": \"e\"\n  },"};
  for (uint32_t c = 0; c < 3; ++c)
    for (uint32_t f = 0; f < 5; ++f) b.part(R_TAIL + 5 * c + f, close[c], flow[f], last[f]);
  /* the pieces of the track's texts, in their order: WN("u") stands for the process (device), WN("r") for the thread (stream),
   * WN("x") for the time's lead */
  b.part(R_PIECES, "\",\n    \"pid\": " WN("u") ",\n    \"tid\": " WN("r") ",\n    \"ts\": " WN("x"));
  b.add(",\n    \"pid\": " WN("u") ",\n    \"tid\": " WN("r") ",\n    \"ts\": " WN("x"));
  b.add("\"device\": " WN("u") ", \"stream\": " WN("r") ", \"hsa_queue\": "); b.flush();
  b.add("\"device\": " WN("u") ", \"context\": "); b.flush();
  b.add(", \"stream\": " WN("r") ", \"correlation\": "); b.flush();
  return b.b;
}

static_assert(KTJ_COPY_H2H == 1 && KTJ_COPY_D2D == 4, "the directions' names are in this order");

constexpr Book BOOK = make_book();
/* characters of the parts' texts, the track's without their numbers; and of these by themselves */
struct Chars { uint32_t of[R_COUNT], track[T_COUNT]; };
constexpr Chars count_chars(const Book& b) {
  Chars c{};
  uint32_t track[T_COUNT] = {}; /* pieces 0-2, 3-5, 6-8, 9-10, 11-12 are a text each */
  for (uint32_t k = 0; k < N_PIECES; ++k)
    track[k < 9 ? k / 3 : k < 11 ? 3 : 4] += KTJ_WD_LEN(b.desc[KTJ_WREF_BASE(b.ref[R_PIECES]) + k]);
  for (uint32_t k = 0; k < T_COUNT; ++k) c.track[k] = track[k];
  for (uint32_t r = 0; r < R_COUNT; ++r)
    for (uint32_t k = 0; k < KTJ_WREF_COUNT(b.ref[r]); ++k) {
      const uint32_t i = KTJ_WREF_BASE(b.ref[r]) + k;
      c.of[r] += KTJ_WD_LEN(b.desc[i]);
      if (b.desc[i] & KTJ_WD_TRACK) c.of[r] += track[KTJ_WD_UNIT(b.desc[i]) / (KTJ_WEAVE_LIT / 16u)];
    }
  return c;
}
constexpr Chars CHARS = count_chars(BOOK);
constexpr bool tracks_fit(const Book& b) { /* with process or device of 22 bits and thread or stream of 47, and no lead */
  uint32_t track[T_COUNT] = {};
  for (uint32_t k = 0; k < N_PIECES; ++k) {
    const uint32_t d = b.desc[KTJ_WREF_BASE(b.ref[R_PIECES]) + k], slot = KTJ_WD_SLOT(d);
    track[k < 9 ? k / 3 : k < 11 ? 3 : 4] += KTJ_WD_LEN(d) + (slot == S_PID ? 7u : slot == S_TID ? 15u : 0u);
  }
  for (uint32_t k = 0; k < T_COUNT; ++k) if (track[k] > KTJ_WEAVE_LIT) return false;
  return true;
}
static_assert(tracks_fit(BOOK), "a track's text is the text of one segment");
/* characters that process, thread and lead may have together */
constexpr uint32_t TRACK_ROOM = KTJ_WEAVE_LIT - (CHARS.track[T_BODY] > CHARS.track[T_FLOW] ? CHARS.track[T_BODY] : CHARS.track[T_FLOW]);
static_assert(BOOK.n_text <= MAX_TEXT && BOOK.n_desc <= MAX_DESC, "the book's tables");
#if defined(__HIP_DEVICE_COMPILE__)
static __device__ constexpr Chars chars_table = CHARS;
#else
static constexpr Chars chars_table = CHARS;
#endif
template <uint32_t R> KTJ_HD KTJ_FI inline uint32_t chars_of() { constexpr uint32_t n = CHARS.of[R]; return n; }

KTJ_HD KTJ_FI inline uint32_t item_slot(uint32_t j) { return j == 0 ? S_X : j == 1 ? S_Y : j == 2 ? S_Z : S_A; }

/* ---- the schemas' texts ---- */
#define KTJ_WEAVE_FIELDS 128u      /* fields of all schemas together (and of those behind, none is taken) */
#define KTJ_WEAVE_KEY 48u          /* longest key */
struct SchemaSize { uint32_t desc, units; };
/* One schema by itself, as if it were the first: its plan, its descriptors, and where the characters of its fields go: place[],
 * in bytes, those behind the field's value << 16, KTJ_WEAVE_COMMA.  Behind others it is moved by what they have. */
#define KTJ_WD_MOVED(desc, units) ((desc) + ((units) << 12))
#define KTJ_WREF_MOVED(ref, descs) ((ref) + (descs))
#define KTJ_PLACE_MOVED(place, units) ((place) + (units) * 16u * (((place) >> 16) ? 0x10001u : 1u))
#define KTJ_WEAVE_COMMA (1u << 15)
KTJ_HD inline SchemaSize lay_out_schema(const ktj_field* field, const uint32_t* key_len, uint32_t n_fields, SchemaPlan* plan, uint32_t* desc, uint32_t* place) {
  SchemaPlan& p = *plan; /* (in LDS on the device: its items have no fixed places) */
  p.args = p.args2 = p.what = p.chars = 0;
  for (uint32_t j = 0; j < 4; ++j) p.item[j] = I_NONE;
  uint32_t n_desc = 0, n_unit = 0, len = 0, d_args = 0, between = 0, between_slot = 0, slot = 0, n_simple = 0, n_array = 0, arrays = 0;
  bool taken = true, comma = false;
  auto end = [&](uint32_t number) {
    if (n_desc >= SCHEMA_DESC || n_unit >= SCHEMA_TEXT) { taken = false; len = 0; return; }
    desc[n_desc++] = KTJ_WD(len, number, SCHEMA_UNIT + n_unit);
    p.chars += len;
    n_unit += (len + 15u) / 16u;
    len = 0;
  };
  /* (a segment that is full ends at a unit's end: the characters lie one behind the other all the same) */
  auto chars = [&](uint32_t n) {
    while (len + n > KTJ_WEAVE_LIT) { n -= KTJ_WEAVE_LIT - len; len = KTJ_WEAVE_LIT; end(S_NONE); }
    len += n;
  };
  auto here = [&]() { return n_unit * 16u + len; };
  auto number = [&](uint32_t j, uint32_t what) {
    if (j >= 4u) { taken = false; return; }
    p.item[j] = what | (slot << 8);
    end(item_slot(j));
  };
  uint32_t numbers = 0;
  bool real = false;
  for (uint32_t f = 0; f < n_fields; ++f) {
    const uint32_t type = field[f].type;
    arrays += type == KTJ_F_I64_ARRAY && field[f].count != 0 ? 1u : 0u;
    numbers += type == KTJ_F_I64 || type == KTJ_F_U64 || type == KTJ_F_BOOL ? 1u : 0u;
    real = real || type == KTJ_F_F64;
  }
  if (arrays > 2u) taken = false;
  real = real && arrays + numbers <= 2u && arrays <= 1u; /* a double takes S_Y and S_Z where the others leave them */
  for (uint32_t f = 0; taken && f < n_fields; ++f) {
    const ktj_field fd = field[f];
    const bool key = fd.key_id != KTJ_NONE, commas = key && comma;
    uint32_t at = here();
    if (key) {
      if (key_len[f] > KTJ_WEAVE_KEY) { taken = false; break; }
      chars((comma ? 2u : 0u) + key_len[f] + 4u);
      comma = true;
    }
    /* a place for a number: S_Z, what the arrays leave of S_X and S_Y, S_A */
    auto simple = [&](uint32_t what) {
      const uint32_t left = (real ? 1u : 2u) - arrays, i = n_simple++, k = real ? i + 1u : i;
      number(k == 0 ? 2u : k <= left ? arrays + k - 1u : k == left + 1u ? 3u : 4u, what);
    };
    switch (fd.type) {
      case KTJ_F_DICT_BEGIN: chars(1); comma = false; break;
      case KTJ_F_DICT_END: chars(1); comma = true; break;
      case KTJ_F_I64: simple(I_I64); break;
      case KTJ_F_U64: simple(I_U64); break;
      case KTJ_F_BOOL: simple(I_BOOL); break;
      case KTJ_F_I64_ARRAY:
        chars(1);
        if (fd.count > 3u) taken = false;
        else if (fd.count) number(n_array++, I_ARRAY + fd.count);
        at |= here() << 16;
        chars(1);
        break;
      case KTJ_F_STR: case KTJ_F_RAW: case KTJ_F_F64:
        if (between) { taken = false; break; }
        if (fd.type == KTJ_F_STR) chars(1);
        if (fd.type == KTJ_F_RAW && !key && n_fields == 1u) p.what |= 4u;
        if (len) end(S_NONE);
        between = fd.type != KTJ_F_F64 ? 1u : real ? 2u : 3u; between_slot = slot;
        p.args = KTJ_WREF(MAX_DESC + d_args, n_desc - d_args);
        d_args = n_desc;
        at |= here() << 16;
        if (fd.type == KTJ_F_STR) chars(1);
        break;
      default: taken = false; break;
    }
    place[f] = at | (commas ? KTJ_WEAVE_COMMA : 0u);
    slot += fd.count;
  }
  if (len) end(S_NONE);
  if (slot > 255u || n_unit > SCHEMA_TEXT) taken = false;
  const uint32_t ref = KTJ_WREF(MAX_DESC + d_args, n_desc - d_args);
  if (between) p.args2 = ref; else p.args = ref;
  p.what |= 1u | (n_fields ? 2u : 0u) | (slot << 8) | (between << 16) | (between_slot << 24);
  SchemaSize size;
  size.desc = taken ? n_desc : 0; size.units = taken ? n_unit : 0;
  if (!taken) p.what = 0;
  return size;
}
/* the characters of one field */
KTJ_HD inline void put_field_text(const ktj_field& fd, const char* key, uint32_t key_len, uint32_t place, char* text) {
  char* t = text + (place & 0x7FFFu);
  if (place & KTJ_WEAVE_COMMA) { *t++ = ','; *t++ = ' '; }
  if (fd.key_id != KTJ_NONE) {
    *t++ = '"';
    for (uint32_t j = 0; j < key_len; ++j) *t++ = key[j];
    *t++ = '"'; *t++ = ':'; *t++ = ' ';
  }
  if (fd.type == KTJ_F_DICT_BEGIN) *t = '{';
  else if (fd.type == KTJ_F_DICT_END) *t = '}';
  else if (fd.type == KTJ_F_I64_ARRAY) { *t = '['; text[place >> 16] = ']'; }
  else if (fd.type == KTJ_F_STR) { *t = '"'; text[place >> 16] = '"'; }
}

/* A bit for each of the first schemas that is not taken whatever its keys are (they lie on the device: a schema whose
 * keys are too long is not among these). */
inline uint32_t schemas_not_taken(const ktj_field* fields, const ktj_schema_desc* schemas, uint32_t n_schemas) {
  const uint32_t key_len[KTJ_WEAVE_FIELDS] = {};
  uint32_t desc[SCHEMA_DESC], place[KTJ_WEAVE_FIELDS], bits = 0, at = 0, n_desc = 0, n_unit = 0;
  for (uint32_t k = 0; k < n_schemas && k < MAX_SCHEMAS; ++k) {
    SchemaPlan plan;
    plan.what = 0;
    if (schemas[k].n_fields <= KTJ_WEAVE_FIELDS - at) {
      const SchemaSize size = lay_out_schema(fields + schemas[k].first_field, key_len, schemas[k].n_fields, &plan, desc, place);
      n_desc += size.desc; n_unit += size.units;
      at += schemas[k].n_fields;
    } else at = KTJ_WEAVE_FIELDS;
    if (!plan.what || n_desc > SCHEMA_DESC || n_unit > SCHEMA_TEXT) bits |= 1u << k;
  }
  return bits;
}

/* ---- records that text_row will refuse, as far as their own numbers say so; for rows inside the capture window.  What it does
 * not say: names beyond KTJ_WEAVE_MAX_RUN, the values of typed arguments, keys, what a device row takes over from a runtime row
 * (counted there), API numbers with no name in the table, leads beside tracks of many digits ---- */
#define KTJ_ELEVEN_DIGITS 100000000000ull
KTJ_HD KTJ_FI inline bool left_by_track(int64_t dev, int64_t res, int64_t rel_ns, int64_t dur) {
  return ((uint64_t)dev >> KTJ_TR_DEV_BITS) != 0 || ((uint64_t)res >> 47) != 0 || rel_ns >= (int64_t)(65536u * KTJ_LEAD_UNIT * 1000u) || dur >= 10000000000ll;
}
/* Times so far apart that their leads differ.  Where that is so for the rows of a workgroup, nearly every row ends the run of
 * the one before it, and k_emit_direct is the better one (10 000 CPU ops over 2^61 ns: 271 us a pass instead of 301). */
KTJ_HD KTJ_FI inline bool far_apart(uint64_t a, uint64_t b) { const uint64_t d = a - b; return (d < 0ull - d ? d : 0ull - d) >= KTJ_LEAD_UNIT * 1000u; }
KTJ_HD KTJ_FI inline bool left_by_three(uint32_t a, uint32_t b, uint32_t c) { /* three_text_of: eleven digits together */
  if (a < 100000u && b < 1000u && c < 1000u) return false;
  return b >= 1000000u || c >= 1000000u || ndigits_u64(a) + ndigits_u64(b) + ndigits_u64(c) > 11;
}
KTJ_HD KTJ_FI inline bool left_generic(const ktj_generic_rec& g, int64_t dev, const EmitCtx& c, uint32_t not_taken) {
  const uint32_t type = g.type & KTJ_M_TYPE_MASK;
  if (type >= 29u || type == KTJ_TYPE_CPU_INSTANT_EVENT || is_counter_type(type)) return true;
  if (g.schema_id < c.n_schemas && (g.schema_id >= MAX_SCHEMAS || ((not_taken >> g.schema_id) & 1u))) return true;
  if (type == KTJ_TYPE_CUDA_SYNC && g.name_id < c.dict.n && (dict_flags(c.dict, g.name_id) & KTJ_SF_STREAM_SYNC)) return true;
  const MatRow m = mat_generic(g, dev);
  const bool wider = type == KTJ_TYPE_GPU_USER_ANNOTATION, flow = (m.meta & KTJ_M_FLOW) != 0;
  bool args = false; /* that are printed whatever they are */
  if (m.ext <= -1000000000 && g.schema_id < c.n_schemas) {
    const ktj_schema_desc sd = c.schemas[g.schema_id];
    args = sd.n_fields != 0 && (sd.n_fields != 1 || c.fields[sd.first_field].type != KTJ_F_RAW);
  }
  return (flow && (wider || (uint64_t)m.flow_id >= KTJ_ELEVEN_DIGITS)) || args ||
         left_by_track(dev, (int64_t)sanitize_tid(m.res), m.ts - c.base_time_ns, m.dur + (wider ? 2 : 0));
}
KTJ_HD KTJ_FI inline bool left_runtime(const ktj_runtime_rec& r, int64_t ts, int64_t dur, const EmitCtx& c, uint32_t n_cids) { /* (beyond them an API has no name) */
  bool left = r.cid >= n_cids || r.id >= KTJ_ELEVEN_DIGITS || left_by_track((int64_t)r.pid, (int64_t)sanitize_tid((int64_t)r.tid), ts - c.base_time_ns, dur);
  if (r.kind == KTJ_RT_KERNEL)
    left = left || left_by_three(r.u.kernel.grid[0], r.u.kernel.grid[1], r.u.kernel.grid[2]) ||
           left_by_three(r.u.kernel.workgroup[0], r.u.kernel.workgroup[1], r.u.kernel.workgroup[2]);
  else if (r.kind == KTJ_RT_COPY) {
    const int32_t kind = (int32_t)r.u.copy.copy_kind;
    left = left || ((r.u.copy.src | r.u.copy.dst) >> 60) != 0 || r.u.copy.size >= KTJ_ELEVEN_DIGITS || kind < -999 || kind > 9999;
  } else if (r.kind == KTJ_RT_MALLOC) left = left || (r.u.malloc_.ptr >> 60) != 0;
  return left;
}
KTJ_HD KTJ_FI inline bool left_device(const ktj_device_rec& d, int64_t ts, int64_t dur, int64_t res, const EmitCtx& c) {
  const uint32_t domain = device_row_domain(d.domain);
  const bool memset_row = domain == KTJ_DOM_MEMSET;
  return (memset_row && (c.create_flags & KTJ_CREATE_CUDA12_ARGS)) || (!memset_row && d.queue >= KTJ_ELEVEN_DIGITS) ||
         (domain == KTJ_DOM_KERNEL_DISPATCH && d.name_id == KTJ_NONE) || d.id >= KTJ_ELEVEN_DIGITS ||
         left_by_track((int64_t)d.device, res, ts - c.base_time_ns, dur);
}

/* ---- numbers as text ---- */
KTJ_HD KTJ_FI inline uint64_t hex8(uint32_t v) { /* eight hexadecimal digits, most significant first */
  uint64_t x = v;                                     /* one digit per byte, most significant in the lowest byte */
  x = ((x & 0xFFFF0000ull) >> 16) | ((x & 0xFFFFull) << 32);
  x = ((x & 0x0000FF000000FF00ull) >> 8) | ((x & 0x000000FF000000FFull) << 16);
  x = ((x & 0x00F000F000F000F0ull) >> 4) | ((x & 0x000F000F000F000Full) << 8);
  const uint64_t letter = ((x + 0x0606060606060606ull) >> 4) & 0x0101010101010101ull;
  return x + 0x3030303030303030ull + letter * 0x27u;
}
/* the last n characters of an eight-character word (n <= 8, 0 gives nothing) */
KTJ_HD KTJ_FI inline uint64_t last_chars(uint64_t a, uint32_t n) { return n ? a >> (8u * (8u - n)) : 0; }
/* up to fifteen characters (while it is being made the count may say more: what is in it does not count then) */
struct Text { uint64_t lo, hi; uint32_t n; };
KTJ_HD KTJ_FI inline Text text_of(uint64_t v) {
  Text t;
  t.hi = 0;
  if (__builtin_expect(v < 100000000u, 1)) {
    const uint64_t a = ascii8((uint32_t)v);
    t.n = 8u - leading_zero_chars(a);
    t.lo = last_chars(a, t.n);
  } else {
    const uint64_t q = v / 100000000u, l = ascii8((uint32_t)(v - q * 100000000u));
    const uint64_t a = ascii8((uint32_t)(q < 100000000u ? q : 99999999u));
    const uint32_t n = 8u - leading_zero_chars(a); /* 1..8 */
    t.lo = n == 8u ? a : last_chars(a, n) | (l << (8u * n));
    t.hi = n == 8u ? l : l >> (64u - 8u * n);
    t.n = 8u + n;
  }
  return t;
}
KTJ_HD KTJ_FI inline Text hex_text_of(uint64_t v) {
  Text t;
  const uint64_t l = hex8((uint32_t)v);
  if ((v >> 32) == 0) { t.n = 8u - leading_zero_chars(l); t.lo = last_chars(l, t.n); t.hi = 0; return t; }
  uint64_t a = hex8((uint32_t)(v >> 32));
  const uint32_t n = 8u - leading_zero_chars(a);
  a = last_chars(a, n);
  t.lo = n == 8u ? a : a | (l << (8u * n));
  t.hi = n == 8u ? l : l >> (64u - 8u * n);
  t.n = 8u + n;
  return t;
}
KTJ_HD KTJ_FI inline void minus(Text& t) { t.hi = (t.hi << 8) | (t.lo >> 56); t.lo = (t.lo << 8) | (uint64_t)'-'; ++t.n; }
KTJ_HD KTJ_FI inline Text signed_text_of(int64_t v) {
  Text t = text_of(v < 0 ? 0ull - (uint64_t)v : (uint64_t)v);
  if (v < 0) minus(t);
  return t;
}
/* n (1..8) more characters */
KTJ_HD KTJ_FI inline void append(Text& t, uint64_t x, uint32_t n) {
  const uint32_t s = (t.n & 7u) * 8u;
  const uint64_t a = x << s, b = (x >> 1) >> (63u - s);
  if (t.n < 8u) { t.lo |= a; t.hi |= b; } else t.hi |= a;
  t.n += n;
}
/* ", " and a number below 10^6 (a larger one: too many characters for any slot) */
KTJ_HD KTJ_FI inline void append_next(Text& t, uint64_t v) {
  if (t.n > 15u || v >= 1000000u) { t.n = 16u; return; }
  uint64_t a;
  uint32_t n;
  if (v < 10000u) {
    const uint32_t x = ascii4((uint32_t)v), z = v >= 1000u ? 0u : v >= 100u ? 1u : v >= 10u ? 2u : 3u;
    a = x >> (8u * z);
    n = 4u - z;
  } else { a = ascii8((uint32_t)v); n = 8u - leading_zero_chars(a); a = last_chars(a, n); }
  append(t, (a << 16) | 0x202Cu, n + 2u);
}
KTJ_HD KTJ_FI inline Text three_text_of(uint64_t a, uint64_t b, uint64_t c) {
  Text t = text_of(a);
  append_next(t, b);
  append_next(t, c);
  return t;
}
KTJ_HD KTJ_FI inline Text time_text_of(int64_t ns) { /* put_ts */
  uint64_t us;
  if (((uint64_t)ns >> 35) == 0) us = (uint32_t)((uint64_t)ns >> 3) / 125u; else us = (uint64_t)ns / 1000u;
  Text t = text_of(us);
  append(t, (ascii4((uint32_t)ns - (uint32_t)us * 1000u) & 0xFFFFFF00u) | (uint32_t)'.', 4);
  return t;
}
/* what stands behind a lead: always fifteen characters */
KTJ_HD KTJ_FI inline Text time_text_behind(uint64_t us, uint32_t ns) {
  const uint32_t high8 = (uint32_t)(us / 1000u);
  Text t;
  t.lo = ascii8(high8);
  t.hi = (uint64_t)((ascii4((uint32_t)us - high8 * 1000u) >> 8) | ((uint32_t)'.' << 24)) | ((uint64_t)(ascii4(ns) >> 8) << 32);
  t.n = 15u;
  return t;
}
/* up to 24 characters, zeros behind them */
struct LongText {
  uint64_t w[3]; uint32_t n;
  KTJ_HD KTJ_FI void up(uint32_t k) { /* k characters further on */
    const uint32_t s = (k & 7u) * 8u;
    if (k >= 16u) { w[2] = w[0]; w[1] = w[0] = 0; }
    else if (k >= 8u) { w[2] = w[1]; w[1] = w[0]; w[0] = 0; }
    w[2] = (w[2] << s) | ((w[1] >> 1) >> (63u - s));
    w[1] = (w[1] << s) | ((w[0] >> 1) >> (63u - s));
    w[0] <<= s;
  }
  KTJ_HD KTJ_FI void down(uint32_t k) {
    const uint32_t s = (k & 7u) * 8u;
    if (k >= 16u) { w[0] = w[2]; w[1] = w[2] = 0; }
    else if (k >= 8u) { w[0] = w[1]; w[1] = w[2]; w[2] = 0; }
    w[0] = (w[0] >> s) | ((w[1] << 1) << (63u - s));
    w[1] = (w[1] >> s) | ((w[2] << 1) << (63u - s));
    w[2] >>= s;
  }
  KTJ_HD KTJ_FI void add(const LongText& o) { w[0] |= o.w[0]; w[1] |= o.w[1]; w[2] |= o.w[2]; }
  /* the first k characters only */
  KTJ_HD KTJ_FI void keep(uint32_t k) {
    const uint64_t part = (1ull << ((k & 7u) * 8u)) - 1u;
    w[0] &= k >= 8u ? ~0ull : part;
    w[1] &= k >= 16u ? ~0ull : k >= 8u ? part : 0u;
    w[2] &= k >= 24u ? ~0ull : k >= 16u ? part : 0u;
  }
  KTJ_HD KTJ_FI void put(uint64_t x, uint32_t k) { /* up to eight more, behind the last */
    LongText t;
    t.w[0] = x; t.w[1] = t.w[2] = 0;
    t.up(n);
    add(t);
    n += k;
  }
};
/* A double as put_f64 prints it, with shifts of the whole text where that takes a turn per character (a size pass over
 * 5 million of them 0.54 -> 0.47 ms). */
KTJ_HD KTJ_FI inline LongText real_text(uint64_t bits) {
  LongText t;
  t.w[0] = t.w[1] = t.w[2] = 0; t.n = 0;
  const bool neg = (bits >> 63) != 0;
  const uint64_t mag = bits & 0x7FFFFFFFFFFFFFFFull;
  if (mag >= 0x7FF0000000000000ull || mag == 0) {
    if (mag == 0) { t.w[0] = neg ? 0x302Dull : 0x30ull; t.n = neg ? 2u : 1u; return t; }
    const uint64_t word = mag > 0x7FF0000000000000ull ? 0x226E616Eull : 0x22666E69ull; /* nan", inf" */
    t.w[0] = neg ? (word << 16) | 0x2D22ull : (word << 8) | 0x22ull;
    t.n = neg ? 6u : 5u;
    return t;
  }
  uint64_t sig;
  int32_t k;
  shortest_decimal(mag, &sig, &k);
  const uint32_t nd = (uint32_t)ndigits_u64(sig);
  const int E = k + (int)nd - 1;
  {
    const uint64_t top = sig / 10000000000000000ull, rest = sig - top * 10000000000000000ull, mid = rest / 100000000ull;
    t.w[0] = ascii8((uint32_t)top); t.w[1] = ascii8((uint32_t)mid); t.w[2] = ascii8((uint32_t)(rest - mid * 100000000ull));
  }
  t.down(24u - nd);
  t.n = nd;
  if (E < 0 && E >= -4) { /* 0.000ddd */
    const uint32_t z = (uint32_t)(1 - E); /* "0." and zeros */
    t.up(z);
    t.w[0] |= 0x3030302E30ull & ((1ull << (8u * z)) - 1u);
    t.n += z;
  } else {
    const bool plain = E >= 0 && E < 16;
    const uint32_t whole = plain ? (uint32_t)E + 1u : 1u; /* digits in front of the point */
    if (nd > whole) {
      LongText behind = t;
      t.keep(whole);
      behind.down(whole);
      behind.up(whole + 1u);
      t.add(behind);
      LongText point;
      point.w[0] = '.'; point.w[1] = point.w[2] = 0;
      point.up(whole);
      t.add(point);
      t.n = nd + 1u;
    } else if (plain) { /* zeros in front of it */
      LongText zeros;
      zeros.w[0] = zeros.w[1] = zeros.w[2] = 0x3030303030303030ull;
      zeros.keep(whole);
      LongText digits = zeros;
      digits.keep(nd);
      zeros.w[0] ^= digits.w[0]; zeros.w[1] ^= digits.w[1]; zeros.w[2] ^= digits.w[2];
      t.add(zeros);
      t.n = whole;
    }
    if (!plain) {
      const uint32_t a = (uint32_t)(E < 0 ? -E : E), hundreds = a / 100u, tens = (a - hundreds * 100u) / 10u, ones = a - hundreds * 100u - tens * 10u;
      const uint64_t two = (uint64_t)('0' + tens) | ((uint64_t)('0' + ones) << 8);
      t.put((uint64_t)'e' | ((uint64_t)(E < 0 ? '-' : '+') << 8) | ((hundreds ? (two << 8) | ('0' + hundreds) : two) << 16), hundreds ? 5u : 4u);
    }
  }
  if (neg) { t.up(1); t.w[0] |= '-'; ++t.n; }
  return t;
}

/* ---- a joined row as text, its length and its tail kind (see tail_kind): false, and nothing that counts in *r, for the rows
 * that only format_activity prints.  *r is where the row waits to be stored, in LDS on the device, block b at b ^ turn (rows of
 * neighbouring lanes are a line apart): nothing of it is held in registers.  wide[wide_at]: this row's, if there are any. ---- */
KTJ_HD KTJ_FI inline bool text_row(const MatRow& m, const EmitCtx& c, const SchemaPlan* schemas, TextRow* r, uint32_t turn, WideText* wide, uint32_t wide_at, uint32_t* len,
                                     uint32_t* tail) {
  const uint32_t meta = m.meta, type = meta & KTJ_M_TYPE_MASK;
  const uint32_t cls = (meta & KTJ_M_CLASS_MASK) >> KTJ_M_CLASS_SHIFT, kind = (meta & KTJ_M_KIND_MASK) >> KTJ_M_KIND_SHIFT;
  const bool device = cls == KTJ_CLASS_DEVICE, generic = cls == KTJ_CLASS_GENERIC, flow = (meta & KTJ_M_FLOW) != 0;
  /* tracks as the row has room for; events that are not complete ones, Stream Sync rows, GPU annotations with a flow event (its
   * time is another), collective arguments */
  if (((uint64_t)m.dev >> KTJ_TR_DEV_BITS) != 0) return false;
  const uint64_t tid = (uint64_t)sanitize_tid(m.res);
  if ((tid >> 47) != 0 || (device && m.res < 0)) return false;
  if (type >= 29u || (generic && (type == KTJ_TYPE_CPU_INSTANT_EVENT || is_counter_type(type)))) return false;
  if ((meta & KTJ_M_SYNC) || (type == KTJ_TYPE_GPU_USER_ANNOTATION && flow) || collective_of(m) != 0) return false;
  bool fits = true, a_long = false;
  auto block = [&](uint32_t slot) KTJ_FI { return r->w[KTJ_TR_BLOCK(slot) ^ turn]; };
  typedef uint64_t __attribute__((may_alias)) word_pair;
  auto two = [](uint32_t* w, uint64_t x) KTJ_FI { *reinterpret_cast<word_pair*>(w) = x; }; /* (eight-byte aligned) */
  auto put = [&](uint32_t slot, const Text& t) KTJ_FI {
    uint32_t* const w = block(slot);
    const uint32_t most = slot == S_A || slot >= S_Z ? 11u : 15u;
    fits = fits && t.n <= most;
    if (slot == S_A) {
      two(w, (t.lo & 0xFFFFFFFFFFFFFFull) | ((uint64_t)t.n << 56));
      a_long = t.n > KTJ_TR_A_NEAR;
      if (a_long) block(S_DUR)[3] = (uint32_t)(t.lo >> 56) | ((uint32_t)t.hi << 8);
    } else {
      two(w, t.lo);
      if (slot >= S_Z) w[2] = (uint32_t)t.hi | (t.n << 24);
      else two(w + 2, t.hi | ((uint64_t)t.n << 56));
    }
    return t.n;
  };
  auto string = [&](uint32_t id, bool is_name, uint32_t* n) KTJ_FI {
    if (id >= c.dict.n) { *n = 0; return 0u; }
#if defined(__HIP_DEVICE_COMPILE__)
    const DictEntry e = c.dict.entries[id];
    *n = is_name ? e.name_len : e.arg_len;
    return (uint32_t)((is_name ? e.name_off : e.arg_off) >> 4);
#else
    *n = (uint32_t)(is_name ? c.dict.name_off[id + 1] - c.dict.name_off[id] : c.dict.arg_off[id + 1] - c.dict.arg_off[id]);
    return id;
#endif
  };
  auto real = [&](uint64_t bits, bool here) KTJ_FI { /* a double */
    const LongText t = real_text(bits);
    if (here) {
      two(block(S_Y), t.w[0]); two(block(S_Y) + 2, t.w[1]);
      two(block(S_Z), t.w[2]); block(S_Z)[2] = 0;
    } else {
      wide[wide_at].w[0] = t.w[0]; wide[wide_at].w[1] = t.w[1]; wide[wide_at].w[2] = t.w[2]; wide[wide_at].w[3] = 0;
    }
    return t.n;
  };
  block(S_Y)[3] = 0; /* (its last byte is not KTJ_ROW_LEFT) */
  uint32_t n = 0; /* the length, but for the strings */
  /* the name */
  uint32_t name = KTJ_TR_NAME_RUN, name_len = 0, at_name = 0, len1 = 0, at_more = 0, between = 0, args = KTJ_TR_NO_ARGS, close = 5u;
  if (meta & KTJ_M_NAME_BUILTIN) {
    if (m.name_id <= KTJ_COPY_D2D) name = R_COPY_NAME + m.name_id;
    else if (m.name_id == KTJ_NAME_MEMSET) { const uint32_t k = (m.aux >> 8) & 0xFFu; name = R_MEMSET_NAME + (k < 8u ? k : 8u); }
    else if (m.name_id != KTJ_NAME_EMPTY) return false;
    if (name != KTJ_TR_NAME_RUN) n += chars_table.of[name];
  } else at_name = string(m.name_id, true, &name_len);
  /* the args */
  bool frag = true;
  if (generic) {
    n += chars_table.of[R_HEAD + type];
    frag = false;
    if (m.aux < c.n_schemas) {
      if (m.aux >= MAX_SCHEMAS) return false;
      const uint32_t what_plan = schemas[m.aux].what;
      if (!(what_plan & 1u) || m.p[0] + ((what_plan >> 8) & 0xFFu) > c.n_args) return false;
      frag = (what_plan & 2u) != 0;
      if (what_plan & 4u) {
        const uint32_t id = (uint32_t)c.args[m.p[0]];
        frag = id < c.dict.n && (dict_flags(c.dict, id) & KTJ_SF_ARG_BLANK) == 0;
      }
      if (frag) {
        args = KTJ_TR_SCHEMA + m.aux;
        n += schemas[m.aux].chars;
        KTJ_NOUNROLL
        for (uint32_t j = 0; j < 4; ++j) {
          const uint32_t item = schemas[m.aux].item[j], what = item & 0xFFu;
          if (what == I_NONE) continue;
          const uint64_t* a = c.args + m.p[0] + (item >> 8);
          Text t;
          if (what == I_BOOL) { t.lo = a[0] ? 0x65757274ull : 0x65736C6166ull; t.hi = 0; t.n = a[0] ? 4u : 5u; }
          else {
            const bool neg = what != I_U64 && (int64_t)a[0] < 0;
            t = text_of(neg ? 0ull - a[0] : a[0]);
            if (neg) minus(t);
          }
          if (what > I_ARRAY + 1u) append_next(t, a[1]);
          if (what > I_ARRAY + 2u) append_next(t, a[2]);
          n += put(item_slot(j), t);
        }
        between = (what_plan >> 16) & 3u;
        if (between == 1u) at_more = string((uint32_t)c.args[m.p[0] + (what_plan >> 24)], false, &len1);
        else if (between) {
          at_more = wide_at;
          len1 = real(c.args[m.p[0] + (what_plan >> 24)], between == 2u);
        }
      }
    }
    if (m.ext == 0 && !frag) close = 0u;
    if (flow) n += put(S_FLOW, signed_text_of(m.flow_id));
  } else {
    const uint32_t id_chars = put(S_FLOW, text_of((uint64_t)m.flow_id));
    n += flow ? 2u * id_chars : id_chars;
    bool triple;
    if (!device) {
      n += chars_of<R_HEAD + KTJ_TYPE_CUDA_RUNTIME>() + put(S_A, text_of(m.aux));
      triple = kind == KTJ_RT_KERNEL;
      const bool copy = kind == KTJ_RT_COPY, sized = (meta & KTJ_M_MALLOC_BYTES) != 0;
      args = copy ? A_COPY : kind == KTJ_RT_MALLOC ? (sized ? A_MALLOC_BYTES : A_MALLOC) : A_DEFAULT;
      if (triple) {
        args = A_LAUNCH;
        if (meta & KTJ_M_HAS_KERNEL_ARG) { args = A_LAUNCH_NAMED; between = 1u; at_more = string((uint32_t)m.p[4], false, &len1); }
      }
      if (copy || kind == KTJ_RT_MALLOC) {
        n += put(S_X, hex_text_of(m.p[0]));
        if (copy) {
          n += put(S_Y, hex_text_of(m.p[1]));
          const Text t = signed_text_of((int64_t)(int32_t)(uint32_t)m.p[3]);
          if (t.n > 4u) return false;
          at_more = (uint32_t)t.lo;
          n += t.n;
        }
      }
      const uint64_t p1 = m.p[1], p2 = m.p[2], p3 = m.p[3]; /* (values: a choice among places would keep m in memory) */
      if (triple || copy || args == A_MALLOC_BYTES) n += put(S_Z, text_of(triple ? p3 : copy ? p2 : p1));
    } else {
      const bool memset_row = kind == KTJ_DOM_MEMSET, size = memset_row || (meta & KTJ_M_HAS_SIZE) != 0;
      bool bandwidth = size;
      triple = !size && (meta & KTJ_M_HAS_GRID) != 0;
      n += chars_table.of[R_HEAD + type] + put(S_A, text_of(m.p[3]));
      if (memset_row) {
        if (c.create_flags & KTJ_CREATE_CUDA12_ARGS) return false;
        bandwidth = m.dur != 0;
        args = bandwidth ? A_MEMSET_BANDWIDTH : A_MEMSET;
      } else {
        const bool copied = kind == KTJ_DOM_MEMORY_COPY;
        const uint32_t direction = m.aux <= KTJ_COPY_D2D ? m.aux : 0u;
        bandwidth = size && m.dur != -1;
        if (size && !bandwidth) args = A_BYTES_ONLY + (copied ? 1u + direction : 0u);
        else args = (copied ? A_COPIED + 3u * direction : (uint32_t)A_KERNEL) + (size ? 1u : triple ? 2u : 0u);
        if (triple) close = 10u;
      }
      if (size) n += put(S_X, text_of(m.p[0]));
      if (bandwidth) {
        const double d = (double)m.p[0] / (memset_row ? (double)m.dur : (double)((uint64_t)m.dur + 1u));
        uint64_t bits; __builtin_memcpy(&bits, &d, 8);
        between = 2u; len1 = real(bits, true);
      }
    }
    n += chars_table.of[R_ARGS + args] + chars_table.of[R_ARGS2 + args];
    if (triple) {
      n += put(S_X, three_text_of((uint32_t)m.p[0], m.p[0] >> 32, (uint32_t)m.p[1])) +
           put(S_Y, three_text_of(m.p[1] >> 32, (uint32_t)m.p[2], m.p[2] >> 32));
    }
  }
  if (name_len > KTJ_WEAVE_MAX_RUN || len1 > KTJ_WEAVE_MAX_RUN) return false;
  /* the times, the External id, the track */
  const bool wider = type == KTJ_TYPE_GPU_USER_ANNOTATION;
  int64_t rel = m.ts - (wider ? 1 : 0) - c.base_time_ns;
  if (rel < 0) rel = 0;
  const uint32_t track = (uint32_t)(ndigits_u64((uint64_t)m.dev) + ndigits_u64(tid));
  uint32_t lead = 0;
  {
    uint32_t k;
    if ((uint64_t)rel < KTJ_LEAD_UNIT * 1000u) k = put(S_TS, time_text_of(rel));
    else {
      const uint64_t us = (uint64_t)rel / 1000u, all = us / KTJ_LEAD_UNIT;
      lead = (uint32_t)all;
      const uint32_t chars = (uint32_t)ndigits_u64(lead);
      if (all > 0xFFFFu || track + chars > TRACK_ROOM) return false;
      k = put(S_TS, time_text_behind(us - all * KTJ_LEAD_UNIT, (uint32_t)rel - (uint32_t)us * 1000u)) + chars;
    }
    n += flow ? 2u * k : k;
  }
  n += put(S_DUR, time_text_of((m.dur < 0 ? 0 : m.dur) + (wider ? 2 : 0)));
  uint32_t body = 0;
  if (m.ext != 0) {
    Text t = signed_text_of(m.ext);
    if (frag) append(t, ',', 1);
    n += chars_of<R_BODY_EXT>() + put(S_EXT, t);
    body = 2u;
  } else {
    n += frag ? chars_of<R_BODY_ARGS>() : chars_of<R_BODY_NONE>();
    body = frag ? 1u : 0u;
  }
  n += track * (1u + (device ? 1u : 0u) + (flow ? 1u : 0u));
  const uint32_t last = close + (flow ? (meta & KTJ_M_FLOW_START ? 1u : 2u) + (meta & KTJ_M_FLOW_FWDBWD ? 2u : 0u) : 0u);
  n += chars_table.of[R_TAIL + last];
  block(S_Z)[3] = type | (name << 5) | (body << 12) | (args << 14) | (last << 21) | (between << 25) | ((uint32_t)(tid >> 42) << 27);
  block(S_EXT)[3] = at_name;
  block(S_FLOW)[3] = name_len | (len1 << 16);
  if (lead) {
    block(S_FLOW)[3] = name_len | (len1 << 16) | KTJ_TR_HAS_LEAD;
    for (uint32_t k = 0; k < 4u; ++k) { uint32_t* const w = &block(S_Z + k)[2]; *w = (*w & 0x0FFFFFFFu) | ((lead >> (4u * k)) << 28); }
  }
  if (!a_long) block(S_DUR)[3] = at_more;
  else fits = fits && (between & 1u) == 0 && args != A_COPY; /* (nothing else is there) */
  two(block(S_A) + 2, (uint64_t)m.dev | (tid << KTJ_TR_DEV_BITS));
  *len = n + name_len + len1;
  *tail = flow ? (meta & KTJ_M_FLOW_START ? 0u : 2u) : close ? 1u : 0u;
  return fits;
}

}  // namespace weave
}  // namespace ktj
#endif
