// Interval gather-copy (gfx950).
//
// One launch moves any number of [src, src + n) -> [dst, dst + n) intervals.  Each
// interval is cut into chunks of 64 x 16 bytes of source (256 elements of a 4-byte
// source, 512 of a 2-byte one); one workgroup owns one chunk and finds its interval by
// a binary search over the records' first_chunk column.  Inside a chunk each lane moves
// units of 16 / max(source, destination element bytes) elements, consecutive lanes
// taking consecutive units, so every load and store instruction of a wave covers one
// contiguous span.
//
// Two ways to move a chunk share that layout.  CopyAligned serves plans whose records all
// start on aligned addresses (the host certifies this): one aligned load and one aligned
// store per unit.  CopyAny serves any plan: it cuts each record's chunks on 128-byte
// lines of the destination, so that only a record's first and last chunk write part of a
// line, and reads its units where they lie with unaligned vector loads.  A load never
// touches a byte outside the source interval.
#include <algorithm>
#include <cstring>

#include "hbt_common.hpp"

namespace hbt {
namespace {

// One wavefront per workgroup reading 16 bytes of source per lane: a workgroup reads
// 1 KB and retires, the shape that streamed fastest against 512 B or 2 KB per
// workgroup and against 256-thread workgroups walking larger chunks.
constexpr int kCopyBlock = 64;
// A cache line: what a store must cover whole for the memory behind the L2 to see one write.
constexpr uint32_t kLineBytes = 128;
// Consecutive chunks that one XCD moves where the source is off the destination's lines
// (xcd_order): a shared source line in every 1 KB chunk is 6% more traffic, and in every
// eighth it is not seen.  One, 2, 4, 8 and 16 chunks: 641 M bf16 elements resharded 417, 407,
// 400, 402 and 415 us; a Llama-3-8B layer gathered to bf16 from 7 shards 228, 216, 218, 212
// and 211.  Records whose lines agree keep the dispatch order: theirs is the slower one so
// (8 shards gathered 196 us, 212 to 224 us in runs).
constexpr int kCopyRun = 8;
// Non-temporal loads and stores: every byte is moved once.
constexpr bool kCopyNT = true;

// A vector of NW dwords (NW = 2 or 4).
template <int NW>
struct Vec {
    typedef uint32_t type __attribute__((ext_vector_type(NW)));
};

// The copy kernel reads its addresses from a table in device memory, so the compiler
// cannot tell which address space they point into and would issue flat loads and
// stores.  These views name global memory (address space 1): global_load/global_store
// instructions, which wait on the vector counter alone.
typedef __attribute__((address_space(1))) uint8_t gbyte;

// Aligned vector load/store of NW dwords, non-temporal when kCopyNT: every byte is moved
// exactly once.
template <int NW>
__device__ __forceinline__ typename Vec<NW>::type ldg(const gbyte* p) {
    typedef typename Vec<NW>::type V;
    typedef __attribute__((address_space(1))) const V GV;
    if constexpr (kCopyNT) return __builtin_nontemporal_load(reinterpret_cast<GV*>(p));
    return *reinterpret_cast<GV*>(p);
}
template <int NW>
__device__ __forceinline__ void stg(gbyte* p, typename Vec<NW>::type x) {
    typedef typename Vec<NW>::type V;
    typedef __attribute__((address_space(1))) V GV;
    if constexpr (kCopyNT) {
        __builtin_nontemporal_store(x, reinterpret_cast<GV*>(p));
    } else {
        *reinterpret_cast<GV*>(p) = x;
    }
}

// NW dwords from an address on an element boundary (2 or 4 bytes): one vector load, which
// the memory pipeline splits where it crosses a line.
template <int NW>
__device__ __forceinline__ typename Vec<NW>::type ldg_any(const gbyte* p) {
    typedef typename Vec<NW>::type V __attribute__((aligned(2)));
    typedef __attribute__((address_space(1))) const V GV;
    if constexpr (kCopyNT) return __builtin_nontemporal_load(reinterpret_cast<GV*>(p));
    return *reinterpret_cast<GV*>(p);
}

// Element semantics.  SB/DB are source/destination element bytes; a 2-byte element is
// bf16, or IEEE fp16 when H is set (a conversion never mixes the two).  Same-size COPY
// is a bit copy; 4->2 narrows fp32 (round to nearest even), 2->4 widens exactly; DIVIDE
// goes through fp32 (true division) and rounds to the destination type.
template <int SB, bool H>
__device__ __forceinline__ float elem_to_f32(uint32_t bits) {
    if constexpr (SB == 4) return __uint_as_float(bits);
    return b16_to_f32<H>(bits);
}
template <int DB, bool H>
__device__ __forceinline__ uint32_t f32_to_elem(float x) {
    if constexpr (DB == 4) return __float_as_uint(x);
    return f32_to_b16<H>(x);
}
// kOpScale: HBT_COPY_OP_DIVIDE by a power of two, run as a multiply by its exact
// reciprocal (passed in place of the divisor); the bits are those of the division.
constexpr int kOpScale = 2;
template <int SB, int OP, bool H>
__device__ __forceinline__ float convert_value(uint32_t bits, float divisor) {
    float x = elem_to_f32<SB, H>(bits);
    if constexpr (OP == HBT_COPY_OP_DIVIDE) x = x / divisor;
    if constexpr (OP == kOpScale) x = x * divisor;
    return x;
}
template <int SB, int DB, int OP, bool H>
__device__ __forceinline__ uint32_t convert(uint32_t bits, float divisor) {
    if constexpr (SB == DB && OP == HBT_COPY_OP_COPY) return bits;
    return f32_to_elem<DB, H>(convert_value<SB, OP, H>(bits, divisor));
}
// Whether a copy rounds fp32 values to a 2-byte destination (a narrowing, or arithmetic on
// 2-byte elements): the vector paths then round two values per packed conversion.
template <int SB, int DB, int OP>
constexpr bool rounds_to_b16() { return DB == 2 && !(SB == 2 && OP == HBT_COPY_OP_COPY); }

template <int EB>
__device__ __forceinline__ uint32_t load_elem(const gbyte* p) {
    typedef __attribute__((address_space(1))) const uint32_t G32;
    typedef __attribute__((address_space(1))) const uint16_t G16;
    if constexpr (EB == 4) return *reinterpret_cast<G32*>(p);
    return *reinterpret_cast<G16*>(p);
}
template <int EB>
__device__ __forceinline__ void store_elem(gbyte* p, uint32_t bits) {
    typedef __attribute__((address_space(1))) uint32_t G32;
    typedef __attribute__((address_space(1))) uint16_t G16;
    if constexpr (EB == 4) {
        *reinterpret_cast<G32*>(p) = bits;
    } else {
        *reinterpret_cast<G16*>(p) = static_cast<uint16_t>(bits);
    }
}

// Elements per lane unit: one 16-byte access on the wider side of the copy.
template <int SB, int DB>
constexpr int unit_elems() { return 16 / (SB > DB ? SB : DB); }
// Elements per chunk (per workgroup): 16 bytes of source per lane, 32 when the
// destination is wider.  A widening chunk writes more than it reads, and its stores do
// not hold the workgroup, so with 1 KB of source the workgroups retired faster than
// their writes drained; same-size and narrowing copies keep 1 KB.
template <int SB, int DB>
constexpr int64_t chunk_elems() { return int64_t(kCopyBlock) * 16 / SB * (SB < DB ? 2 : 1); }

// Unpack the U elements held in `words` (SB bytes each) into element bit patterns.
template <int SB, int U>
__device__ __forceinline__ void unpack_unit(const uint32_t (&words)[U * SB / 4], uint32_t (&e)[U]) {
    if constexpr (SB == 4) {
#pragma unroll
        for (int i = 0; i < U; ++i) e[i] = words[i];
    } else {
#pragma unroll
        for (int i = 0; i < U / 2; ++i) {
            e[2 * i] = words[i] & 0xFFFFu;
            e[2 * i + 1] = words[i] >> 16;
        }
    }
}
template <int DB, int U>
__device__ __forceinline__ void pack_unit_store(gbyte* d, const uint32_t (&e)[U]) {
    constexpr int NW = U * DB / 4;
    typename Vec<NW>::type x;
    if constexpr (DB == 4) {
#pragma unroll
        for (int i = 0; i < U; ++i) x[i] = e[i];
    } else {
#pragma unroll
        for (int i = 0; i < U / 2; ++i) x[i] = e[2 * i] | (e[2 * i + 1] << 16);
    }
    stg<NW>(d, x);
}

// Converts one unit as loaded and stores it.
template <int SB, int DB, int OP, bool H>
__device__ __forceinline__ void store_unit(gbyte* d, const typename Vec<unit_elems<SB, DB>() * SB / 4>::type& x,
                                           float divisor) {
    constexpr int U = unit_elems<SB, DB>();
    constexpr int kSrcWords = U * SB / 4;
    uint32_t words[kSrcWords];
#pragma unroll
    for (int i = 0; i < kSrcWords; ++i) words[i] = x[i];
    uint32_t e[U];
    unpack_unit<SB, U>(words, e);
    if constexpr (rounds_to_b16<SB, DB, OP>()) {
        // Two values per packed conversion, each the bits f32_to_b16 gives.
        float f[U];
#pragma unroll
        for (int i = 0; i < U; ++i) f[i] = convert_value<SB, OP, H>(e[i], divisor);
        uint32_t w[U / 2];
        pack_rounded<H ? HBT_DTYPE_F16 : HBT_DTYPE_BF16, U / 2>(f, w);
        typename Vec<U / 2>::type o;
#pragma unroll
        for (int i = 0; i < U / 2; ++i) o[i] = w[i];
        stg<U / 2>(d, o);
    } else {
#pragma unroll
        for (int i = 0; i < U; ++i) e[i] = convert<SB, DB, OP, H>(e[i], divisor);
        pack_unit_store<DB, U>(d, e);
    }
}

// The interval a chunk belongs to.
struct Record {
    int64_t src;  // 0: write zeros
    int64_t dst;
    int64_t n;
    int64_t first;  // its first chunk
};

// The record that owns `chunk`: the last one whose first_chunk <= chunk (records with no
// chunks are dropped by the host, so first_chunk strictly increases).  The search runs on
// the scalar unit: its loads hit the scalar cache and do not queue behind the vector
// traffic of the waves in flight (a wave-wide search over vector loads waits behind that
// traffic and was slower).  With hints (the table followed by hints[j] = the record owning
// chunk j * kHintStride) the search starts at the hinted record and steps forward, at most
// as many records as start inside one hint stride; without them it bisects the whole
// table, log2(count) dependent loads before the workgroup's first data load.
constexpr int kHintShift = 8;  // one hint per 256 chunks
__device__ __forceinline__ Record owning_record(const int64_t* __restrict__ table, int64_t count,
                                                int64_t chunk, const int64_t* __restrict__ hints) {
    int64_t lo = 0;
    if (hints != nullptr) {
        lo = hints[chunk >> kHintShift];
        lo = lo < 0 ? 0 : (lo < count ? lo : count - 1);  // a wrong hint stays inside the table
        while (lo + 1 < count && table[4 * (lo + 1) + 3] <= chunk) ++lo;
    } else {
        int64_t hi = count - 1;
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) >> 1;
            if (table[4 * mid + 3] <= chunk) {
                lo = mid;
            } else {
                hi = mid - 1;
            }
        }
    }
    const int64_t* rec = table + 4 * lo;
    return Record{rec[0], rec[1], rec[2], rec[3]};
}

// A plan of up to kRows records in the launch's own arguments, with a hint for every 2^shift
// chunks (kRowHints of them cover the plan), four to a word: the record that owns the first
// of them.  A plan built for one use, such as an unpack into fresh tensors, then needs no
// table built in pinned memory and uploaded ahead of the launch: 52 GPT-2 tensors rebuilt from
// 5 ragged shards (542 MB, 101 us of kernel) took 406 us a call with the table and took 115 us
// without, the rows counted by arithmetic; a Llama-3-8B layer gathered from 8 shards 199 and
// 197 us.  HBT_COPY_MAX_ROWS records are 3.9 KB, inside the 4 KB a launch's arguments may take;
// the host writes them at every launch, so a plan of at most kFewRows records takes 0.8 KB:
// the call 3.1 us in place of 4.5, where one over a device table takes 3.2.
constexpr int kFewRows = 16;
constexpr int kRowHints = 256;
constexpr uint32_t kHintSplit = 128;  // set when another record starts among the hint's chunks
template <int kRows>
struct RowTable {
    Record rec[kRows];
    uint32_t hint[kRowHints / 4];
    int32_t count;
    int32_t shift;
};
static_assert(HBT_COPY_MAX_ROWS <= kHintSplit, "a hint is one byte: a record and the split bit");
static_assert(sizeof(RowTable<HBT_COPY_MAX_ROWS>) + 32 <= 4096, "the arguments of a launch");
template <int kRows>
__device__ __forceinline__ Record owning_record(const RowTable<kRows>& rows, int64_t chunk) {
    const uint32_t j = static_cast<uint32_t>(chunk >> rows.shift);
    const uint32_t hint = (rows.hint[j >> 2] >> (8 * (j & 3u))) & 0xFFu;
    int r = static_cast<int>(hint & (kHintSplit - 1u));
    if ((hint & kHintSplit) != 0) {
        while (r + 1 < rows.count && rows.rec[r + 1].first <= chunk) ++r;
    }
    return rows.rec[r];  // one indexed read: a Record copied on two paths moves the table to scratch
}

// Any plan.  A record's chunk c covers elements [line + c * kChunk, line + (c + 1) * kChunk)
// of it, `line` being the elements before its destination's first 128-byte line (chunk 0
// takes those too), cut at the record's end: the same number of chunks as the table counts,
// the last of them possibly empty.  Every chunk but a record's first and last then writes
// whole lines, where chunks counted from the record's start write two partial lines each,
// shared between two XCDs' L2 caches.  Units are read by one unaligned vector load each, where two
// aligned loads and a shift read every line twice.  1 GiB moved between misaligned
// addresses, GB/s (read + written), chunks from the record's start with two loads, then
// this: source 2 bytes off 5,160 and 6,240; destination 2 off 4,600 and 6,210; both
// 4,590 and 6,250; destination 16 off 5,850 and 6,230.
template <int SB, int DB, int OP, bool H>
struct CopyAny {
    typedef float Divisor;
    static __device__ __forceinline__ void run(const Record& rec, int64_t c, float divisor);
};
template <int SB, int DB, int OP, bool H>
__device__ __forceinline__ void CopyAny<SB, DB, OP, H>::run(const Record& rec, int64_t c, float divisor) {
    static_assert(kCopyBlock == 64, "a workgroup is one wave; its chunk is whole wave-wide spans of 16-byte source loads");
    const gbyte* src = reinterpret_cast<const gbyte*>(static_cast<uintptr_t>(rec.src));
    gbyte* dst = reinterpret_cast<gbyte*>(static_cast<uintptr_t>(rec.dst));
    const int64_t n = rec.n;
    constexpr int64_t kChunk = chunk_elems<SB, DB>();
    constexpr int U = unit_elems<SB, DB>();
    constexpr int kSrcWords = U * SB / 4;
    constexpr int kPerLane = static_cast<int>(kChunk / U / kCopyBlock);
    static_assert(kChunk == int64_t(kPerLane) * kCopyBlock * U, "a chunk is whole units on every lane");
    static_assert(kLineBytes / DB <= kCopyBlock, "one lane per element of a head");

    const int64_t line = ((kLineBytes - (static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst)) & (kLineBytes - 1u))) &
                          (kLineBytes - 1u)) / DB;
    // The source of the first whole line starts off a line, so every chunk's does.  Widening
    // chunks read 2 KB for the 4 KB they write, and the order those leave in counts for more: a
    // 275 M-element bf16 to fp32 reshard 291 us in runs and 281 us without.
    if (SB >= DB && src != nullptr && ((reinterpret_cast<uintptr_t>(src) + line * SB) & (kLineBytes - 1u)) != 0)
        c = xcd_order<kCopyRun>(c, (n + kChunk - 1) / kChunk);
    const int64_t e0 = c == 0 ? 0 : line + c * kChunk;
    const int64_t past = line + (c + 1) * kChunk;
    const int64_t len = (past < n ? past : n) - e0;
    if (len <= 0) return;
    gbyte* d = dst + e0 * DB;
    const gbyte* s = src != nullptr ? src + e0 * SB : nullptr;

    // Elements before the first line (chunk 0) and after the last whole unit, one per lane.
    int64_t head = c == 0 ? line : 0;
    if (head > len) head = len;
    const int64_t units = (len - head) / U;
    const int64_t tail_begin = head + units * U;
    if (threadIdx.x < head) {
        const int64_t e = threadIdx.x;
        const uint32_t bits = s != nullptr ? convert<SB, DB, OP, H>(load_elem<SB>(s + e * SB), divisor) : 0u;
        store_elem<DB>(d + e * DB, bits);
    }
    if (threadIdx.x < len - tail_begin) {
        const int64_t e = tail_begin + threadIdx.x;
        const uint32_t bits = s != nullptr ? convert<SB, DB, OP, H>(load_elem<SB>(s + e * SB), divisor) : 0u;
        store_elem<DB>(d + e * DB, bits);
    }

    // Units per lane: kPerLane (4 for bf16 -> fp32, else 1).  Every unit's loads are
    // issued before the first store, so a workgroup pays one memory round trip.
    gbyte* dbody = d + head * DB;
    if (s == nullptr) {
        uint32_t zero[U];
#pragma unroll
        for (int i = 0; i < U; ++i) zero[i] = 0u;
#pragma unroll
        for (int j = 0; j < kPerLane; ++j) {
            const int64_t u = threadIdx.x + j * kCopyBlock;
            if (u < units) pack_unit_store<DB, U>(dbody + u * U * DB, zero);
        }
        return;
    }
    const gbyte* sbody = s + head * SB;
    typename Vec<kSrcWords>::type x[kPerLane];
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) {
        const int64_t u = threadIdx.x + j * kCopyBlock;
        if (u < units) x[j] = ldg_any<kSrcWords>(sbody + u * U * SB);
    }
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) {
        const int64_t u = threadIdx.x + j * kCopyBlock;
        if (u < units) store_unit<SB, DB, OP, H>(dbody + u * U * DB, x[j], divisor);
    }
}

// Aligned-record copy: every record's destination is 16-byte aligned and its source is
// aligned to the unit's source width (the host certifies this for the whole plan), so a
// lane moves its unit with one aligned load and one aligned store.  A chunk's units past
// the record's end are masked off; a record whose length is not a whole number of units
// finishes with an element loop in its last chunk.
template <int SB, int DB, int OP, bool H>
struct CopyAligned {
    typedef float Divisor;
    static __device__ __forceinline__ void run(const Record& rec, int64_t c, float divisor);
};
template <int SB, int DB, int OP, bool H>
__device__ __forceinline__ void CopyAligned<SB, DB, OP, H>::run(const Record& rec, int64_t c, float divisor) {
    constexpr int U = unit_elems<SB, DB>();
    constexpr int kSrcWords = U * SB / 4;
    constexpr int64_t kChunk = chunk_elems<SB, DB>();
    constexpr int kPerLane = static_cast<int>(kChunk / U / kCopyBlock);
    static_assert(kChunk == int64_t(kPerLane) * kCopyBlock * U, "a chunk is whole units on every lane");
    const int64_t e0 = c * kChunk;
    const int64_t n = rec.n;
    const int64_t len = (n - e0) < kChunk ? (n - e0) : kChunk;
    const int64_t units = len / U;
    const gbyte* s = reinterpret_cast<const gbyte*>(static_cast<uintptr_t>(rec.src));
    gbyte* d = reinterpret_cast<gbyte*>(static_cast<uintptr_t>(rec.dst)) + e0 * DB;
    if (s == nullptr) {
        uint32_t zero[U];
#pragma unroll
        for (int i = 0; i < U; ++i) zero[i] = 0u;
#pragma unroll
        for (int j = 0; j < kPerLane; ++j) {
            const int64_t u = threadIdx.x + j * kCopyBlock;
            if (u < units) pack_unit_store<DB, U>(d + u * U * DB, zero);
        }
        if (threadIdx.x < len - units * U) store_elem<DB>(d + (units * U + threadIdx.x) * DB, 0u);
        return;
    }
    s += e0 * SB;
    typename Vec<kSrcWords>::type x[kPerLane];
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) {
        const int64_t u = threadIdx.x + j * kCopyBlock;
        if (u < units) x[j] = ldg<kSrcWords>(s + u * U * SB);
    }
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) {
        const int64_t u = threadIdx.x + j * kCopyBlock;
        if (u < units) store_unit<SB, DB, OP, H>(d + u * U * DB, x[j], divisor);
    }
    if (threadIdx.x < len - units * U) {
        const int64_t e = units * U + threadIdx.x;
        store_elem<DB>(d + e * DB, convert<SB, DB, OP, H>(load_elem<SB>(s + e * SB), divisor));
    }
}

// ---- conversions through double ---------------------------------------------------------
// The dtype pairs the kernels above do not move: float64 to or from another dtype, float64
// divided by the AVG divisor (the pre-divide of float64 DDP buckets), and bf16 <-> fp16.
// Each value widens exactly to double and narrows as torch's Tensor.to does: kept for a
// float64 destination, else to fp32 with one rounding to nearest even, then, for a 2-byte
// destination, to that dtype (double -> fp32 -> bf16/fp16, as c10's conversions go;
// bf16 <-> fp16 through the exact fp32 value).  DIVIDE divides the double by the divisor,
// correctly rounded, as torch's div_ on a float64 tensor does; a power-of-two divisor runs
// as a multiply by its exact reciprocal (kOpScale), with the same bits.  A chunk is 1 KB
// of source, as in the kernels above.
template <int D>
constexpr int elem_bytes() { return D == HBT_DTYPE_F64 ? 8 : (D == HBT_DTYPE_F32 ? 4 : 2); }

template <int D>
__device__ __forceinline__ double widen_elem(const gbyte* p) {
    typedef __attribute__((address_space(1))) const double G64;
    if constexpr (D == HBT_DTYPE_F64) return *reinterpret_cast<G64*>(p);
    else if constexpr (D == HBT_DTYPE_F32) return static_cast<double>(__uint_as_float(load_elem<4>(p)));
    else return static_cast<double>(b16_to_f32<D == HBT_DTYPE_F16>(load_elem<2>(p)));
}
template <int D>
__device__ __forceinline__ void narrow_store(gbyte* p, double x) {
    typedef __attribute__((address_space(1))) double G64;
    if constexpr (D == HBT_DTYPE_F64) {
        *reinterpret_cast<G64*>(p) = x;
    } else if constexpr (D == HBT_DTYPE_F32) {
        store_elem<4>(p, __float_as_uint(static_cast<float>(x)));
    } else {
        store_elem<2>(p, f32_to_b16<D == HBT_DTYPE_F16>(static_cast<float>(x)));
    }
}
template <int OP>
__device__ __forceinline__ double apply_op(double x, double divisor) {
    if constexpr (OP == HBT_COPY_OP_DIVIDE) return x / divisor;
    if constexpr (OP == kOpScale) return x * divisor;
    return x;
}

// NW dwords at p (4 * NW bytes, aligned to that), non-temporal when kCopyNT.
template <int NW>
__device__ __forceinline__ void load_words(const gbyte* p, uint32_t (&w)[NW]) {
    if constexpr (NW == 1) {
        typedef __attribute__((address_space(1))) const uint32_t G32;
        if constexpr (kCopyNT) w[0] = __builtin_nontemporal_load(reinterpret_cast<G32*>(p));
        else w[0] = *reinterpret_cast<G32*>(p);
    } else {
        const typename Vec<NW>::type v = ldg<NW>(p);
#pragma unroll
        for (int i = 0; i < NW; ++i) w[i] = v[i];
    }
}
template <int NW>
__device__ __forceinline__ void store_words(gbyte* p, const uint32_t (&w)[NW]) {
    if constexpr (NW == 1) {
        typedef __attribute__((address_space(1))) uint32_t G32;
        if constexpr (kCopyNT) __builtin_nontemporal_store(w[0], reinterpret_cast<G32*>(p));
        else *reinterpret_cast<G32*>(p) = w[0];
    } else {
        typename Vec<NW>::type v;
#pragma unroll
        for (int i = 0; i < NW; ++i) v[i] = w[i];
        stg<NW>(p, v);
    }
}
// U elements of dtype D held in dwords, to and from their double values (widening exact,
// narrowing as narrow_store narrows).
template <int D, int U>
__device__ __forceinline__ void words_to_f64(const uint32_t (&w)[U * elem_bytes<D>() / 4], double (&x)[U]) {
    if constexpr (D == HBT_DTYPE_F64) {
#pragma unroll
        for (int i = 0; i < U; ++i) x[i] = __hiloint2double(static_cast<int>(w[2 * i + 1]), static_cast<int>(w[2 * i]));
    } else if constexpr (D == HBT_DTYPE_F32) {
#pragma unroll
        for (int i = 0; i < U; ++i) x[i] = static_cast<double>(__uint_as_float(w[i]));
    } else {
#pragma unroll
        for (int i = 0; i < U / 2; ++i) {
            x[2 * i] = static_cast<double>(b16_to_f32<D == HBT_DTYPE_F16>(w[i] & 0xFFFFu));
            x[2 * i + 1] = static_cast<double>(b16_to_f32<D == HBT_DTYPE_F16>(w[i] >> 16));
        }
    }
}
template <int D, int U>
__device__ __forceinline__ void f64_to_words(const double (&x)[U], uint32_t (&w)[U * elem_bytes<D>() / 4]) {
    if constexpr (D == HBT_DTYPE_F64) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            w[2 * i] = static_cast<uint32_t>(__double2loint(x[i]));
            w[2 * i + 1] = static_cast<uint32_t>(__double2hiint(x[i]));
        }
    } else if constexpr (D == HBT_DTYPE_F32) {
#pragma unroll
        for (int i = 0; i < U; ++i) w[i] = __float_as_uint(static_cast<float>(x[i]));
    } else {
#pragma unroll
        for (int i = 0; i < U / 2; ++i)
            w[i] = f32_to_b16<D == HBT_DTYPE_F16>(static_cast<float>(x[2 * i])) |
                   (f32_to_b16<D == HBT_DTYPE_F16>(static_cast<float>(x[2 * i + 1])) << 16);
    }
}

// Any plan: lane l converts elements l, l + 64, ... of its chunk, so every load and store
// instruction of the wave covers one contiguous span.
template <int SD, int DD, int OP>
struct ConvertAny {
    typedef double Divisor;
    static __device__ __forceinline__ void run(const Record& rec, int64_t c, double divisor);
};
template <int SD, int DD, int OP>
__device__ __forceinline__ void ConvertAny<SD, DD, OP>::run(const Record& rec, int64_t c, double divisor) {
    constexpr int64_t SB = elem_bytes<SD>();
    constexpr int64_t DB = elem_bytes<DD>();
    constexpr int64_t kChunk = chunk_elems<SB, DB>();
    const int64_t e0 = c * kChunk;
    const int64_t n = rec.n;
    const int64_t len = (n - e0) < kChunk ? (n - e0) : kChunk;
    const gbyte* s = reinterpret_cast<const gbyte*>(static_cast<uintptr_t>(rec.src));
    gbyte* d = reinterpret_cast<gbyte*>(static_cast<uintptr_t>(rec.dst)) + e0 * DB;
    if (s != nullptr) s += e0 * SB;
    for (int64_t i = threadIdx.x; i < len; i += kCopyBlock) {
        narrow_store<DD>(d + i * DB, s != nullptr ? apply_op<OP>(widen_elem<SD>(s + i * SB), divisor) : 0.0);
    }
}

// Aligned plans (every destination 16-byte aligned, every source aligned to its unit): a
// lane moves units of U = 16 / max(source, destination bytes) elements, one access of
// U * bytes on each side (16 on the wider side; 8 or 4 on the narrower one), consecutive
// lanes on consecutive units; a 1 KB-of-source chunk is kPerLane units per lane (1 for a
// float64 source; a widening chunk is 2 KB of source, 4 or 8 units per lane), all loaded
// before the first store.
// The bits are ConvertAny's.
template <int SD, int DD, int OP>
struct ConvertAligned {
    typedef double Divisor;
    static __device__ __forceinline__ void run(const Record& rec, int64_t c, double divisor);
};
template <int SD, int DD, int OP>
__device__ __forceinline__ void ConvertAligned<SD, DD, OP>::run(const Record& rec, int64_t c, double divisor) {
    constexpr int SB = elem_bytes<SD>();
    constexpr int DB = elem_bytes<DD>();
    constexpr int U = 16 / (SB > DB ? SB : DB);
    constexpr int SW = U * SB / 4;
    constexpr int DW = U * DB / 4;
    constexpr int64_t kChunk = chunk_elems<SB, DB>();
    constexpr int kPerLane = static_cast<int>(kChunk / (int64_t(kCopyBlock) * U));
    static_assert(kChunk == int64_t(kPerLane) * kCopyBlock * U, "a chunk is whole units on every lane");
    const int64_t e0 = c * kChunk;
    const int64_t n = rec.n;
    const int64_t len = (n - e0) < kChunk ? (n - e0) : kChunk;
    const int64_t units = len / U;
    const gbyte* s = reinterpret_cast<const gbyte*>(static_cast<uintptr_t>(rec.src));
    gbyte* d = reinterpret_cast<gbyte*>(static_cast<uintptr_t>(rec.dst)) + e0 * DB;
    if (s == nullptr) {
        uint32_t zero[DW];
#pragma unroll
        for (int i = 0; i < DW; ++i) zero[i] = 0u;
#pragma unroll
        for (int j = 0; j < kPerLane; ++j) {
            const int64_t u = threadIdx.x + j * kCopyBlock;
            if (u < units) store_words<DW>(d + u * U * DB, zero);
        }
        if (threadIdx.x < len - units * U) narrow_store<DD>(d + (units * U + threadIdx.x) * DB, 0.0);
        return;
    }
    s += e0 * SB;
    uint32_t w[kPerLane][SW];
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) {
        const int64_t u = threadIdx.x + j * kCopyBlock;
        if (u < units) load_words<SW>(s + u * U * SB, w[j]);
    }
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) {
        const int64_t u = threadIdx.x + j * kCopyBlock;
        if (u < units) {
            double x[U];
            words_to_f64<SD, U>(w[j], x);
#pragma unroll
            for (int i = 0; i < U; ++i) x[i] = apply_op<OP>(x[i], divisor);
            uint32_t o[DW];
            f64_to_words<DD, U>(x, o);
            store_words<DW>(d + u * U * DB, o);
        }
    }
    if (threadIdx.x < len - units * U) {
        const int64_t e = units * U + threadIdx.x;
        narrow_store<DD>(d + e * DB, apply_op<OP>(widen_elem<SD>(s + e * SB), divisor));
    }
}

// ---- launches ------------------------------------------------------------------------
template <typename Mover>
__global__ __launch_bounds__(kCopyBlock) void copy_table_kernel(const int64_t* __restrict__ table, int64_t count,
                                                                typename Mover::Divisor divisor, int64_t chunk_base,
                                                                const int64_t* __restrict__ hints) {
    const int64_t chunk = chunk_base + static_cast<int64_t>(blockIdx.x);
    const Record rec = owning_record(table, count, chunk, hints);
    Mover::run(rec, chunk - rec.first, divisor);
}
template <typename Mover, int kRows>
__global__ __launch_bounds__(kCopyBlock) void copy_rows_kernel(RowTable<kRows> rows, typename Mover::Divisor divisor,
                                                               int64_t chunk_base) {
    const int64_t chunk = chunk_base + static_cast<int64_t>(blockIdx.x);
    const Record rec = owning_record(rows, chunk);
    Mover::run(rec, chunk - rec.first, divisor);
}

// Where a launch finds its records: a device table, or the arguments (few or rows non-null,
// few where the plan fits it).
struct Plan {
    const char* who;
    const int64_t* table;
    int64_t count;
    const int64_t* hints;
    const RowTable<kFewRows>* few;
    const RowTable<HBT_COPY_MAX_ROWS>* rows;
    int64_t chunks;
    bool aligned;
    hipStream_t stream;
};
template <typename Mover>
int32_t launch_mover(const Plan& p, typename Mover::Divisor divisor) {
    return launch_sliced(p.who, p.chunks, kCopyBlock, [&](int64_t first, dim3 grid) {
        if (p.few != nullptr) {
            copy_rows_kernel<Mover, kFewRows><<<grid, kCopyBlock, 0, p.stream>>>(*p.few, divisor, first);
        } else if (p.rows != nullptr) {
            copy_rows_kernel<Mover, HBT_COPY_MAX_ROWS><<<grid, kCopyBlock, 0, p.stream>>>(*p.rows, divisor, first);
        } else {
            copy_table_kernel<Mover><<<grid, kCopyBlock, 0, p.stream>>>(p.table, p.count, divisor, first, p.hints);
        }
    });
}
template <int SD, int DD, int OP>
int32_t launch_convert_pair(const Plan& p, double divisor) {
    return p.aligned ? launch_mover<ConvertAligned<SD, DD, OP>>(p, divisor) : launch_mover<ConvertAny<SD, DD, OP>>(p, divisor);
}
template <int SD>
int32_t launch_convert_from(const Plan& p, int32_t dst_dtype) {
    if (dst_dtype == HBT_DTYPE_F64) return launch_convert_pair<SD, HBT_DTYPE_F64, HBT_COPY_OP_COPY>(p, 1.0);
    if (dst_dtype == HBT_DTYPE_F32) return launch_convert_pair<SD, HBT_DTYPE_F32, HBT_COPY_OP_COPY>(p, 1.0);
    if (dst_dtype == HBT_DTYPE_BF16) return launch_convert_pair<SD, HBT_DTYPE_BF16, HBT_COPY_OP_COPY>(p, 1.0);
    return launch_convert_pair<SD, HBT_DTYPE_F16, HBT_COPY_OP_COPY>(p, 1.0);
}
int32_t launch_convert(const Plan& p, int32_t src_dtype, int32_t dst_dtype) {
    if (src_dtype == HBT_DTYPE_F64) return launch_convert_from<HBT_DTYPE_F64>(p, dst_dtype);
    if (src_dtype == HBT_DTYPE_F32) return launch_convert_from<HBT_DTYPE_F32>(p, dst_dtype);
    if (src_dtype == HBT_DTYPE_BF16) return launch_convert_from<HBT_DTYPE_BF16>(p, dst_dtype);
    return launch_convert_from<HBT_DTYPE_F16>(p, dst_dtype);
}

template <int SB, int DB, int OP, bool H = false>
int32_t launch_copy(const Plan& p, float divisor) {
    return p.aligned ? launch_mover<CopyAligned<SB, DB, OP, H>>(p, divisor) : launch_mover<CopyAny<SB, DB, OP, H>>(p, divisor);
}

// Conversions and division for 4- and 2-byte elements; H: the 2-byte side is fp16.
// Division by a power of two (the AVG pre-divide at a power-of-two world size) runs as a
// multiply by the exact reciprocal: the same bits, without the division sequence.
template <int OP, bool H>
int32_t launch_arith_op(const Plan& p, int ssz, int dsz, float divisor) {
    if (ssz == 4 && dsz == 4) return launch_copy<4, 4, OP>(p, divisor);
    if (ssz == 2 && dsz == 2) return launch_copy<2, 2, OP, H>(p, divisor);
    if (ssz == 4) return launch_copy<4, 2, OP, H>(p, divisor);
    return launch_copy<2, 4, OP, H>(p, divisor);
}
template <bool H>
int32_t launch_arith(const Plan& p, int ssz, int dsz, int32_t op, float divisor) {
    if (op == HBT_COPY_OP_DIVIDE) {
        const float recip = exact_reciprocal(divisor);
        if (recip != 0.0f) return launch_arith_op<kOpScale, H>(p, ssz, dsz, recip);
        return launch_arith_op<HBT_COPY_OP_DIVIDE, H>(p, ssz, dsz, divisor);
    }
    // conversions (same-dtype copies are bit copies)
    if (ssz == 4) return launch_copy<4, 2, HBT_COPY_OP_COPY, H>(p, divisor);
    return launch_copy<2, 4, HBT_COPY_OP_COPY, H>(p, divisor);
}

// Launches a validated plan (a known dtype pair and op, at least one chunk).
int32_t launch_plan(const Plan& p, int32_t src_dtype, int32_t dst_dtype, int32_t op, float divisor) {
    const int ssz = dtype_size(src_dtype);
    const int dsz = dtype_size(dst_dtype);
    if (op == HBT_COPY_OP_DIVIDE && src_dtype == HBT_DTYPE_F64 && dst_dtype == HBT_DTYPE_F64) {
        const float recip = exact_reciprocal(divisor);
        if (recip != 0.0f) return launch_convert_pair<HBT_DTYPE_F64, HBT_DTYPE_F64, kOpScale>(p, recip);
        return launch_convert_pair<HBT_DTYPE_F64, HBT_DTYPE_F64, HBT_COPY_OP_DIVIDE>(p, divisor);
    }
    if (op == HBT_COPY_OP_COPY && src_dtype == dst_dtype) {
        // Bit copy; fp64 moves as pairs of dwords (the host doubles its numels).
        if (ssz == 2) return launch_copy<2, 2, HBT_COPY_OP_COPY>(p, divisor);
        if (ssz == 4) return launch_copy<4, 4, HBT_COPY_OP_COPY>(p, divisor);
        set_error("%s: 8-byte elements must be passed as dword pairs (F32)", p.who);
        return HBT_ERR_UNSUPPORTED;
    }
    const bool wide = ssz == 8 || dsz == 8;
    const bool mixed_16 = (src_dtype == HBT_DTYPE_BF16 && dst_dtype == HBT_DTYPE_F16) ||
                          (src_dtype == HBT_DTYPE_F16 && dst_dtype == HBT_DTYPE_BF16);
    if (wide || mixed_16) {
        if (op != HBT_COPY_OP_COPY) {
            set_error("%s: division moves data within one dtype (F64, F32, BF16 or F16) or "
                      "between F32 and a 2-byte dtype (got %d -> %d)", p.who, src_dtype, dst_dtype);
            return HBT_ERR_UNSUPPORTED;
        }
        return launch_convert(p, src_dtype, dst_dtype);
    }
    if (src_dtype == HBT_DTYPE_F16 || dst_dtype == HBT_DTYPE_F16) return launch_arith<true>(p, ssz, dsz, op, divisor);
    return launch_arith<false>(p, ssz, dsz, op, divisor);
}

bool copy_op_ok(const char* who, int32_t src_dtype, int32_t dst_dtype, int32_t op) {
    if (dtype_size(src_dtype) == 0 || dtype_size(dst_dtype) == 0 ||
        (op != HBT_COPY_OP_COPY && op != HBT_COPY_OP_DIVIDE)) {
        set_error("%s: bad dtype pair (%d, %d) or op %d", who, src_dtype, dst_dtype, op);
        return false;
    }
    return true;
}

}  // namespace
}  // namespace hbt

using namespace hbt;

extern "C" {

int64_t hbt_copy_chunk_elems(int32_t src_dtype, int32_t dst_dtype) {
    const int ssz = dtype_size(src_dtype);
    const int dsz = dtype_size(dst_dtype);
    if (ssz == 0 || dsz == 0) return -1;
    // 1 KB of source, 2 KB when widening (the convert kernels' chunks are the copy
    // kernels'); F64 -> F64: the chunk of the DIVIDE op (a same-dtype COPY moves F32 dword
    // pairs).
    return int64_t(kCopyBlock) * 16 / ssz * (ssz < dsz ? 2 : 1);
}

int32_t hbt_copy_intervals(const int64_t* table, int64_t count, int64_t total_chunks,
                           int32_t src_dtype, int32_t dst_dtype, int32_t op, float divisor,
                           int32_t flags, void* stream) {
    clear_error();
    if (count < 0 || total_chunks < 0 || (count > 0 && table == nullptr)) {
        set_error("hbt_copy_intervals: bad table/count/total_chunks");
        return HBT_ERR_INVALID_ARGUMENT;
    }
    if ((flags & ~(HBT_COPY_ALIGNED | HBT_COPY_HINTS)) != 0) {
        set_error("hbt_copy_intervals: unknown flags 0x%x", static_cast<unsigned>(flags));
        return HBT_ERR_INVALID_ARGUMENT;
    }
    const bool aligned = (flags & HBT_COPY_ALIGNED) != 0;
    if (count == 0 || total_chunks == 0) return HBT_OK;
    if (!copy_op_ok("hbt_copy_intervals", src_dtype, dst_dtype, op)) return HBT_ERR_INVALID_ARGUMENT;
    // The hints follow the count records of 4 int64 each.
    const int64_t* hints = (flags & HBT_COPY_HINTS) != 0 ? table + 4 * count : nullptr;
    return launch_plan(Plan{"hbt_copy_intervals", table, count, hints, nullptr, nullptr, total_chunks, aligned, as_stream(stream)},
                       src_dtype, dst_dtype, op, divisor);
}

int32_t hbt_copy_rows(const int64_t* rows, int32_t count, int32_t src_dtype, int32_t dst_dtype, int32_t op,
                      float divisor, void* stream) {
    clear_error();
    if (count < 0 || count > HBT_COPY_MAX_ROWS || (count > 0 && rows == nullptr)) {
        set_error("hbt_copy_rows: bad rows/count (%d of at most %d)", count, HBT_COPY_MAX_ROWS);
        return HBT_ERR_INVALID_ARGUMENT;
    }
    if (!copy_op_ok("hbt_copy_rows", src_dtype, dst_dtype, op)) return HBT_ERR_INVALID_ARGUMENT;
    int64_t scale = 1;
    if (src_dtype == HBT_DTYPE_F64 && dst_dtype == HBT_DTYPE_F64 && op == HBT_COPY_OP_COPY) {
        src_dtype = dst_dtype = HBT_DTYPE_F32;  // an 8-byte element moves as two dwords
        scale = 2;
    }
    const int64_t chunk = hbt_copy_chunk_elems(src_dtype, dst_dtype);
    const uint64_t ssz = static_cast<uint64_t>(dtype_size(src_dtype)), dsz = static_cast<uint64_t>(dtype_size(dst_dtype));
    const uint64_t src_align = 16 * ssz / (ssz > dsz ? ssz : dsz);
    RowTable<HBT_COPY_MAX_ROWS> tab;  // what the plan does not fill is never read
    tab.count = 0;
    int64_t chunks = 0;
    bool aligned = true;
    for (int32_t i = 0; i < count; ++i) {
        const int64_t src = rows[3 * i], dst = rows[3 * i + 1], n = rows[3 * i + 2];
        if (n < 0 || (n > 0 && dst == 0)) {
            set_error("hbt_copy_rows: row %d has a null destination or a negative count", i);
            return HBT_ERR_INVALID_ARGUMENT;
        }
        if (n == 0) continue;  // the search wants strictly increasing first chunks
        aligned = aligned && static_cast<uint64_t>(dst) % 16 == 0 && static_cast<uint64_t>(src) % src_align == 0;
        tab.rec[tab.count++] = Record{src, dst, n * scale, chunks};
        chunks += (n * scale + chunk - 1) / chunk;
    }
    if (chunks == 0) return HBT_OK;
    tab.shift = 0;
    while (((chunks - 1) >> tab.shift) >= kRowHints) ++tab.shift;
    std::memset(tab.hint, 0, sizeof tab.hint);
    int r = 0;
    for (int64_t j = 0; j <= (chunks - 1) >> tab.shift; ++j) {
        while (r + 1 < tab.count && tab.rec[r + 1].first <= (j << tab.shift)) ++r;
        const bool split = r + 1 < tab.count && tab.rec[r + 1].first < ((j + 1) << tab.shift);
        tab.hint[j >> 2] |= (static_cast<uint32_t>(r) | (split ? kHintSplit : 0u)) << (8 * (j & 3));
    }
    Plan plan{"hbt_copy_rows", nullptr, tab.count, nullptr, nullptr, &tab, chunks, aligned, as_stream(stream)};
    RowTable<kFewRows> few;
    if (tab.count <= kFewRows) {
        std::copy(tab.rec, tab.rec + tab.count, few.rec);
        std::memcpy(few.hint, tab.hint, sizeof few.hint);
        few.count = tab.count;
        few.shift = tab.shift;
        plan.few = &few;
    }
    return launch_plan(plan, src_dtype, dst_dtype, op, divisor);
}

}  // extern "C"
