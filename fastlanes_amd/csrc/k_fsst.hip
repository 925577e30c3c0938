// k_fsst.hip -- FSST string pages on gfx950.
//
// Page per vector (include/fls/cor/exp/fsst/fsst_exp.hpp:35-52, src/cor/lyt/vec.cpp:160-207): buffer 0 holds the
// 1024 compressed strings back to back, buffer 1 their cumulative end offsets (u32) in transposed order.
// Decoding follows include/fls/encoder/assert_eq.hpp:166-210: untranspose the offsets, then decode each string
// with fsst_decompress (include/fls/cor/prm/fsst/fsst.h:152-258): code < 255 emits symbol[code] (len[code] bytes),
// code 255 emits the next byte literally.
//
// A block of 256 threads owns one segment (256 strings of a vector), whose compressed bytes it takes in chunks of 8 KiB, 32
// bytes (a granule) per thread, read straight from HBM into registers. Launches:
//   k_fsst_count  every granule's and segment's decoded size, and the strings' ends in order;
//   k_fsst_scan   the vectors' output bases, when they are too many for each block to sum them itself;
//   k_fsst        per chunk: one block scan of the granules' sizes; each thread joins its symbols into 8-byte words of the
//                 LDS image of the output (44 of its 76 vector instructions per four codes), which is copied out with
//                 16-byte stores aligned to the output, and leaves the packed exclusive prefix of its codes' lengths in
//                 LDS: a string's end is its granule's base plus one byte of it.
// The bases came from a decoupled look-back in one pass over the compressed bytes before: its dispatch-order tickets (one
// same-address atomic per segment) and waits took 48 of 135 us for 2^21 strings of 36 bytes. Every symbol was OR-ed into
// a zeroed image by an LDS atomic; now a word is stored by the one thread that has its last byte, and threads that have
// only earlier bytes of it OR them in after a barrier. (Writing each symbol's 8 bytes at its own unaligned place, two
// instructions per code, measured 135 us: unaligned LDS writes take about one cycle per lane.) Escapes are found from two
// 32-bit masks of a granule, its bytes of 255 and the strings' ends in it; while every thread looked its ends up and walked
// its escapes, a column with 3% of its bytes escaped took 102 us where it now takes 85. 2^21 strings: 151 -> 71 us
// a call, k_fsst 42, bound by its vector instructions. The build refuses a k_fsst that spills registers: two
// intermediate forms of it that did (to scratch) gave wrong bytes in a hundredth of the segments, others from run to run; what
// made the difference is not known.
// A vector with a malformed segment (non-monotone offsets) takes a per-string path that reads and writes global memory byte
// by byte, for all four of its segments: the granules' sizes are kept by byte position, which is one segment's own only
// while no segment of the vector reaches back over another.
#include <algorithm>

#include "../../include/fls_gpu.h"
#include "gpu_internal.hpp"
#include "page_kernels.hpp"

namespace fls {

namespace {

constexpr unsigned kSeg      = 256;         // strings per segment (= threads per block)
constexpr unsigned kSegPerV  = 1024 / kSeg;
constexpr unsigned kWaves    = kSeg / 64;
constexpr uint32_t kShare    = 32;          // compressed bytes per thread and chunk
constexpr uint32_t kChunk    = kShare * kSeg;
constexpr uint32_t kOutLds   = 12 * 1024;   // bytes of the LDS image of decoded output
constexpr uint32_t kMaxComp  = 1u << 28;    // compressed bytes of a segment whose decoded size is below 2^32
constexpr unsigned kWideCount = 1024;       // vectors of a page that k_fsst_count takes with 1024 threads each
constexpr unsigned kDirect   = 1024;        // vectors of a column whose sizes each block sums itself (4 loads per thread)

// error bits (StringPlan::d_err)
constexpr uint32_t kErrCap = 4;

enum : int { FS_OFFSETS = 0, FS_BYTES = 1, FS_ALL = 2 };

// Place in LDS of the end offset of string i, which is transposed: i = r + 8*ORDER[b] + 64c sits at 128r + 16b + c. Rows
// of 140 dwords and runs of 17 keep 32 consecutive strings on 16 banks; unpadded they share two.
constexpr unsigned kEndRow = 140;
__device__ __forceinline__ unsigned end_place(unsigned i) { return (i & 7) * kEndRow + order8((i >> 3) & 7) * 17 + (i >> 6); }

// Exclusive scan of one value per thread over the block; returns the block total in *total.
template <typename U>
__device__ __forceinline__ U block_exclusive_scan(U x, U* wsum, U* total) {
    const unsigned lane = threadIdx.x % 64, w = threadIdx.x / 64;
    U              inc  = x;
    for (unsigned d = 1; d < 64; d <<= 1) {
        const U y = __shfl_up(inc, d, 64);
        if (lane >= d) inc += y;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    U before = 0, all = 0;
    for (unsigned k = 0; k < kWaves; ++k) {
        const U s = wsum[k];
        if (k < w) before += s;
        all += s;
    }
    *total = all;
    return before + inc - x;
}

// 32 bytes of a granule into registers: two 16-byte loads; the last, partial granule of a segment by dwords and its
// last bytes (nothing at or past `avail` is read).
__device__ __forceinline__ void load_granule(const uint8_t* p, uint32_t avail, uint32_t (&wd)[8]) {
    if (avail >= kShare) {
        const v4u a = *reinterpret_cast<const v4u_ua*>(p), b = *reinterpret_cast<const v4u_ua*>(p + 16);
        wd[0] = a[0], wd[1] = a[1], wd[2] = a[2], wd[3] = a[3], wd[4] = b[0], wd[5] = b[1], wd[6] = b[2], wd[7] = b[3];
    } else {
        uint32_t rest = 0;
        for (uint32_t k = avail & ~3u; k < avail; ++k) rest |= (uint32_t)p[k] << (8 * (k & 3u));
        static_for<8>([&](auto d) {
            wd[d.value] = 4 * d.value == (avail & ~3u) ? rest : 0u;
            if (4 * d.value + 4 <= avail) wd[d.value] = *reinterpret_cast<const u32_ua*>(p + 4 * d.value);
        });
    }
}
// 0x80 in every byte of w that is 255.
__device__ __forceinline__ uint32_t ff_bytes(uint32_t w) { return ((w & 0x7f7f7f7fu) + 0x01010101u) & w & 0x80808080u; }
__device__ __forceinline__ bool has_ff(const uint32_t (&wd)[8]) {
    uint32_t z = 0;
    static_for<8>([&](auto d) { z |= ff_bytes(wd[d.value]); });
    return z != 0;
}
// Bit j: byte j of the granule is 255.
__device__ __forceinline__ uint32_t ff_mask(const uint32_t (&wd)[8]) {
    uint32_t ff = 0;
    static_for<8>([&](auto D) {
        constexpr unsigned d = decltype(D)::value;
        ff |= (__builtin_amdgcn_udot4(ff_bytes(wd[d]), 0x08040201u, 0u, false) >> 7) << (4 * d);
    });
    return ff;
}
template <unsigned J>
__device__ __forceinline__ uint32_t byte_of(const uint32_t (&wd)[8]) {
    return (wd[J / 4] >> (8 * (J % 4))) & 255u;
}

// What k_fsst_count leaves for k_fsst per segment: decoded bytes, those of the vector's segments before it (kMalformed:
// the vector's offsets are not monotone), and the place of its compressed bytes in the vector's.
struct FsstSeg {
    uint64_t total, before;
    uint32_t s0, n;
};
constexpr uint64_t kMalformed = 1ull << 63, kEscapes = 1ull << 62;  // in `before`; kEscapes: some granule is kSpecial

// A segment's compressed bytes `seg`, n of them, and the ends of its strings (LDS, from its start).
struct Segment {
    const uint8_t*  seg;
    uint32_t        n;
    const uint32_t* end;
};

// Place of a segment's first granule in StringPlan::d_sizes: granules of 32 bytes from the column's start, one more per
// segment before it for the partial ones (segments that follow one another in memory: no two share a place).
__device__ __forceinline__ uint64_t sizes_at(uint64_t page_off, const uint8_t* page, const uint8_t* bytes, uint64_t seg) {
    return (page_off + (uint64_t)(bytes - page)) / kShare + seg;
}
// In d_sizes: the granule holds, or starts with, part of an escape; its first byte is an escape's literal.
constexpr uint32_t kSpecial = 0x8000, kLiteral = 0x4000, kSize = kLiteral - 1;

// A thread's granule of the chunk at c0: its bytes (0 past the segment), its place in the segment, how many bytes the
// segment has there.
struct Granule {
    uint32_t wd[8];
    uint32_t q0, lim;
};
__device__ __forceinline__ Granule open_granule(const Segment& g, uint32_t c0, unsigned tid) {
    Granule r;
    r.q0  = c0 + tid * kShare;
    r.lim = r.q0 < g.n ? (g.n - r.q0 < kShare ? g.n - r.q0 : kShare) : 0;
    if (r.lim) {
        load_granule(g.seg + r.q0, g.n - r.q0, r.wd);
    } else {
        static_for<8>([&](auto d) { r.wd[d.value] = 0u; });
    }
    return r;
}

// Bit k of m as byte k, 0 or 255.
__device__ __forceinline__ uint32_t spread4(uint32_t m) { return (((m & 15u) * 0x00204081u) & 0x01010101u) * 255u; }
// Escapes of a granule, bit j for its byte j: `esc` the escapes that emit the byte after them (one whose string ends
// right after it emits 0), `none` the bytes that emit nothing (literals, and bytes past the segment).
struct Escapes {
    uint32_t esc, none;
};
// Where strings end in a granule: bit j of `before`, right before its byte j; `after`, right after its last byte.
struct Ends {
    uint32_t before;
    bool     after;
};
// ff: the bytes that are 255; literal: the first byte is one. Inside a string every second byte of a run of 255 is a literal
// (a run begins with an escape code: after a code or a literal comes a code). Which bytes lie at an even distance from their
// run's start is the parity of the last start at or before them, spread upwards in five steps.
__device__ __forceinline__ Escapes find_escapes(uint32_t ff, const Ends& e, uint32_t lim, bool literal) {
    const uint32_t past = lim >= kShare ? 0u : ~0u << lim, in = literal, f = ff & ~past & ~in;
    const uint32_t starts = f & (~(f << 1) | e.before);
    uint32_t       even = starts & 0x55555555u, open = ~starts;
    for (unsigned d = 1; d < 32; d *= 2) {
        even |= open & (even << d);
        open &= open << d;
    }
    const uint32_t codes = f & ~(even ^ 0x55555555u);
    return {codes & ~(e.before >> 1 | (uint32_t)e.after << 31), ((codes << 1 | in) & ~e.before) | past};
}
// What a granule (a whole one) says of the byte after it: `lit`, that it is a literal (the run of 255 before it, inside its
// string, is of odd length); `keeps`, that it is one if the granule's own first byte is: a granule of nothing but 255
// inside one string, because 32 is even.
struct After {
    bool lit, keeps;
};
__device__ __forceinline__ After after_granule(uint32_t ff, const Ends& e) {
    const uint32_t run = ff == ~0u ? 32u : (uint32_t)__builtin_clz(~ff);
    const uint32_t own = e.before ? (uint32_t)__builtin_clz(e.before) + 1 : 32u;  // bytes of the granule in its last string
    return {!e.after && ((run < own ? run : own) & 1u) != 0, run == 32 && !e.before && !e.after};
}
// The ends in granule i + lane, by a whole wave; bits: kEndWords words of LDS of its own.
constexpr unsigned kEndWords = 65;
__device__ __forceinline__ Ends window_ends(const uint32_t* end, uint32_t i, unsigned lane, uint32_t* bits) {
    wave_sync();  // the last window's have been read
    bits[lane] = 0u;
    if (lane == 0) bits[64] = 0u;
    wave_sync();
    static_for<kSeg / 64>([&](auto k) {
        const uint32_t at = end[lane + 64 * decltype(k)::value] - i * kShare;
        if (at <= 64 * kShare) atomicOr(&bits[at / kShare], 1u << (at % kShare));
    });
    wave_sync();
    return {bits[lane], (bits[lane + 1] & 1u) != 0};
}
// Whether granule `at` (not the first) starts on a literal, by a whole wave: 64 granules back at a time until one says so.
__device__ __forceinline__ bool starts_on_literal(const Segment& g, uint32_t at, unsigned lane, uint32_t* bits) {
    if (g.seg[at * kShare - 1] != 255) return false;
    while (at) {
        const uint32_t n = at < 64 ? at : 64, i = at - n;
        const Ends     e = window_ends(g.end, i, lane, bits);
        After          a {false, true};
        if (lane < n) {
            uint32_t wd[8];
            load_granule(g.seg + (i + lane) * kShare, kShare, wd);
            a = after_granule(ff_mask(wd), e);
        }
        const uint64_t says = __ballot(!a.keeps);
        if (says) return (__ballot(a.lit) >> (63 - __builtin_clzll(says))) & 1u;
        at = i;
    }
    return false;  // the segment's first byte is a code
}

// Values the compiler cannot carry over from before: it would take the table addresses out of all forms of emit_granule,
// in registers that it then spills.
__device__ __forceinline__ void forget(uint32_t (&w)[8]) {
    asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]), "+v"(w[4]), "+v"(w[5]), "+v"(w[6]), "+v"(w[7]));
}

// Joins a thread's symbols into the 8-byte words of the LDS image. acc holds the bytes of the word not yet complete.
struct Emit {
    uint8_t* image;
    uint64_t acc;
    uint32_t at;  // bit position in the image
    // x: `bits` bits, 0 above them. WIDE: bits may be 64
    template <bool WIDE>
    __device__ __forceinline__ void add(uint64_t x, uint32_t bits) {
        const uint64_t lo = acc | (x << (at & 63u));
        const uint64_t hi = WIDE ? (x >> 8) >> (~(at + 7u) & 63u) : x >> (-at & 63u);  // the bytes past the word
        const uint32_t to   = at + bits;
        const bool     full = (at ^ to) >= 64u;
        if (full) *reinterpret_cast<uint64_t*>(image + ((at >> 3) & ~7u)) = lo;
        acc = full ? hi : lo;
        at  = to;
    }
};
// Emits the granule's symbols and packs their lengths into lk. KIND 0 (symbols of at most 3 bytes): a table entry is the
// symbol and its bits, two codes are one addition. KIND 1 (at most 7): the entry's top byte is the length. KIND 2: the
// lengths are a table of their own. Bytes that emit nothing have been replaced by 255, whose symbol is empty, and
// `none` (only then) drops their lengths.
template <int KIND, bool NONE>
__device__ __forceinline__ void emit_granule(const uint32_t (&wd_in)[8], uint32_t none, const uint64_t* sym,
                                             const uint8_t* len, Emit& o, uint32_t (&lk)[8]) {
    uint32_t wd[8];
    static_for<8>([&](auto d) { wd[d] = wd_in[d]; });
    forget(wd);
    if constexpr (NONE) asm volatile("" : "+v"(none));
    static_for<8>([&](auto D) {
        constexpr unsigned d = decltype(D)::value;
        const uint32_t     drop = NONE ? spread4(none >> (4 * d)) : 0u;
        uint64_t           x[4];
        uint32_t           l[4];  // KIND 0: bits
        static_for<4>([&](auto k) {
            const uint32_t c = byte_of<4 * d + decltype(k)::value>(wd);
            x[k]             = sym[c];
            if constexpr (KIND == 2) l[k] = len[c];
        });
        static_for<4>([&](auto k) {
            if constexpr (KIND == 0) l[k] = (uint32_t)(x[k] >> 32), x[k] &= 0xffffffffull;
            if constexpr (KIND == 1) l[k] = (uint32_t)(x[k] >> 56), x[k] &= 0x00ffffffffffffffull;
            if constexpr (NONE) l[k] &= ~(drop >> (8 * decltype(k)::value));
        });
        // (the asm keeps the packing here: sunk to its use it would hold every length in a register of its own)
        if constexpr (KIND == 0) {
            lk[d] = (l[0] | (l[1] << 8) | (l[2] << 16) | (l[3] << 24)) >> 3;  // at most 3 each: no bit crosses a byte
            asm volatile("" : "+v"(lk[d]));
            o.template add<false>(x[0] | (x[1] << l[0]), l[0] + l[1]);
            o.template add<false>(x[2] | (x[3] << l[2]), l[2] + l[3]);
        } else {
            lk[d] = l[0] | (l[1] << 8) | (l[2] << 16) | (l[3] << 24);
            asm volatile("" : "+v"(lk[d]));
            static_for<4>([&](auto k) { o.template add<KIND == 2>(x[k], 8 * l[k]); });
        }
        if constexpr (d % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    });
}
// Exclusive prefix of the granule's packed lengths into its 32 bytes of `pre` (at most 248: a byte each).
__device__ __forceinline__ void granule_prefix(const uint32_t (&lk)[8], uint8_t* p) {
    uint32_t run = 0, ex[8];
    static_for<8>([&](auto d) {
        uint32_t t = lk[d] + (lk[d] << 8);
        t += t << 16;  // inclusive prefix within the dword
        ex[d] = (t << 8) + __builtin_amdgcn_perm(run, run, 0u);  // run in every byte
        run += t >> 24;
    });
    *reinterpret_cast<v4u*>(p)      = v4u {ex[0], ex[1], ex[2], ex[3]};
    *reinterpret_cast<v4u*>(p + 16) = v4u {ex[4], ex[5], ex[6], ex[7]};
}
// Decoded bytes of the granule (codes and escapes alike; dropped bytes not).
__device__ __forceinline__ uint32_t granule_size(const uint32_t (&wd)[8], uint32_t none, const uint8_t* len) {
    uint32_t s = 0;
    static_for<8>([&](auto d) {
        uint32_t l[4];
        static_for<4>([&](auto k) { l[k] = len[byte_of<4 * decltype(d)::value + decltype(k)::value>(wd)]; });
        if (none)
            static_for<4>([&](auto k) { l[k] = (none >> (4 * decltype(d)::value + decltype(k)::value)) & 1u ? 0u : l[k]; });
        s += l[0] + l[1] + l[2] + l[3];
        if constexpr (decltype(d)::value % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    });
    return s;
}

// Decoded length of one string, byte by byte from global memory.
__device__ __forceinline__ uint32_t string_length(const uint8_t* cb, uint32_t s, uint32_t e, const uint8_t* len) {
    uint32_t tot = 0;
    for (uint32_t q = s; q < e;) {
        const unsigned c = cb[q];
        if (c == 255) tot += 1, q += 2;
        else tot += len[c], q += 1;
    }
    return tot;
}
// One string decoded from global memory to global memory, byte by byte, into out[w, stop).
__device__ __forceinline__ void decode_string_global(const uint8_t* cb, uint32_t s, uint32_t e, const FsstTableDev* table,
                                                     uint8_t* out, uint64_t w, uint64_t stop) {
    for (uint32_t q = s; q < e && w < stop;) {
        const unsigned c = cb[q];
        if (c == 255) {
            out[w++] = q + 1 < e ? cb[q + 1] : 0;
            q += 2;
        } else {
            const uint64_t x = table->symbol[c];
            const unsigned n = table->len[c];
            for (unsigned b = 0; b < n && w < stop; ++b) out[w++] = (uint8_t)(x >> (8 * b));
            q += 1;
        }
    }
}

// One block per vector: its segments' decoded sizes and places (FsstSeg), every string's end within its segment, and every
// granule's decoded size. Bound by the length reads from LDS and, per block, by the chain offsets -> bytes -> lengths.
// GROUPS: segments at a time, 256 threads each. 4 (the chain once) while two rounds of such blocks, two per compute unit,
// hold the page: 2^19 strings of 36 bytes decode in 27 us against 33 with 1; beyond that 1, whose eight small blocks per
// compute unit overlap their chains: 2^21 strings count in 23 us against 31. (A block per segment, which reads the
// vector's offsets four times, took 34 us.)
template <unsigned GROUPS>
__global__ __launch_bounds__(kSeg* GROUPS, 8) void k_fsst_count(const uint8_t* __restrict__ page, uint64_t page_off,
                                                                const FsstTableDev* __restrict__ table, uint64_t seg0,
                                                                FsstSeg* __restrict__ segs, uint64_t* __restrict__ vecs,
                                                                uint32_t* __restrict__ str_end,
                                                                uint16_t* __restrict__ sizes) {
    __shared__ uint8_t  len[256];
    __shared__ uint32_t ends[8 * kEndRow], end[1024];  // transposed from the vector's start, then in order from the segment's
    __shared__ uint64_t wsum[kSegPerV][kWaves];
    __shared__ uint32_t malformed, escapes, bits[GROUPS * kWaves][kEndWords];
    const unsigned      t = threadIdx.x, tid = t % kSeg, lane = t % 64, v = blockIdx.x;
    const unsigned      group = __builtin_amdgcn_readfirstlane(t / kSeg);
    const uint8_t*      cb  = vbuf(page, 2, v, 0);
    const uint64_t      seg = seg0 + (uint64_t)v * kSegPerV;
    if (t < 256) {
        const v4u q = *reinterpret_cast<const v4u_ua*>(vbuf(page, 2, v, 1) + 16 * t);  // transposed 4 t .. 4 t + 3
        static_for<4>([&](auto k) { ends[(t >> 5) * kEndRow + ((t >> 2) & 7) * 17 + 4 * (t & 3) + k] = q[k.value]; });
        len[t] = table->len[t];
    }
    if (t == 0) malformed = 0, escapes = 0;
    __syncthreads();
    auto bound = [&](unsigned h) {  // of the segments
        return h ? (uint32_t)__builtin_amdgcn_readfirstlane(ends[end_place(h * kSeg - 1)]) : 0u;
    };
    auto span = [&](unsigned h) {
        const uint32_t a = bound(h), b = bound(h + 1);
        return a <= b && b - a <= kMaxComp;
    };
    for (unsigned h = group; h < kSegPerV; h += GROUPS) {
        const unsigned i = h * kSeg + tid;
        const uint32_t e = ends[end_place(i)], s = i ? ends[end_place(i - 1)] : 0u, s0 = bound(h);
        end[i]                          = e - s0;
        str_end[(seg + h) * kSeg + tid] = e - s0;
        if (!(span(h) && s0 <= s && s <= e && e <= bound(h + 1))) malformed = 1;
    }
    __syncthreads();
    for (unsigned h = group; h < kSegPerV; h += GROUPS) {
        const uint32_t s0 = bound(h);
        const Segment  g {cb + s0, span(h) ? bound(h + 1) - s0 : 0u, end + h * kSeg};
        uint32_t       own = 0;  // below 2^32: kMaxComp
        if (!malformed) {
            uint16_t* const at = sizes + sizes_at(page_off, page, g.seg, seg + h);
            // a wave's granules follow one another, so that what a literal needs to know of the bytes before it is carried
            // along (a walk back over its run for every granule made a segment of escapes cost the square of its length; a
            // string of 2 MB of 255 takes 2.2 ms a call)
            const uint32_t n = (g.n + kShare - 1) / kShare, per = ((n + kWaves - 1) / kWaves + 63) & ~63u;
            const uint32_t first = __builtin_amdgcn_readfirstlane(tid / 64) * per, stop = first + per < n ? first + per : n;
            bool           carry = first && first < stop && starts_on_literal(g, first, lane, bits[t / 64]);
            for (uint32_t i = first; i < stop; i += 64) {
                const Granule r       = open_granule(g, i * kShare, lane);
                bool          literal = false;
                const bool    special = r.lim && has_ff(r.wd);
                uint32_t      none = r.lim >= kShare ? 0u : ~0u << r.lim, flags = 0;
                if (__any(special) || carry) {
                    const Ends     e  = window_ends(g.end, i, lane, bits[t / 64]);
                    const uint32_t ff = ff_mask(r.wd);
                    After          a {false, false};
                    if (r.lim >= kShare) a = after_granule(ff, e);
                    const uint64_t says = __ballot(!a.keeps), lit = __ballot(a.lit), before = says & ((1ull << lane) - 1);
                    literal = before ? (lit >> (63 - __builtin_clzll(before))) & 1u : carry;
                    carry   = says ? (lit >> (63 - __builtin_clzll(says))) & 1u : carry;
                    if (r.lim && (special || literal)) {
                        none  = find_escapes(ff, e, r.lim, literal).none;
                        flags = literal ? kSpecial | kLiteral : kSpecial;
                    }
                    if (lane == 0) atomicOr(&escapes, 1u << h);
                }
                if (r.lim) {
                    const uint32_t size = granule_size(r.wd, none, len);
                    at[i + lane]        = (uint16_t)(size | flags);
                    own += size;
                }
            }
        } else {
            own = string_length(cb, tid ? end[h * kSeg + tid - 1] + s0 : s0, end[h * kSeg + tid] + s0, len);
        }
        uint64_t mine = own;
        for (unsigned d = 32; d >= 1; d >>= 1) mine += __shfl_xor((unsigned long long)mine, d, 64);
        if (lane == 0) wsum[h][tid / 64] = mine;
    }
    __syncthreads();
    if (t == 0) {
        uint64_t vec = 0;
        for (unsigned k = 0; k < kSegPerV; ++k) {
            uint64_t all = 0;
            for (unsigned w = 0; w < kWaves; ++w) all += wsum[k][w];
            segs[seg + k] = {all, vec | (malformed ? kMalformed : 0) | ((escapes >> k) & 1u ? kEscapes : 0), bound(k), span(k) ? bound(k + 1) - bound(k) : 0u};
            vec += all;
        }
        vecs[seg / kSegPerV] = vec;
    }
}

// Exclusive sums of n vectors' decoded sizes, one block.
__global__ __launch_bounds__(1024) void k_fsst_scan(const uint64_t* __restrict__ vecs, uint64_t* __restrict__ bases,
                                                    uint32_t n) {
    __shared__ uint64_t wsum[16];
    __shared__ uint64_t carry;
    const unsigned      tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    uint64_t            base = 0;
    constexpr unsigned  K    = 2;  // sizes per thread and round
    for (uint32_t r = 0; r < n; r += 1024 * K) {
        uint64_t x[K], s = 0;
        static_for<K>([&](auto k) {
            const uint32_t i = r + tid * K + k;
            x[k]             = i < n ? vecs[i] : 0ull;
        });
        static_for<K>([&](auto k) { s += x[k]; });
        uint64_t inc = s;
        for (unsigned d = 1; d < 64; d <<= 1) {
            const uint64_t y = __shfl_up((unsigned long long)inc, d, 64);
            if (lane >= d) inc += y;
        }
        if (lane == 63) wsum[wave] = inc;
        __syncthreads();
        uint64_t b = base + inc - s;
        for (unsigned w = 0; w < wave; ++w) b += wsum[w];
        if (tid == 1023) carry = b + s;
        static_for<K>([&](auto k) {
            const uint32_t i = r + tid * K + k;
            if (i < n) bases[i] = b;
            b += x[k];
        });
        __syncthreads();
        base = carry;
    }
}

// MODE FS_OFFSETS writes the n+1 string end offsets; FS_BYTES writes the bytes at the caller's offsets; FS_ALL writes
// both. `offsets` is indexed from the column's first string; `first_string` is the page's. segs: the column's
// segments; vecs / bases: its vectors' decoded sizes and the sums before each (nullptr: at most kDirect vectors, summed
// here); seg0: the page's first segment.
// About 24 KB of LDS and at most 80 VGPRs: six blocks of four waves per compute unit.
template <int MODE>
__global__ __launch_bounds__(kSeg, 6) void k_fsst(const uint8_t* __restrict__ page, uint64_t page_off,
                                               const FsstTableDev* __restrict__ table, uint64_t first_string,
                                               uint64_t* __restrict__ offsets, uint8_t* __restrict__ out, uint64_t cap,
                                               uint32_t* err, const FsstSeg* __restrict__ segs,
                                               const uint64_t* __restrict__ vecs, const uint64_t* __restrict__ bases, const uint32_t* __restrict__ str_end,
                                               const uint16_t* __restrict__ sizes, uint64_t seg0) {
    constexpr bool EMIT = MODE != FS_OFFSETS;
    __shared__ uint64_t sym[256];  // FsstTableDev::packed
    __shared__ uint8_t  len[256];
    __shared__ __attribute__((aligned(16))) uint8_t pre[kChunk];  // per compressed byte of the chunk: decoded bytes
                                                                  // before it in its granule
    __shared__ uint32_t end[kSeg];                                // of each string, from the segment's start
    __shared__ uint32_t sbase[kSeg];                              // decoded bytes of the chunk before each granule
    __shared__ uint32_t wsum[kWaves];
    __shared__ uint64_t wsum64[kWaves];
    __shared__ uint32_t window;
    __shared__ uint32_t ends[kSeg + 1];  // bit j of word i: a string ends right before byte j of the chunk's granule i
    __shared__ __attribute__((aligned(16))) uint8_t image[kOutLds + 32];
    const unsigned  tid = threadIdx.x;
    const uint64_t  seg = seg0 + blockIdx.x;
    const FsstSeg   st  = segs[seg];
    const uint32_t  kind = table->kind;
    const uint8_t*  cb   = vbuf(page, 2, blockIdx.x / kSegPerV, 0);
    const Segment   g {cb + st.s0, st.n, end};
    const uint16_t* size_at = sizes + sizes_at(page_off, page, g.seg, seg);
    Granule         r  = open_granule(g, 0, tid);
    uint32_t        sz = r.lim ? size_at[r.q0 / kShare] : 0u;
    const uint64_t  vec = seg / kSegPerV, seg_total = st.total;
    uint64_t* const oseg     = offsets + first_string + (uint64_t)blockIdx.x * kSeg;
    uint64_t        seg_base = 0, before = 0;
    bool            given_ok = true;
    if constexpr (MODE == FS_BYTES) {
        seg_base = oseg[0];
        given_ok = oseg[kSeg] >= seg_base && oseg[kSeg] - seg_base == seg_total;
    } else {
        seg_base = st.before & ~(kMalformed | kEscapes);
        if (bases) seg_base += bases[vec];
        else
            for (uint64_t k = tid; k < vec; k += kSeg) before += vecs[k];
    }
    sym[tid] = table->packed[tid], len[tid] = table->len[tid];
    end[tid] = str_end[seg * kSeg + tid];  // read back where it is needed: one register less through the emission
    if (MODE != FS_BYTES && !bases) {
        for (unsigned d = 32; d >= 1; d >>= 1) before += __shfl_xor((unsigned long long)before, d, 64);
        if (tid % 64 == 0) wsum64[tid / 64] = before;
        __syncthreads();
        for (unsigned w = 0; w < kWaves; ++w) seg_base += wsum64[w];
        seg_base = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(seg_base >> 32)) << 32) |
                   (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)seg_base);
    }
    if (MODE != FS_BYTES && seg == 0 && tid == 0) oseg[0] = 0;
    const bool fits = seg_base <= cap && seg_total <= cap - seg_base;
    if (!(st.before & kMalformed) && given_ok) {
        const bool emit = EMIT && fits;
        if (EMIT && !fits && tid == 0) atomicOr(err, kErrCap);
        uint32_t done = 0;     // decoded bytes of the chunks before
        uint32_t end_rel = 0;  // this string's end
        for (uint32_t c0 = 0; c0 < g.n; c0 += kChunk) {
            if (c0) r = open_granule(g, c0, tid), sz = r.lim ? size_at[r.q0 / kShare] : 0u;
            const uint32_t size = sz & kSize;
            const bool     esc  = (st.before & kEscapes) != 0;  // uniform
            if (esc) {
                ends[tid] = 0u;
                if (tid == 0) ends[kSeg] = 0u;
            }
            uint32_t total;
            const uint32_t at = block_exclusive_scan(size, wsum, &total);
            total             = __builtin_amdgcn_readfirstlane(total);  // the same in every lane: scalar from here on
            if (total > seg_total - done) {  // never more than what the capacity was tested with
                if (tid == 0) atomicOr(err, kErrCap);
                total = (uint32_t)(seg_total - done);
            }
            if constexpr (MODE != FS_BYTES) sbase[tid] = at;
            if (esc) {
                const uint32_t e = end[tid] - c0;
                if (e <= kChunk) atomicOr(&ends[e / kShare], 1u << (e % kShare));
                __syncthreads();
            }
            Escapes es {0, 0};
            if (sz & kSpecial)
                es = find_escapes(ff_mask(r.wd), Ends {ends[tid], (ends[tid + 1] & 1u) != 0}, r.lim, sz & kLiteral);
            else if (r.lim < kShare) es.none = ~0u << r.lim;
            const bool drops = es.none != 0;
            if (drops) static_for<8>([&](auto d) { r.wd[d] |= spread4(es.none >> (4 * decltype(d)::value)); });
            // the image starts at the output's place within 16 bytes; windows of it while the chunk has more (offsets
            // alone: the words are dropped)
            uint8_t* const dst = out + seg_base + done;
            const uint32_t sh  = EMIT ? (uint32_t)((uintptr_t)dst & 15u) : 0u;
            bool           ends_done = MODE == FS_BYTES;
            for (uint32_t w0 = 0; w0 < total || !ends_done;) {  // bytes [w0, w1) of the chunk, whole granules
                uint32_t w1 = total;
                if (total - w0 > kOutLds) {  // uniform
                    if (tid == 0) window = total;
                    __syncthreads();
                    if (at >= w0 && at + size - w0 > kOutLds) atomicMin(&window, at);
                    __syncthreads();
                    w1 = __builtin_amdgcn_readfirstlane(window);
                }
                const bool mine = at >= w0 && at + size <= w1 && r.lim;
                // the last word may have no byte that completes it
                if (tid == 0) *reinterpret_cast<uint64_t*>(image + ((sh + w1 - w0) & ~7u)) = 0ull;
                Emit o {image, 0ull, 8 * (sh + at - w0)};
                if (mine) {
                    uint32_t lk[8];
                    if constexpr (!EMIT) {  // lengths alone
                        if (__any(drops)) emit_granule<2, true>(r.wd, es.none, sym, len, o, lk);
                        else emit_granule<2, false>(r.wd, 0u, sym, len, o, lk);
                    } else if (__any(drops)) {
                        if (kind == 0) emit_granule<0, true>(r.wd, es.none, sym, len, o, lk);
                        else if (kind == 1) emit_granule<1, true>(r.wd, es.none, sym, len, o, lk);
                        else emit_granule<2, true>(r.wd, es.none, sym, len, o, lk);
                    } else {
                        if (kind == 0) emit_granule<0, false>(r.wd, 0u, sym, len, o, lk);
                        else if (kind == 1) emit_granule<1, false>(r.wd, 0u, sym, len, o, lk);
                        else emit_granule<2, false>(r.wd, 0u, sym, len, o, lk);
                    }
                    granule_prefix(lk, pre + kShare * tid);
                }
                __syncthreads();
                if (mine && EMIT) {
                    if (o.at & 63u)
                        atomicOr(reinterpret_cast<unsigned long long*>(image + ((o.at >> 3) & ~7u)), (unsigned long long)o.acc);
                    for (uint32_t m = es.esc; m; m &= m - 1) {  // the escapes' bytes, 0 so far
                        const uint32_t j = (uint32_t)__builtin_ctz(m), b = sh + at - w0 + pre[kShare * tid + j];
                        atomicOr(reinterpret_cast<uint32_t*>(image + (b & ~3u)),
                                 (uint32_t)g.seg[r.q0 + j + 1] << (8 * (b & 3u)));
                    }
                }
                if (!ends_done && w1 == total) {  // every granule's prefix is there
                    const uint32_t e = end[tid];
                    if (e >= c0 && e - c0 < kChunk && e < g.n) end_rel = done + sbase[(e - c0) / kShare] + pre[e - c0];
                    ends_done = true;
                }
                __syncthreads();
                if (emit) {
                    // copy-out: whole 16-byte words of the output, then the bytes before the first and after the last
                    uint8_t*       base0 = dst - sh + w0;  // image byte 0
                    const uint32_t lo = sh, hi = sh + w1 - w0, lo16 = (lo + 15) & ~15u, hi16 = hi & ~15u;
                    for (uint32_t k = lo16 + 16 * tid; k < hi16; k += 16 * kSeg)
                        *reinterpret_cast<v4u_ua*>(base0 + k) = *reinterpret_cast<const v4u*>(image + k);
                    const uint32_t head = lo16 < hi ? lo16 : hi, tail = hi16 > head ? hi16 : head;
                    if (lo + tid < head) base0[lo + tid] = image[lo + tid];
                    if (tail + tid < hi) base0[tail + tid] = image[tail + tid];
                }
                w0 = w1;
                if (w0 >= total) break;
                __syncthreads();  // the image is free again
            }
            done += total;
            if (g.n - c0 > kChunk) __syncthreads();  // pre, sbase and the scan's sums are free again
        }
        if (end[tid] == g.n) end_rel = done;
        if constexpr (MODE != FS_BYTES) oseg[tid + 1] = seg_base + end_rel;
    } else {
        // per string: malformed offsets (clamped, so that every read stays inside the vector), or the caller's offsets
        // do not fit the segment
        __syncthreads();
        const uint32_t stop_c = end[tid] + st.s0, s_in = tid ? end[tid - 1] + st.s0 : st.s0, s = s_in < stop_c ? s_in : stop_c;
        uint64_t       w0, stop;
        if (MODE != FS_BYTES || given_ok) {
            const uint64_t tot = string_length(cb, s, stop_c, len);
            uint64_t       all;
            w0   = seg_base + block_exclusive_scan(tot, wsum64, &all);
            stop = w0 + tot;
            if constexpr (MODE != FS_BYTES) oseg[tid + 1] = stop;
        } else {
            w0 = oseg[tid], stop = oseg[tid + 1];  // the caller's offsets, string by string
        }
        if constexpr (EMIT) {
            if (stop > cap || stop < w0) atomicOr(err, kErrCap);
            else decode_string_global(cb, s, stop_c, table, out, w0, stop);
        }
    }
}

__global__ void k_zero_first(uint64_t* offsets) { offsets[0] = 0; }

template <int MODE>
int launch_pages(const Column& col, StringPlan& sp, const uint8_t* dev_enc, uint64_t* dev_offsets, uint8_t* dev_bytes,
                 uint64_t cap, hipStream_t s) {
    auto* const     segs  = static_cast<FsstSeg*>(sp.d_segs);
    uint64_t* const vecs  = sp.d_vecs;
    uint64_t* const bases = sp.n_vec > kDirect ? vecs + sp.n_vec : nullptr;
    for (size_t i = 0; i < col.pages.size(); ++i) {
        const PageEntry& pe = col.pages[i];
        if (!pe.vec_c) continue;
        const bool wide = pe.vec_c <= kWideCount;
        hipLaunchKernelGGL(wide ? k_fsst_count<4> : k_fsst_count<1>, dim3(pe.vec_c), dim3(wide ? 4 * kSeg : kSeg), 0, s,
                           dev_enc + pe.page_off, pe.page_off, sp.d_tables + i, pe.out_index / kSeg, segs, vecs, sp.d_ends,
                           sp.d_sizes);
    }
    if (bases && MODE != FS_BYTES) hipLaunchKernelGGL(k_fsst_scan, dim3(1), dim3(1024), 0, s, vecs, bases, (uint32_t)sp.n_vec);
    for (size_t i = 0; i < col.pages.size(); ++i) {
        const PageEntry& pe = col.pages[i];
        if (!pe.vec_c) continue;
        hipLaunchKernelGGL(k_fsst<MODE>, dim3(pe.vec_c * kSegPerV), dim3(kSeg), 0, s, dev_enc + pe.page_off, pe.page_off,
                           sp.d_tables + i, pe.out_index, dev_offsets, dev_bytes, cap, sp.d_err, segs, vecs, bases,
                           sp.d_ends, sp.d_sizes, pe.out_index / kSeg);
    }
    if (MODE != FS_BYTES && col.n_values == 0) {
        // offsets[0] of an empty column, by a kernel: a memset node recorded into a caller's captured graph is not
        // reliable on replay
        hipLaunchKernelGGL(k_zero_first, dim3(1), dim3(1), 0, s, dev_offsets);
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? FLS_OK : hip_fail(e, "kernel launch");
}

}  // namespace

int strings_prepare(const Column& col, const uint8_t* host, StringPlan& sp) {
    (void)host;
    std::vector<FsstTableDev> tabs(col.pages.size());
    for (size_t i = 0; i < col.pages.size(); ++i) {
        std::memset(&tabs[i], 0, sizeof(FsstTableDev));
        unsigned max_len = 0;
        for (int c = 0; c < 255; ++c) {
            // bytes beyond a symbol's length must be zero: the decoder ORs whole symbols into its output words
            const unsigned l = col.pages[i].fsst.len[c];
            uint64_t       x = col.pages[i].fsst.symbol[c];
            if (l < 8) x &= (1ull << (8 * l)) - 1;
            tabs[i].symbol[c] = x, tabs[i].len[c] = (uint8_t)l;
            max_len = std::max(max_len, l);
        }
        FsstTableDev& t = tabs[i];
        t.len[255]      = 1;  // an escape emits one byte
        t.kind          = max_len <= 3 ? 0 : max_len <= 7 ? 1 : 2;
        for (int c = 0; c < 256; ++c)
            t.packed[c] = t.kind == 0   ? t.symbol[c] | (uint64_t)(8 * t.len[c]) << 32
                          : t.kind == 1 ? t.symbol[c] | (uint64_t)t.len[c] << 56
                                        : t.symbol[c];
    }
    sp.n_vec           = col.n_values / 1024;
    const uint64_t nsg = sp.n_vec * kSegPerV;
    hipError_t     e;
    if ((e = hipMalloc(&sp.d_tables, tabs.size() * sizeof(FsstTableDev) + 1)) != hipSuccess) return hip_fail(e, "hipMalloc");
    if ((e = hipMemcpy(sp.d_tables, tabs.data(), tabs.size() * sizeof(FsstTableDev), hipMemcpyHostToDevice)) != hipSuccess)
        return hip_fail(e, "hipMemcpy");
    if ((e = hipMalloc(&sp.d_segs, nsg * sizeof(FsstSeg) + 1)) != hipSuccess) return hip_fail(e, "hipMalloc");
    if ((e = hipMalloc(&sp.d_vecs, 2 * sp.n_vec * sizeof(uint64_t) + 1)) != hipSuccess) return hip_fail(e, "hipMalloc");
    if ((e = hipMalloc(&sp.d_ends, nsg * kSeg * sizeof(uint32_t) + 1)) != hipSuccess) return hip_fail(e, "hipMalloc");
    if ((e = hipMalloc(&sp.d_sizes, (col.size / kShare + nsg + 1) * sizeof(uint16_t))) != hipSuccess) return hip_fail(e, "hipMalloc");
    if ((e = hipMalloc(&sp.d_err, 4)) != hipSuccess) return hip_fail(e, "hipMalloc");
    if ((e = hipMemset(sp.d_err, 0, 4)) != hipSuccess) return hip_fail(e, "hipMemset");
    return FLS_OK;
}

void strings_release(StringPlan& sp) {
    if (sp.d_tables) (void)hipFree(sp.d_tables);
    if (sp.d_segs) (void)hipFree(sp.d_segs);
    if (sp.d_ends) (void)hipFree(sp.d_ends);
    if (sp.d_vecs) (void)hipFree(sp.d_vecs);
    if (sp.d_sizes) (void)hipFree(sp.d_sizes);
    if (sp.d_err) (void)hipFree(sp.d_err);
    sp = StringPlan {};
}

int strings_offsets(const Column& col, StringPlan& sp, const uint8_t* dev_enc, uint64_t* dev_offsets, hipStream_t s) {
    return launch_pages<FS_OFFSETS>(col, sp, dev_enc, dev_offsets, nullptr, 0, s);
}

int strings_decode(const Column& col, StringPlan& sp, const uint8_t* dev_enc, const uint64_t* dev_offsets,
                   uint8_t* dev_bytes, uint64_t cap, hipStream_t s) {
    return launch_pages<FS_BYTES>(col, sp, dev_enc, const_cast<uint64_t*>(dev_offsets), dev_bytes, cap, s);
}

int strings_decode_all(const Column& col, StringPlan& sp, const uint8_t* dev_enc, uint64_t* dev_offsets,
                       uint8_t* dev_bytes, uint64_t cap, hipStream_t s) {
    return launch_pages<FS_ALL>(col, sp, dev_enc, dev_offsets, dev_bytes, cap, s);
}

int strings_check(StringPlan& sp, hipStream_t s) {
    uint32_t   h = 0;
    hipError_t e = hipMemcpyAsync(&h, sp.d_err, 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return hip_fail(e, "check");
    return h ? fail(FLS_E_DATA, "string offsets exceed the output capacity") : FLS_OK;
}

}  // namespace fls
