// k_wave.hip -- one wave per vector, output order straight from the packed rows: integer pages of 64-bit values, RLE
// and dictionary pages of 32/64-bit values (k_wave_rle and k_wave_dict, below).
//
// Integer pages. The wave stages its vector's packed rows in LDS (16-byte chunks, loaded one vector ahead) and then every lane takes
// the output positions that it will store: iteration k, lane l holds values 128 k + 2 l and the next, which are positions
// p = 2 (l % 32) and p + 1 of FastLanes lane 2 k + l / 32, so a store instruction writes 1 KiB of consecutive output and
// nothing is staged on the way out. p does not depend on k: a lane's two bit offsets, LDS addresses and shifts are set
// once per vector, and an iteration reads them at a constant 16 bytes further (the rows of FastLanes lanes i and i + 2
// are 16 bytes apart). DELTA scans the differences over the 32 lanes of a half wave.
//
// The form that this replaces gave a thread a whole FastLanes lane (64 values by a compile-time bit width, through 34 KB
// of LDS per wave, so four waves per compute unit): 113.9 us for 65536 vectors of int64 timestamps (DELTA, bit width 7;
// 537 MB out, 69 MB in), 103.0 us here, 5.9 TB/s against 6.9 of a fill. A predicate on 32768 FFOR vectors of bit width
// 17, where the old form staged every value in LDS to compare it: 68.9 us, 30.1 us here. Blocks of two waves measured
// best from 32768 vectors on (DELTA: 103.5 us, four waves 106.5, eight 111.7).
//
// Bit widths are run-time values (uniform over the wave). Rows sit 144 bytes apart in LDS, so that the eight rows that
// the lanes of an instruction read at small bit widths are on different banks; a value is cut from two dwords (bit
// widths up to 32) or three.
// Page layout and expressions: page_kernels.hpp (int_meta).
#include "launch.hpp"
#include "page_kernels.hpp"

namespace fls {
namespace {

constexpr unsigned kRow    = 144;  // LDS bytes per packed row of 128
constexpr unsigned kAhead  = 4;    // 16-byte chunks per lane loaded ahead: bit widths up to 32
constexpr unsigned kLbRows = 128;  // LDS bytes of a DELTA vector's lane bases

// Inclusive sum over the first 32 lanes or the last 32 (WAVE: over all 64).
template <bool WAVE>
__device__ __forceinline__ uint32_t lane_scan(uint32_t x) {
    x += __builtin_amdgcn_update_dpp(0u, x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0u, x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0u, x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0u, x, 0x118, 0xf, 0xf, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0u, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    if constexpr (WAVE) x += __builtin_amdgcn_update_dpp(0u, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
    return x;
}
template <bool WAVE>
__device__ __forceinline__ uint64_t lane_scan(uint64_t x) {
    const unsigned lane = threadIdx.x % 64;
    for (unsigned d = 1; d < (WAVE ? 64 : 32); d <<= 1) {
        const uint64_t y = __shfl_up((unsigned long long)x, d, WAVE ? 64 : 32);
        if ((WAVE ? lane : lane % 32) >= d) x += y;
    }
    return x;
}

template <typename T>
__device__ __forceinline__ T uniform(T x) {
    if constexpr (sizeof(T) == 8)
        return (T)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)x >> 32)) << 32) |
                   (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)x));
    else return (T)__builtin_amdgcn_readfirstlane((uint32_t)x);
}

// Packed rows of a vector: the first kAhead chunks of every lane, in flight while the vector before is decoded.
struct Ahead {
    v4u c[kAhead];
};
__device__ __forceinline__ void load_ahead(const uint8_t* pk, uint32_t chunks, unsigned lane, Ahead& a) {
    static_for<kAhead>([&](auto k) {
        const uint32_t c = lane + 64u * decltype(k)::value;
        if (c < chunks) a.c[k] = ld16(pk + 16 * c);
    });
}
__device__ __forceinline__ uint32_t row_place(uint32_t c) { return (c >> 3) * kRow + (c & 7) * 16; }
__device__ __forceinline__ void stage_rows(const uint8_t* pk, uint32_t chunks, unsigned lane, const Ahead& a, uint8_t* rows) {
    static_for<kAhead>([&](auto k) {
        const uint32_t c = lane + 64u * decltype(k)::value;
        if (c < chunks) *reinterpret_cast<v4u*>(rows + row_place(c)) = a.c[k];
    });
    for (uint32_t c = lane + 64u * kAhead; c < chunks; c += 64u) *reinterpret_cast<v4u*>(rows + row_place(c)) = ld16(pk + 16 * c);
}

// LDS bytes of a wave of k_wave_rle: (lane base, differences) pairs and up to 1024 run values.
__host__ __device__ constexpr unsigned rle_wave_lds(unsigned value_bytes) { return 256 + 1024 * value_bytes; }

// MODE 0 UNCOMPRESSED, 1 FFOR, 2 DELTA, as k_page_int. SEL: a predicate's bitmap instead of values; iteration k, lane l
// then holds value 64 k + l alone, so that a ballot is the bitmap's word k.
template <int MODE, bool NT, bool SEL>
__global__ __launch_bounds__(kMaxBlock) void k_wave_int64(const uint8_t* __restrict__ page, WaveMeta pm, uint32_t vec_c,
                                                          uint8_t* __restrict__ out, SelArgs sa, uint32_t wave_lds) {
    extern __shared__ __attribute__((aligned(16))) uint8_t fls_lds[];
    constexpr unsigned P  = MODE == 0 ? 0 : (MODE == 2 ? 3 : 2);
    constexpr unsigned NV = SEL ? 1 : 2, IT = 16 / NV;  // values per lane and iteration, iterations
    const unsigned     lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    uint8_t* const     lb   = fls_lds + wave * wave_lds;  // DELTA lane bases, then the rows
    uint8_t* const     rows = lb + (MODE == 2 ? kLbRows : 0);
    const unsigned     p    = SEL ? lane : 2 * (lane % 32), half = SEL ? 0 : lane / 32;
    const unsigned     j    = 8 * (p % 8) + order8(p / 8);
    const uint64_t     N = vec_c, stride = (uint64_t)gridDim.x * (blockDim.x / 64);
    uint64_t           v = (uint64_t)blockIdx.x * (blockDim.x / 64) + wave;
    auto meta   = [&](uint64_t u) { return int_meta<64, MODE>(page, pm, u, lane % 16); };
    // (never more rows than the launch's LDS was sized for, whatever the page holds)
    auto width  = [&](const IntMeta& m) -> uint32_t { return MODE == 0 ? 64u : min(uniform(m.bw), pm.bw_max); };
    auto packed = [&](const IntMeta& m) { return page + pm.off[P] + uniform(m.ep); };
    IntMeta m0 {}, m1 {};
    Ahead   a;
    if (v < N) {
        m0 = meta(v);
        load_ahead(packed(m0), 8 * width(m0), lane, a);
    }
    if (v + stride < N) m1 = meta(v + stride);
    for (; v < N; v += stride) {
        const uint32_t bw   = width(m0);
        const uint64_t base = MODE == 0 ? 0ull : uniform(m0.base);
        stage_rows(packed(m0), 8 * bw, lane, a, rows);
        if constexpr (MODE == 2)
            if (lane < 16) reinterpret_cast<uint64_t*>(lb)[lane] = m0.lb;
        m0 = m1;
        if (v + stride < N) load_ahead(packed(m0), 8 * width(m0), lane, a);
        if (v + 2 * stride < N) m1 = meta(v + 2 * stride);
        wave_sync();
        // a lane's values start at bit j * bw (and (j + 8) * bw) of their FastLanes lane: dword d of it sits in row
        // d / 2, and dword d + 2 one row further
        const uint8_t* at[NV];
        int32_t        next[NV];
        uint32_t       sh[NV];
        static_for<NV>([&](auto e) {
            const uint32_t bit = (j + 8 * decltype(e)::value) * bw, d = bit >> 5;
            at[e]              = rows + (d >> 1) * kRow + 4 * (d & 1) + 8 * half;
            next[e]            = d & 1 ? (int32_t)kRow - 4 : 4;
            sh[e]              = bit & 31;
        });
        const uint64_t mask = bw >= 64 ? ~0ull : ((1ull << bw) - 1);
        uint64_t       word = 0;
        uint32_t       cnt  = 0;
        auto           done = [&](auto k, const uint64_t (&x)[NV]) {
            if constexpr (SEL) {
                const uint64_t b = __ballot(sa.dbl ? sel_pred<uint64_t, true>(x[0], sa) : sel_pred<uint64_t, false>(x[0], sa));
                if (lane == decltype(k)::value) word = b;
                cnt += (uint32_t)__popcll(b);
            } else {
                st16<NT>(out + v * 8192 + 1024 * k + 16 * lane, v4u {(uint32_t)x[0], (uint32_t)(x[0] >> 32), (uint32_t)x[NV - 1],
                                                                    (uint32_t)(x[NV - 1] >> 32)});
            }
        };
        constexpr unsigned SB = SEL ? 8 : 16;  // LDS bytes between the rows of an iteration and the next
        auto dword = [&](const uint8_t* q) { return *reinterpret_cast<const uint32_t*>(q); };
        if (MODE == 2 && bw <= 26) {
            // 64 differences sum to less than 2^32 without their base, which is added p + 1 times
            uint64_t pb[NV];
            static_for<NV>([&](auto e) { pb[e] = base * (p + 1 + decltype(e)::value); });
            static_for<IT>([&](auto k) {
                uint32_t u[NV];
                static_for<NV>([&](auto e) {
                    u[e] = __builtin_amdgcn_alignbit(dword(at[e] + SB * k + next[e]), dword(at[e] + SB * k), sh[e]) & (uint32_t)mask;
                });
                const uint32_t s = lane_scan<SEL>(NV == 2 ? u[0] + u[NV - 1] : u[0]);
                const uint64_t b = *reinterpret_cast<const uint64_t*>(lb + SB * k + 8 * half);
                uint64_t       x[NV];
                if constexpr (NV == 2) x[0] = b + pb[0] + (s - u[1]);
                x[NV - 1] = b + pb[NV - 1] + s;
                done(k, x);
            });
        } else {
            static_for<IT>([&](auto k) {
                uint64_t x[NV];
                static_for<NV>([&](auto e) {
                    const uint32_t lo = dword(at[e] + SB * k), mid = dword(at[e] + SB * k + next[e]);
                    const uint32_t a0 = __builtin_amdgcn_alignbit(mid, lo, sh[e]);
                    uint32_t       a1 = 0;
                    if (bw > 32) a1 = __builtin_amdgcn_alignbit(dword(at[e] + SB * k + kRow), mid, sh[e]);
                    x[e] = (((uint64_t)a1 << 32 | a0) & mask) + base;
                });
                if constexpr (MODE == 2) {
                    const uint64_t s = lane_scan<SEL>(NV == 2 ? x[0] + x[NV - 1] : x[0]);
                    const uint64_t b = *reinterpret_cast<const uint64_t*>(lb + SB * k + 8 * half);
                    if constexpr (NV == 2) x[0] = b + s - x[1];
                    x[NV - 1] = b + s;
                }
                done(k, x);
            });
        }
        if constexpr (SEL) {
            if (lane < 16) sa.bitmap[v * 16 + lane] = word;
            if (lane == 0) sa.counts[v] = cnt;
        }
        wave_sync();
    }
}

// RLE pages of 32/64-bit values whose positions have bit width 0 or 1 (as k_page_rle_lanes: every page the encoders
// write). A position lane's 16 differences are one u16 word, so position p of lane i is its lane base plus a bit
// count of the word under a mask that depends on p alone. The wave puts the 64 lanes' (base, word) pairs and the
// vector's run values into LDS, and every lane takes the positions that it will store: value o lies in lane
// (o / 64) + 16 ord4(o / 16 % 4) at p = o % 16, so its masks are set once and an iteration reads the pair at a constant
// offset. The run values of the next vector (the first 256) and the metadata of the one after are in flight meanwhile.
// The form before (k_page_rle, which still serves plain positions and wider differences) decoded two position lanes a
// thread by a compile-time bit width and staged every value in LDS on its way out: 89.5 us for 65536 vectors of uint32
// with runs of 16 (268 MB out, 35 MB in), 47.6 us here, 6.4 TB/s; 64-bit values 66.6 and 44.5 us (32768 vectors), runs
// of two 101 and 83 us; a predicate on 65536 vectors of uint32 73.9 and 52.0 us.
constexpr unsigned kRunsAhead = 4;

template <typename T, bool NT, bool SEL>
__global__ __launch_bounds__(kMaxBlock) void k_wave_rle(const uint8_t* __restrict__ page, PageMeta pm, uint32_t vec_c,
                                                        uint8_t* __restrict__ out, uint32_t* err, SelArgs sa, RunSrc rs) {
    extern __shared__ __attribute__((aligned(16))) uint8_t fls_lds[];
    constexpr unsigned NV = SEL ? 1 : 16 / sizeof(T), IT = 16 / NV;  // values per lane and iteration, iterations
    const unsigned     lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    uint32_t* const    pair = reinterpret_cast<uint32_t*>(fls_lds + wave * rle_wave_lds(sizeof(T)));
    T* const           lr   = reinterpret_cast<T*>(pair + 64);
    const unsigned     q = NV * lane, p = q % 16;
    const uint32_t*    at = pair + q / 64 + 16 * ord4(q / 16 % 4);
    uint32_t           M[NV];  // the differences up to the lane's value e, in the high half (prefix_mask16)
    static_for<NV>([&](auto e) {
        const unsigned n = p + decltype(e)::value;
        M[e] = (n < 8 ? 0x5555u & ((2u << (2 * n)) - 1) : 0x5555u | (0xaaaau & ((4u << (2 * (n - 8))) - 1))) << 16;
    });
    const uint64_t N = vec_c, stride = (uint64_t)gridDim.x * (blockDim.x / 64);
    uint64_t       v = (uint64_t)blockIdx.x * (blockDim.x / 64) + wave;
    auto meta = [&](uint64_t u) {
        RleMeta r = rle_meta<2>(page, pm, u, N, lane >> 1, rs.bytes, rs.lbase);
        r.lb      = (r.lb >> (16 * (lane & 1))) & 0xffffu;  // rle_meta reads the u32 of lanes 2t, 2t + 1
        r.r0 = uniform(r.r0), r.r1 = uniform(r.r1), r.bw = uniform(r.bw), r.base = uniform(r.base) & 0xffffu, r.ep = uniform(r.ep);
        return r;
    };
    auto word = [&](const RleMeta& r) {  // the lane's differences
        return r.bw ? (uint32_t)*reinterpret_cast<const u16_ua*>(page + pm.off[4] + r.ep + 2 * lane) : 0u;
    };
    auto n_of    = [&](const RleMeta& r) { return (r.r1 - r.r0) >> rs.esh; };
    auto runs_of = [&](const RleMeta& r) { return rs.base + (uint64_t)(r.r0 >> rs.esh) * sizeof(T); };
    auto load_runs = [&](const RleMeta& r, T (&dst)[kRunsAhead]) {
        const uint8_t* rp = runs_of(r);
        const uint32_t n  = n_of(r);
        static_for<kRunsAhead>([&](auto k) {
            const uint32_t i = lane + 64 * decltype(k)::value;
            if (i < n) dst[k] = load_t<T>(rp + (uint64_t)i * sizeof(T));
        });
    };
    RleMeta  m0 {}, m1 {};
    uint32_t w0 = 0, w1 = 0;
    T        ahead[kRunsAhead];
    if (v < N) m0 = meta(v), w0 = word(m0), load_runs(m0, ahead);
    if (v + stride < N) m1 = meta(v + stride), w1 = word(m1);
    for (; v < N; v += stride) {
        const uint32_t n = n_of(m0), last = n - 1, base = m0.base;
        const uint8_t* rp = runs_of(m0);
        // the largest position of the lane before a u16 wrap, were there one
        const uint32_t top = m0.lb + 16 * base + (uint32_t)__builtin_popcount(w0);
        const bool     plain = n && base == 0 && n <= 1024 && !__any(top > last);  // (n = 0: no position is in range)
        pair[lane] = m0.lb | w0 << 16;
        static_for<kRunsAhead>([&](auto k) {
            const uint32_t i = lane + 64 * decltype(k)::value;
            if (i < n) lr[i] = ahead[k];
        });
        if (n > 64 * kRunsAhead)
            for (uint32_t i = lane + 64 * kRunsAhead; i < n && i < 1024; i += 64) lr[i] = load_t<T>(rp + (uint64_t)i * sizeof(T));
        m0 = m1, w0 = w1;
        if (v + stride < N) load_runs(m0, ahead);
        if (v + 2 * stride < N) m1 = meta(v + 2 * stride), w1 = word(m1);
        wave_sync();
        uint64_t bits = 0;
        uint32_t cnt  = 0;
        auto     decode = [&](auto value) {
            static_for<IT>([&](auto k) {
                const uint32_t x = at[NV * decltype(k)::value];
                T              vals[NV];
                static_for<NV>([&](auto e) { vals[e] = value((x & 0xffffu) + (uint32_t)__builtin_popcount(x & M[e]), e); });
                if constexpr (SEL) {
                    const uint64_t b = __ballot(sizeof(T) == 8 && sa.dbl ? sel_pred<T, true>(vals[0], sa) : sel_pred<T, false>(vals[0], sa));
                    if (lane == decltype(k)::value) bits = b;
                    cnt += (uint32_t)__popcll(b);
                } else {
                    st16<NT>(out + v * (1024 * sizeof(T)) + 1024 * decltype(k)::value + 16 * lane, *reinterpret_cast<const v4u*>(vals));
                }
            });
        };
        if (plain) {
            decode([&](uint32_t pos, auto) { return lr[pos]; });
        } else if (n) {  // a FFOR base, positions that wrap or leave the runs (clamped, reported), more runs than LDS holds
            bool bad = false;
            decode([&](uint32_t pos, auto e) {
                pos = (pos + (p + decltype(e)::value + 1) * base) & 0xffffu;
                bad |= pos > last;
                pos = pos < last ? pos : last;
                return n <= 1024 ? lr[pos] : load_t<T>(rp + (uint64_t)pos * sizeof(T));
            });
            if (bad) atomicOr(err, 1u);
        } else if (lane == 0) {  // the host rejects such pages; never read an empty run buffer
            atomicOr(err, 1u);
        }
        if constexpr (SEL) {
            if (lane < 16) sa.bitmap[v * 16 + lane] = bits;
            if (lane == 0) sa.counts[v] = cnt;
        }
        wave_sync();
    }
}

// Dictionary pages of 32/64-bit values: u32 codes (VAR 1 raw, 2 FFOR, 7 DELTA; dict_vector has the layout), out[i] = dict[code[i]]. As
// k_wave_int64, with the codes' rows of 32 lanes: value o is position p = o % 32 of code lane o / 64 + 16 (o / 32 % 2).
// A lane holds the 16 bytes that it stores, NV values from one code lane, and gathers them from the dictionary: IN_LDS,
// every block first copies it there or (hz.chunks) decodes its HZL chunks into it; else from L2. DELTA sums over the
// 32 / NV lanes that share a code lane. The form before decoded a code lane a thread by a compile-time bit width and
// staged every value in LDS on its way out: 97.2 us for 65536 vectors of int32 with 4096 keys (two pages; 268 MB out,
// 101 MB in), 76.6 us here; 60000 keys (from L2) 186 and 121 us; DELTA codes 158 and 117 us; 32768 vectors of int64 with
// 2000 keys 99.8 and 61.0 us, with 40000 101.7 and 75 us; 2000 vectors of int32 10.7 and 7.0 us. What is left over a copy's
// rate is the start of each page (metadata, rows and dictionary are loads that wait for each other).
// A predicate takes the same lanes, whose bits are joined across the 8 or 16 lanes of a bitmap dword; a dictionary in LDS is
// tested once as it is filled and holds outcomes instead of values. With a value per lane and a ballot per 64 of them, it
// took longer than the form before on large pages: 16384 vectors of int32, 50 sorted keys, 13.9 us then, 21.4, 12.1 now (FFOR
// codes; DELTA codes 15.5, 26.0, 13.9); 4096 Zipf keys 24.9, 24.8, 17.1; 30000 sorted keys (from L2, DELTA codes) 18.4, 22.1,
// 17.8.
template <unsigned G>
__device__ __forceinline__ uint32_t group_scan(uint32_t x, unsigned lane) {  // inclusive, over groups of G lanes
    if constexpr (G == 32) return lane_scan<false>(x);
    static_for<4>([&](auto d) {
        constexpr unsigned n = 1u << decltype(d)::value;
        if constexpr (n < G) {
            const uint32_t y = __builtin_amdgcn_update_dpp(0u, x, 0x110 + n, 0xf, 0xf, false);  // row_shr
            x += lane % G >= n ? y : 0u;
        }
    });
    return x;
}

// OR over groups of 8 or 16 lanes.
template <unsigned G>
__device__ __forceinline__ uint32_t group_or(uint32_t x) {
    x |= __builtin_amdgcn_update_dpp(0u, x, 0xb1, 0xf, 0xf, false);   // quad_perm 1 0 3 2
    x |= __builtin_amdgcn_update_dpp(0u, x, 0x4e, 0xf, 0xf, false);   // quad_perm 2 3 0 1
    x |= __builtin_amdgcn_update_dpp(0u, x, 0x141, 0xf, 0xf, false);  // half mirror
    if constexpr (G == 16) x |= __builtin_amdgcn_update_dpp(0u, x, 0x140, 0xf, 0xf, false);  // mirror
    return x;
}

// A block decodes a dictionary's HZL chunks (no exceptions) into LDS, four values a thread at once: chunk headers, then
// packed words, are two rounds of loads for 2048 values. Full chunks hold 1024 values and the raw tail follows them.
// keep(v): what LDS keeps of value v.
template <typename D, typename F>
__device__ __forceinline__ void fill_dict(const HzlSrc& hz, uint32_t dict_n, D* ldict, F keep) {
    constexpr unsigned DW = 8 * sizeof(D), L = 1024 / DW;
    for (uint32_t b0 = 0; b0 < dict_n; b0 += 4 * blockDim.x) {
        D        lo[4], hi[4], base[4];
        uint32_t bw[4], sh[4];
        static_for<4>([&](auto u) {
            const uint32_t b = b0 + decltype(u)::value * blockDim.x;
            if (b >= dict_n) return;
            uint32_t g = b + threadIdx.x;
            g          = g < dict_n ? g : dict_n - 1;
            const uint32_t  c  = __builtin_amdgcn_readfirstlane(min(g >> 10, hz.n_chunks - 1)), k = g - (c << 10);
            const HzlChunk& ch = hz.chunks[c];
            const uint8_t*  in = hz.enc + ch.src;
            bw[u] = ch.bw, base[u] = (D)ch.base;
            const uint32_t bit = k / L * bw[u], w = bit / DW, lane = k % L;
            sh[u] = bit % DW;
            // the tail: value k as it stands; bit width 0: any bytes (the chunk's header) and an empty mask
            const uint32_t o0 = bw[u] == 255 ? k : w * L + lane, o1 = bw[u] == 255 ? k : (w + 1 < bw[u] ? w + 1 : w) * L + lane;
            const uint8_t* at = bw[u] ? in : in - 12;
            lo[u] = load_t<D>(at + (bw[u] ? (uint64_t)o0 * sizeof(D) : 0ull));
            hi[u] = load_t<D>(at + (bw[u] ? (uint64_t)o1 * sizeof(D) : 0ull));
        });
        static_for<4>([&](auto u) {
            const uint32_t b = b0 + decltype(u)::value * blockDim.x;
            if (b >= dict_n) return;
            D v = bw[u] == 255 ? lo[u] : (D)((lo[u] >> sh[u]) | (sh[u] ? hi[u] << (DW - sh[u]) : (D)0));
            if (bw[u] < DW) v &= ((D)1 << bw[u]) - 1;
            if (bw[u] != 255) v += base[u];
            if (b + threadIdx.x < dict_n) ldict[b + threadIdx.x] = keep(v);
        });
    }
}

template <typename T, int VAR, bool NT, bool IN_LDS, bool SEL>
__global__ __launch_bounds__(kMaxBlock) void k_wave_dict(const uint8_t* __restrict__ page, WaveMeta pm, uint32_t vec_c,
                                                         const T* __restrict__ dict, uint32_t dict_n,
                                                         uint8_t* __restrict__ out, uint32_t* err, SelArgs sa, HzlSrc hz,
                                                         uint32_t dict_lds, uint32_t wave_lds) {
    extern __shared__ __attribute__((aligned(16))) uint8_t fls_lds[];
    if (dict_n == 0) return;  // the host rejects such pages
    constexpr unsigned P  = VAR == 1 ? 0 : (VAR == 7 ? 3 : 2);
    constexpr unsigned NV = 16 / sizeof(T), IT = 16 / NV;  // values per lane and iteration, iterations
    constexpr unsigned GL = 32 / NV;                       // SEL: lanes that share a dword of the bitmap (at least IT)
    T* const ldict = reinterpret_cast<T*>(fls_lds);
    const unsigned lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    uint8_t* const lb   = fls_lds + dict_lds + wave * wave_lds;  // DELTA lane bases, then the rows
    uint8_t* const rows = lb + (VAR == 7 ? kLbRows : 0);
    const unsigned q = NV * lane, p = q % 32, col = q / 64 + 16 * (q / 32 % 2);  // an iteration on: NV code lanes further
    const uint32_t last = dict_n - 1;
    const uint64_t N = vec_c, stride = (uint64_t)gridDim.x * (blockDim.x / 64);
    uint64_t       v = (uint64_t)blockIdx.x * (blockDim.x / 64) + wave;
    auto meta   = [&](uint64_t u) { return code_meta<VAR>(page, pm, u, lane % 32); };
    auto width  = [&](const CodeMeta& m) -> uint32_t { return VAR == 1 ? 32u : min(uniform(m.bw), pm.bw_max); };
    auto packed = [&](const CodeMeta& m) { return page + pm.off[P] + uniform(m.ep); };
    CodeMeta m0 {}, m1 {};
    Ahead    a;
    bool     bad = false;
    if (v < N) {
        m0 = meta(v);
        load_ahead(packed(m0), 8 * width(m0), lane, a);
    }
    if (v + stride < N) m1 = meta(v + stride);
    if constexpr (IN_LDS) {
        auto keep = [&](T x) { return SEL ? (T)sel_pred<T, false>(x, sa) : x; };  // a predicate's outcome for each entry
        if (hz.chunks) fill_dict(hz, dict_n, ldict, keep);
        else
            for (uint32_t i = threadIdx.x; i < dict_n; i += blockDim.x) ldict[i] = keep(dict[i]);
        __syncthreads();
    }
    for (; v < N; v += stride) {
        const uint32_t bw   = width(m0);
        const uint32_t base = VAR == 1 ? 0u : uniform(m0.base);
        stage_rows(packed(m0), 8 * bw, lane, a, rows);
        if constexpr (VAR == 7)
            if (lane < 32) reinterpret_cast<uint32_t*>(lb)[lane] = m0.lb;
        m0 = m1;
        if (v + stride < N) load_ahead(packed(m0), 8 * width(m0), lane, a);
        if (v + 2 * stride < N) m1 = meta(v + 2 * stride);
        wave_sync();
        const uint32_t mask = bw >= 32 ? ~0u : (1u << bw) - 1;
        uint32_t       word = 0;  // SEL: the bitmap's dword 2 NV (lane % GL) + lane / GL
        const uint8_t* at[NV];    // the dword that the lane's first code e starts in; the next is a row further
        uint32_t       sh[NV];
        static_for<NV>([&](auto e) {
            const uint32_t bit = j_of_p<32>(p + decltype(e)::value) * bw;
            at[e]              = rows + (bit >> 5) * kRow + 4 * col;
            sh[e]              = bit & 31;
        });
        static_for<IT>([&](auto k) {
            constexpr unsigned S = 4 * NV * decltype(k)::value;
            auto     dword = [&](const uint8_t* r) { return *reinterpret_cast<const uint32_t*>(r + S); };
            uint32_t c[NV];
            T        vals[NV];
            static_for<NV>([&](auto e) { c[e] = (__builtin_amdgcn_alignbit(dword(at[e] + kRow), dword(at[e]), sh[e]) & mask) + base; });
            if constexpr (VAR == 7) {
                static_for<NV - 1>([&](auto e) { c[e + 1] += c[e]; });
                const uint32_t before = group_scan<32 / NV>(c[NV - 1], lane) - c[NV - 1] +
                                        *reinterpret_cast<const uint32_t*>(lb + S + 4 * col);
                static_for<NV>([&](auto e) { c[e] += before; });
            }
            static_for<NV>([&](auto e) {
                bad |= c[e] > last;
                c[e]    = min(c[e], last);
                vals[e] = IN_LDS ? ldict[c[e]] : dict[c[e]];
            });
            if constexpr (SEL) {
                uint32_t b = 0;  // the lane's values' bits in their dword, then all of the dword
                static_for<NV>([&](auto e) {
                    b |= (IN_LDS ? (uint32_t)vals[e] : (uint32_t)in_range<T>(vals[e], sa)) << decltype(e)::value;
                });
                b = group_or<GL>(b << (NV * (lane % GL)));
                if (lane % GL == decltype(k)::value) word = b;
            } else {
                st16<NT>(out + v * (1024 * sizeof(T)) + 1024 * decltype(k)::value + 16 * lane, *reinterpret_cast<const v4u*>(vals));
            }
        });
        if constexpr (SEL) {
            if (!IN_LDS) word = sa.none ? 0u - (uint32_t)(sa.none_val != 0) : word ^ (0u - (uint32_t)(sa.inv != 0));
            if (lane % GL >= IT) word = 0;
            else reinterpret_cast<uint32_t*>(sa.bitmap)[v * 32 + 2 * NV * (lane % GL) + lane / GL] = word;
            const uint32_t n = lane_scan<true>((uint32_t)__builtin_popcount(word));
            if (lane == 63) sa.counts[v] = n;
        }
        wave_sync();
    }
    if (bad) atomicOr(err, 2u);
}

}  // namespace

hipError_t page_int64_wave(int mode, const uint8_t* page, const WaveMeta& pm, uint32_t vec_c, uint8_t* out,
                           const SelArgs* sel, hipStream_t s) {
    Tune           t  = tune_for(mode == 0 ? FAM_PAGE_UNC : mode == 1 ? FAM_PAGE_FFOR : FAM_PAGE_DELTA, 64, 255);
    const unsigned bw = mode == 0 ? 64u : pm.bw_max ? pm.bw_max : 1u;
    const unsigned wl = (bw + 1) * kRow + (mode == 2 ? kLbRows : 0);  // a value's last dword may lie in the row after
    unsigned       waves = t.block / 64;
    while (waves > 1 && waves * wl > 65536) --waves;
    t.block            = (uint16_t)(64 * waves);
    const dim3     g(grid_for(vec_c, t, 64)), b(t.block);
    const SelArgs  sa = sel ? *sel : SelArgs {};
#define L(M, NT, SL) hipLaunchKernelGGL((k_wave_int64<M, NT, SL>), g, b, waves * wl, s, page, pm, vec_c, out, sa, wl)
#define LM(M)                      \
    if (sel) L(M, false, true);    \
    else if (t.nt & 1) L(M, true, false); \
    else L(M, false, false);
    if (mode == 0) {
        LM(0)
    } else if (mode == 1) {
        LM(1)
    } else {
        LM(2)
    }
#undef LM
#undef L
    return hipGetLastError();
}

template <typename T>
static hipError_t rle_wave(const uint8_t* page, const PageMeta& pm, uint32_t vec_c, uint8_t* out, uint32_t* err,
                           const SelArgs* sel, const RunSrc& rs, hipStream_t s) {
    Tune           t     = tune_for(FAM_PAGE_RLE, 8 * sizeof(T), 255);
    const unsigned wl    = rle_wave_lds(sizeof(T));
    unsigned       waves = t.block / 64;
    while (waves > 1 && waves * wl > 65536) --waves;
    t.block          = (uint16_t)(64 * waves);
    const dim3    g(grid_for(vec_c, t, 64)), b(t.block);
    const SelArgs sa = sel ? *sel : SelArgs {};
#define L(NT, SL) hipLaunchKernelGGL((k_wave_rle<T, NT, SL>), g, b, waves * wl, s, page, pm, vec_c, out, err, sa, rs)
    if (sel) L(false, true);
    else if (t.nt & 1) L(true, false);
    else L(false, false);
#undef L
    return hipGetLastError();
}
hipError_t page_rle_wave(unsigned W, const uint8_t* page, const PageMeta& pm, uint32_t vec_c, uint8_t* out, uint32_t* err,
                         const SelArgs* sel, const RunSrc* runs, hipStream_t s) {
    const RunSrc rs = runs ? *runs : RunSrc {page + pm.off[0], pm.off[1] - pm.off[0], W == 64 ? 3u : 2u};
    return W == 64 ? rle_wave<uint64_t>(page, pm, vec_c, out, err, sel, rs, s) : rle_wave<uint32_t>(page, pm, vec_c, out, err, sel, rs, s);
}

template <typename T>
static hipError_t dict_wave(int var, const uint8_t* page, const WaveMeta& pm, uint32_t vec_c, const void* dict, uint32_t dict_n,
                            uint8_t* out, uint32_t* err, const SelArgs* sel, const HzlSrc* hz, hipStream_t s) {
    const T*       d  = static_cast<const T*>(dict);
    Tune           t  = tune_for(FAM_PAGE_DICT, 8 * sizeof(T), 255);
    const unsigned bw = var == 1 ? 32u : pm.bw_max ? pm.bw_max : 1u;
    const unsigned wl = (bw + 1) * kRow + (var == 7 ? kLbRows : 0);
    // a dictionary of up to 32 KiB goes to LDS: a block's waves fit beside it
    const bool     in_lds = (uint64_t)dict_n * sizeof(T) <= 32768;
    const unsigned dl     = in_lds ? (dict_n * (unsigned)sizeof(T) + 15) & ~15u : 0u;
    unsigned       waves  = t.block / 64;
    while (waves > 1 && dl + waves * wl > 65536) --waves;
    t.block = (uint16_t)(64 * waves);
    // every block fills its own copy, so few blocks that stride over many vectors, the same number each (65536 vectors of
    // int32, 4096 keys: 256 blocks of 8 waves 76 us, 1024 80 us, a block per 8 vectors 84); without a copy no cap
    // (60000 keys: 121 us, 1536 blocks 150)
    if (!in_lds) t.max_blocks = 0;
    unsigned blocks = grid_for(vec_c, t, 64);
    if (t.max_blocks) {
        const uint64_t steps = (vec_c + (uint64_t)blocks * waves - 1) / ((uint64_t)blocks * waves);
        blocks               = (unsigned)((vec_c + steps * waves - 1) / (steps * waves));
    }
    const dim3    g(blocks), b(t.block);
    const SelArgs sa = sel ? *sel : SelArgs {};
    // without HZL exceptions every block decodes the chunks itself; otherwise the HZL kernels fill the global copy first
    const bool   fused = in_lds && hz && !hz->exc;
    const HzlSrc hs    = fused ? *hz : HzlSrc {};
    if (hz && !fused) {
        const hipError_t e = launch_hzl(8 * sizeof(T), hz->enc, hz->chunks, hz->n_chunks,
                                        reinterpret_cast<uint8_t*>(const_cast<T*>(d)), hz->exc != 0, s);
        if (e != hipSuccess) return e;
    }
#define L(V, NT, K, SL) \
    hipLaunchKernelGGL((k_wave_dict<T, V, NT, K, SL>), g, b, dl + waves * wl, s, page, pm, vec_c, d, dict_n, out, err, sa, hs, dl, wl)
#define LK(V, K)                    \
    if (sel) L(V, false, K, true);  \
    else if (t.nt & 1) L(V, true, K, false); \
    else L(V, false, K, false);
#define LV(V)        \
    if (in_lds) {    \
        LK(V, true)  \
    } else {         \
        LK(V, false) \
    }
    if (var == 1) {
        LV(1)
    } else if (var == 2) {
        LV(2)
    } else {
        LV(7)
    }
#undef LV
#undef LK
#undef L
    return hipGetLastError();
}
hipError_t page_dict_wave(unsigned W, int var, const uint8_t* page, const WaveMeta& pm, uint32_t vec_c, const void* dict,
                          uint32_t dict_n, uint8_t* out, uint32_t* err, const SelArgs* sel, const HzlSrc* hz, hipStream_t s) {
    return W == 64 ? dict_wave<uint64_t>(var, page, pm, vec_c, dict, dict_n, out, err, sel, hz, s)
                   : dict_wave<uint32_t>(var, page, pm, vec_c, dict, dict_n, out, err, sel, hz, s);
}

}  // namespace fls
