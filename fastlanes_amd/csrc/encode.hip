// encode.hip -- GPU encoder for integer columns: UNCOMPRESSED (pool id 0), FFOR (1), DELTA (11) and RLE (6, 7)
// pages, byte for byte what the host encoder (encode_from_memory) writes.
//
// Encode RPNs: UNCOMPRESSED {TRS, MEM_CPY} (include/fls/cor/exp/uncompressed/uncompressed_exp.hpp:32-47), FFOR
// {TRS, ANALYZE, FFOR} (include/fls/cor/exp/ffor/ffor_exp.hpp:39-46), DELTA {TRS, RSUM, ANALYZE, FFOR}
// (include/fls/cor/exp/delta/delta_exp.hpp:39-46); ANALYZE takes base = min and bw = the bit length of max - min
// (src/cor/prm/ffor/ffor_analyze.cpp:78-102, exact); pages as TCompressor::FlushPage / Page::Absorb
// (src/cor/eng/compressor.cpp:41-86, src/cor/lyt/page/page.cpp:87-130).
//
// Three launches and one read-back of the total size:
//   k_enc_analyze  each vector's base and bit width (RLE: its run count), one wave per vector;
//   k_enc_layout   prefix sums of them and the page table (65535 vectors and 128 MiB per page at most), exactly the
//                  host encoder's split, by one block;
//   k_enc_pack     every vector's buffers and entry points, the pages' headers, one wave per vector.
// The pack kernel writes nothing when the total exceeds the caller's capacity, so the layout never visits the host.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "../../include/fls_gpu.h"
#include "decode_core.hpp"
#include "gpu_internal.hpp"

namespace fls {
namespace {

template <typename T>
__device__ __forceinline__ T wave_min(T x) {
    for (int d = 32; d >= 1; d >>= 1) {
        const T y = __shfl_xor(x, d, 64);
        x         = y < x ? y : x;
    }
    return x;
}
template <typename T>
__device__ __forceinline__ T wave_max(T x) {
    for (int d = 32; d >= 1; d >>= 1) {
        const T y = __shfl_xor(x, d, 64);
        x         = y > x ? y : x;
    }
    return x;
}
__device__ __forceinline__ void enc_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A block of the analyze and pack kernels takes a group of 32 consecutive vectors, a wave an equal run of them (their
// small metadata stores share cache lines); prefix sums are kept per group, and a wave scans a group's widths with one
// lane per vector. Large columns run 4 waves of 8 vectors; while the groups are too few to fill the device, 16 waves
// of 2, because a wave's vectors follow one another: 64 vectors of uint32 37 us with 8 in a row, 31 us with 2.
constexpr unsigned kEncGroup = 32, kEncMaxWaves = 16;
__host__ __device__ constexpr unsigned enc_waves(uint32_t n_vec) {
    return (n_vec + kEncGroup - 1) / kEncGroup < 1024 ? kEncMaxWaves : 4;
}

// 16 values of T as SZ registers of 16 bytes; value k sits in register k * SZ / 16.
template <typename T>
struct Vals {
    v4u                  r[sizeof(T)];
    __device__ __forceinline__ T at(unsigned k) const {
        constexpr unsigned per = 16 / sizeof(T);
        const v4u          q   = r[k / per];
        const unsigned     e   = k % per;
        if constexpr (sizeof(T) == 8) return (T)((uint64_t)q[2 * e] | ((uint64_t)q[2 * e + 1] << 32));
        else if constexpr (sizeof(T) == 4) return (T)q[e];
        else if constexpr (sizeof(T) == 2) return (T)(q[e / 2] >> (16 * (e % 2)));
        else return (T)(q[e / 4] >> (8 * (e % 4)));
    }
};
// The vector in memory order: register c of lane l is the vector's 16-byte chunk 64 c + l (each load 1 KiB).
template <typename T>
__device__ __forceinline__ void load_linear(const T* x, unsigned lane, Vals<T>& v) {
    const uint8_t* p = reinterpret_cast<const uint8_t*>(x);
    static_for<sizeof(T)>([&](auto c) { v.r[c] = *reinterpret_cast<const v4u_ua*>(p + 1024 * c + 16 * lane); });
}

struct EncSum {
    uint64_t bits, runs;
};

// The block's bit widths and run counts summed for the layout; `b` and `r` are lane 0's sums of the wave.
__device__ __forceinline__ void group_sum(uint32_t b, uint32_t r, EncSum* sums) {
    __shared__ uint32_t wb[kEncMaxWaves], wr[kEncMaxWaves];
    if (threadIdx.x % 64 == 0) wb[threadIdx.x / 64] = b, wr[threadIdx.x / 64] = r;
    __syncthreads();
    if (threadIdx.x == 0) {
        EncSum s {};
        for (unsigned w = 0; w < blockDim.x / 64; ++w) s.bits += wb[w], s.runs += wr[w];
        sums[blockIdx.x] = s;
    }
}
// Base and bit width of one vector's FFOR (MODE 1: of the values, MODE 2: of their differences from the previous value
// inside the aligned W-value segment, 0 at a segment start -- the unrsum of the transposed lane order): base = min,
// bw = bit length of max - min. SGN: min and max of int64 columns compare as signed values
// (ffor_prm::ResolveAnalyzeFunc, src/cor/prm/ffor/ffor_analyze.cpp:145-160), done here on the values with their sign
// bit flipped. A wave reads its vector with 1 KiB loads and has the next vector's in flight; a lane's first
// difference needs its neighbour's last value, which a shuffle brings (a 1 KiB chunk starts a segment in every type).
template <typename T, int MODE, bool SGN>
__global__ __launch_bounds__(64 * kEncMaxWaves) void k_enc_analyze(const T* __restrict__ x, uint32_t n_vec,
                                                                uint8_t* __restrict__ bw, uint64_t* __restrict__ base,
                                                                EncSum* __restrict__ sums) {
    using C              = std::conditional_t<sizeof(T) == 8, unsigned long long, unsigned>;  // shuffle type
    constexpr C    bias  = SGN ? (C)((T)1 << (8 * sizeof(T) - 1)) : (C)0;
    constexpr unsigned W = 8 * sizeof(T), per = 16 / sizeof(T);
    const unsigned lane  = threadIdx.x % 64;
    const uint32_t run   = kEncGroup * 64 / blockDim.x;
    const uint32_t v0    = blockIdx.x * kEncGroup + threadIdx.x / 64 * run;
    const uint32_t end   = v0 + run < n_vec ? v0 + run : n_vec;
    uint32_t       bits = 0;
    Vals<T>        nx {};
    if (v0 < end) load_linear(x + (uint64_t)v0 * 1024, lane, nx);
    for (uint32_t v = v0; v < end; ++v) {
        const Vals<T> cur = nx;
        if (v + 1 < end) load_linear(x + (uint64_t)(v + 1) * 1024, lane, nx);
        C mn = (C)(T)~(T)0, mx = 0;
        auto add = [&](T d) {
            const C val = (C)d ^ bias;
            mn          = val < mn ? val : mn;
            mx          = val > mx ? val : mx;
        };
        static_for<sizeof(T)>([&](auto c) {
            constexpr unsigned k0 = decltype(c)::value * per;
            T                  prev = 0;
            if constexpr (MODE == 2) prev = (T)__shfl_up((C)cur.at(k0 + per - 1), 1, 64);
            static_for<per>([&](auto e) {
                const T val = cur.at(k0 + e);
                if constexpr (MODE == 2) {
                    constexpr bool inner = decltype(e)::value % W != 0;
                    if (inner || (lane * per) % W != 0) add((T)(val - prev));
                    else add((T)0);
                    prev = val;
                } else {
                    add(val);
                }
            });
        });
        mn = wave_min<C>(mn), mx = wave_max<C>(mx);
        if (lane == 0) {
            const uint64_t d = (uint64_t)(T)(mx - mn);
            const uint32_t b = d ? 64 - (uint32_t)__clzll((long long)d) : 0;
            bw[v]            = (uint8_t)b;
            base[v]          = (uint64_t)(T)(mn ^ bias);
            bits += b;
        }
    }
    group_sum(bits, 0, sums);
}

// RLE (include/fls/cor/exp/rle/rle_exp.hpp:37-74, split of src/cor/lyt/vec.cpp:50-71): a vector's run values
// (one per change of value), and per value its u16 run index, transposed; VAR 1 stores the indexes, VAR 2 their
// 64 lane bases and the FFOR of their in-segment differences (16-value segments of u16), which are the run-start
// flags themselves: 0 at a segment start, else 1 where a run starts -- so base 0 and bw 0 or 1.
// Run-start flags of the vector's values 16 l .. 16 l + 15 (lane l), and those values.
template <typename T>
__device__ __forceinline__ uint32_t run_flags(const T* x, unsigned lane, Vals<T>& v) {
    using C          = std::conditional_t<sizeof(T) == 8, unsigned long long, unsigned>;
    const uint8_t* p = reinterpret_cast<const uint8_t*>(x) + 16 * sizeof(T) * lane;
    static_for<sizeof(T)>([&](auto c) { v.r[c] = *reinterpret_cast<const v4u_ua*>(p + 16 * c); });
    T        prev = (T)__shfl_up((C)v.at(15), 1, 64);
    uint32_t f    = 0;
    static_for<16>([&](auto k) {
        const T val = v.at(k);
        f |= (uint32_t)((lane == 0 && k == 0) || val != prev) << k;
        prev = val;
    });
    return f;
}
// Analysis, one wave per vector: runs[v] = number of runs, bw[v] = the difference FFOR's bit width (VAR 2).
template <typename T>
__global__ __launch_bounds__(64 * kEncMaxWaves) void k_enc_rle_analyze(const T* __restrict__ x, uint32_t n_vec,
                                                                    uint8_t* __restrict__ bw, uint64_t* __restrict__ runs,
                                                                    EncSum* __restrict__ sums) {
    const unsigned lane = threadIdx.x % 64;
    const uint32_t run  = kEncGroup * 64 / blockDim.x;
    const uint32_t v0   = blockIdx.x * kEncGroup + threadIdx.x / 64 * run;
    uint32_t       bits = 0, all = 0;
    for (uint32_t v = v0; v < v0 + run && v < n_vec; ++v) {
        Vals<T>        val;
        const uint32_t f = run_flags(x + (uint64_t)v * 1024, lane, val);
        unsigned       n = __builtin_popcount(f);
        for (int d = 32; d >= 1; d >>= 1) n += __shfl_xor(n, d, 64);
        const bool any = __ballot((f & ~1u) != 0) != 0;  // a run starts inside a segment
        if (lane == 0) runs[v] = n, bw[v] = any ? 1 : 0;
        bits += any, all += n;
    }
    group_sum(bits, all, sums);
}

struct EncPage {
    uint64_t start;    // byte offset of the page in the output
    uint64_t b0, r0;   // sums of the bit widths and run counts of the vectors before it
    uint32_t v0, vec_c, more;
    uint32_t off[6];   // buffer offsets from the page start
};
struct EncTotal {
    uint64_t size, pages;
};

// What the layout and pack kernels share: the encoder's mode (0 UNCOMPRESSED, 1 FFOR, 2 DELTA, 3 / 4 RLE with plain /
// DELTA positions); per vector its bit width and FFOR base (RLE: run count); per group of kEncGroup vectors the sums of
// the bit widths and run counts, which the layout kernel turns into sums over the groups before it (one entry more).
struct EncArgs {
    uint32_t  n_vec, mode, arr_c, sz;
    uint8_t   exp_t, var;
    uint8_t*  bw;
    uint64_t* base;
    EncSum*   sums;
    EncPage*  pages;
    EncTotal* total;
    uint64_t  capacity;
    EncTotal* host_total;  // where the host reads the total (nullptr: it copies `total`)
};

// Sums over the vectors before v (after the layout kernel's scan).
__device__ __forceinline__ EncSum enc_sum_at(const EncArgs& a, uint32_t v) {
    if (a.mode == 0) return {};
    EncSum s = a.sums[v / kEncGroup];
    for (uint32_t u = v / kEncGroup * kEncGroup; u < v; ++u) {
        s.bits += a.bw[u];
        if (a.mode >= 3) s.runs += a.base[u];
    }
    return s;
}

// One block. A vector's bytes are a constant of the mode plus 128 per bit of width plus sz per run, so the sums of
// widths and runs give every page's extent; pages are even splits of at most 65535 vectors that end early before
// the vector that would bring them to 128 MiB (found by two rounds of one probe per thread). Summing per group of 32
// vectors keeps the block's serial part short: with every vector's prefix written here the kernel took 109 us for
// 65536 vectors, and the host loop over a copy of the bit widths that it replaces 300 us with its copies.
__global__ __launch_bounds__(1024) void k_enc_layout(EncArgs a, uint32_t per_pg) {
    __shared__ EncSum ws[16];
    const unsigned tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    if (a.mode) {
        const uint32_t n_g = (a.n_vec + kEncGroup - 1) / kEncGroup, per = (n_g + 1023) / 1024;
        const uint32_t lo = tid * per < n_g ? tid * per : n_g, hi = n_g - lo < per ? n_g : lo + per;
        EncSum         s {};
        for (uint32_t g = lo; g < hi; ++g) s.bits += a.sums[g].bits, s.runs += a.sums[g].runs;
        EncSum inc = s;
        for (unsigned d = 1; d < 64; d <<= 1) {
            const uint64_t y = __shfl_up((unsigned long long)inc.bits, d, 64), z = __shfl_up((unsigned long long)inc.runs, d, 64);
            if (lane >= d) inc.bits += y, inc.runs += z;
        }
        if (lane == 63) ws[wave] = inc;
        __syncthreads();
        EncSum x {inc.bits - s.bits, inc.runs - s.runs};
        for (unsigned w = 0; w < wave; ++w) x.bits += ws[w].bits, x.runs += ws[w].runs;
        for (uint32_t g = lo; g < hi; ++g) {
            const EncSum own = a.sums[g];
            a.sums[g]        = x;
            x.bits += own.bits, x.runs += own.runs;
        }
        if (hi == n_g && lo < hi) a.sums[n_g] = x;
        __syncthreads();
    }
    // bytes of one vector besides its packed rows and run values, and the buffers' sizes in a page
    const uint32_t fixed = a.mode == 0   ? 1024 * a.sz
                           : a.mode == 1 ? 1 + a.sz
                           : a.mode == 2 ? 129 + a.sz
                           : a.mode == 3 ? 2048
                                         : 131;
    const uint64_t per_bit = a.mode == 3 ? 0 : 128;
    uint64_t       pos = 0;
    uint32_t       v0 = 0, p = 0;
    EncSum         s0 {};  // at v0
    while (v0 < a.n_vec) {
        uint32_t m    = a.n_vec - v0 < per_pg ? a.n_vec - v0 : per_pg;
        auto     size = [&](uint32_t c, EncSum s) {  // bytes of a page of c vectors, with the sums at its end
            return 8 + (uint64_t)c * (fixed + 4 * a.arr_c) + (s.bits - s0.bits) * per_bit + (s.runs - s0.runs) * a.sz;
        };
        EncSum   s1   = enc_sum_at(a, v0 + m);
        if (size(m, s1) >= kDataPageMax) {  // uniform over the block
            auto           fits = [&](uint32_t c) { return size(c, enc_sum_at(a, v0 + c)) < kDataPageMax; };
            const uint32_t c1 = 64 * (tid + 1);
            const uint32_t k  = 64 * (uint32_t)__syncthreads_count(c1 <= m && fits(c1)), c2 = k + tid + 1;
            const uint32_t n  = k + (uint32_t)__syncthreads_count(tid < 64 && c2 <= m && fits(c2));
            m                 = n ? n : 1;
            s1                = enc_sum_at(a, v0 + m);
        }
        const uint64_t b1 = s1.bits - s0.bits, r1 = s1.runs - s0.runs;
        uint64_t       off = 8 + 4ull * a.arr_c * m;
        EncPage        pg {};
        pg.start = pos, pg.b0 = s0.bits, pg.r0 = s0.runs, pg.v0 = v0, pg.vec_c = m, pg.more = v0 + m < a.n_vec;
        auto           buf = [&](uint32_t& at, uint64_t bytes) { at = (uint32_t)off, off += bytes; };
        switch (a.mode) {
        case 0: buf(pg.off[0], (uint64_t)m * 1024 * a.sz); break;
        case 1: buf(pg.off[0], m), buf(pg.off[1], (uint64_t)m * a.sz), buf(pg.off[2], 128 * b1); break;
        case 2:
            buf(pg.off[0], 128ull * m), buf(pg.off[1], m), buf(pg.off[2], (uint64_t)m * a.sz), buf(pg.off[3], 128 * b1);
            break;
        case 3: buf(pg.off[0], r1 * a.sz), buf(pg.off[1], 2048ull * m); break;
        default:
            buf(pg.off[0], r1 * a.sz), buf(pg.off[1], 128ull * m), buf(pg.off[2], m), buf(pg.off[3], 2ull * m);
            buf(pg.off[4], 128 * b1);
            break;
        }
        if (tid == 0) a.pages[p] = pg;
        pos += off, v0 += m, s0 = s1, ++p;
    }
    if (tid == 0) {
        *a.total = {pos, p};
        if (a.host_total) *a.host_total = {pos, p};
    }
}

template <typename T>
__device__ __forceinline__ void st_ua(uint8_t* p, T x) {
    if constexpr (sizeof(T) == 1) *p = x;
    else if constexpr (sizeof(T) == 2) *reinterpret_cast<u16_ua*>(p) = x;
    else if constexpr (sizeof(T) == 4) *reinterpret_cast<u32_ua*>(p) = x;
    else *reinterpret_cast<u64_ua*>(p) = x;
}

// Page of vector v (the last whose first vector is at most v).
__device__ __forceinline__ uint32_t page_of(const EncArgs& a, uint32_t v) {
    uint32_t lo = 0, hi = (uint32_t)a.total->pages;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (a.pages[mid].v0 <= v) lo = mid;
        else hi = mid;
    }
    return lo;
}

// The group of the wave's vectors, vector g of it in lane g: bit widths, FFOR bases or run counts, and the sums of the
// widths and runs before each.
struct GroupMeta {
    uint32_t bw;
    uint64_t base, bits, runs;
};
template <bool RLE>
__device__ __forceinline__ GroupMeta group_meta(const EncArgs& a, uint32_t group, unsigned lane) {
    const uint32_t v = group * kEncGroup + lane;
    GroupMeta      m {};
    if (lane < kEncGroup && v < a.n_vec) m.bw = a.bw[v], m.base = a.base[v];
    uint32_t b = m.bw, r = RLE ? (uint32_t)m.base : 0u;
    for (unsigned d = 1; d < kEncGroup; d <<= 1) {
        const uint32_t y = __shfl_up(b, d, 64), z = RLE ? __shfl_up(r, d, 64) : 0u;
        if (lane >= d) b += y, r += z;
    }
    const EncSum s = a.sums[group];
    m.bits = s.bits + b - m.bw, m.runs = s.runs + r - (RLE ? (uint32_t)m.base : 0u);
    return m;
}
template <typename U>
__device__ __forceinline__ U lane_value(U x, unsigned k) {
    if constexpr (sizeof(U) == 8)
        return (U)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((uint32_t)((uint64_t)x >> 32), k) << 32) |
                   (uint32_t)__builtin_amdgcn_readlane((uint32_t)x, k));
    else return (U)__builtin_amdgcn_readlane((uint32_t)x, k);
}

// Header and buffer offsets of a page, by the wave that packs its first vector.
__device__ __forceinline__ void page_head(const EncArgs& a, const EncPage& pg, uint8_t* p, unsigned lane) {
    if (lane == 0) {
        st_ua<uint32_t>(p, (uint32_t)a.exp_t | ((uint32_t)a.var << 8));
        st_ua<uint32_t>(p + 4, (pg.vec_c & 0xffffu) | (pg.more << 16));
    }
    if (lane < a.arr_c) {
        uint32_t o = pg.off[0];
        static_for<5>([&](auto k) { o = lane == k + 1 ? pg.off[k + 1] : o; });
        st_ua<uint32_t>(p + 8 + 4 * lane, o);
    }
}

// A thread's part of a transposed vector, in lane order: W = 64 lane t % 16, values j in [16 q, 16 q + 16) with
// q = t / 16; W = 32 lane t % 32, half t / 32; W = 16 lane t; W = 8 lanes t and t + 64, 8 values each. Value j of a
// lane sits at p with j = j_of_p(p) (fls_lanes.hpp), so a part is runs of 2, 4, 8 or 16 consecutive input values:
// sizeof(T) loads of 16 bytes. slot(c, e): place in the part of element e of load c.
template <typename T>
struct Part {
    static constexpr unsigned W = 8 * sizeof(T), L = 1024 / W, per = 16 / sizeof(T);
    __device__ static __forceinline__ unsigned lane_of(unsigned t) { return W == 64 ? t % 16 : W == 32 ? t % 32 : t; }
    __device__ static __forceinline__ unsigned part_of(unsigned t) { return W == 64 ? t / 16 : W == 32 ? t / 32 : 0; }
    static constexpr unsigned slot(unsigned c, unsigned e) {
        if constexpr (W == 64) return 8 * e + order8(c);
        else if constexpr (W == 32) return 4 * e + ord4(c);
        else if constexpr (W == 16) return 2 * e + c;
        else return e;
    }
    __device__ static __forceinline__ void load(const T* x, unsigned t, Vals<T>& v) {
        const uint8_t* p = reinterpret_cast<const uint8_t*>(x + seg_start<(int)W>(lane_of(t)) + part_of(t) * per);
        constexpr unsigned step = W == 16 ? 16 : 8 * sizeof(T);  // bytes between a part's loads
        static_for<sizeof(T)>([&](auto c) { v.r[c] = *reinterpret_cast<const v4u_ua*>(p + step * c); });
    }
};

// FFOR / DELTA / UNCOMPRESSED (bit width W, base 0): one wave per vector. Every thread packs
// the 16 values of its part and ORs its words into the vector's zeroed packed rows in LDS (a word that two parts share
// gets both; 8/16-bit lanes belong to one thread and are stored plainly), which leave as 16-byte stores. All 64 lanes
// work for every type; with one thread per lane (16 or 32 of 128 threads) and word-sized stores this kernel took
// 170 us for 2^26 uint32 values at 7 bits. The runs are taken from the column's end: what the analyze pass read last is
// still in the last-level cache.
template <typename T, int MODE>
__global__ __launch_bounds__(64 * kEncMaxWaves) void k_enc_pack(const T* __restrict__ x, EncArgs a, uint8_t* __restrict__ out) {
    using P                 = Part<T>;
    using C                 = std::conditional_t<sizeof(T) == 8, unsigned long long, unsigned>;
    constexpr unsigned W = P::W, L = P::L, SZ = sizeof(T), per = P::per;
    extern __shared__ __attribute__((aligned(16))) uint8_t enc_lds[];  // 128 W bytes per wave
    if (a.total->size > a.capacity) return;
    const unsigned lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const unsigned i = P::lane_of(lane), h = P::part_of(lane);
    uint8_t*       lr  = enc_lds + wave * (128 * W);
    const uint32_t run = kEncGroup * 64 / blockDim.x;
    const uint32_t grp = gridDim.x - 1 - blockIdx.x;
    const uint32_t v0  = grp * kEncGroup + wave * run;
    const uint32_t end = v0 + run < a.n_vec ? v0 + run : a.n_vec;
    if (v0 >= end) return;
    GroupMeta      gm {};
    if constexpr (MODE != 0) gm = group_meta<false>(a, grp, lane);
    uint32_t       pi = page_of(a, v0);
    EncPage        pg = a.pages[pi];
    Vals<T>        nx {};
    P::load(x + (uint64_t)v0 * 1024, lane, nx);
    for (uint32_t v = v0; v < end; ++v) {
        const Vals<T> cur = nx;
        if (v + 1 < end) P::load(x + (uint64_t)(v + 1) * 1024, lane, nx);
        if (v - pg.v0 == pg.vec_c) pg = a.pages[++pi];
        const uint32_t r = v - pg.v0;
        uint8_t*       p = out + pg.start;
        if (r == 0) page_head(a, pg, p, lane);
        uint8_t*           ep = p + 8 + 4 * a.arr_c + 4ull * a.arr_c * (r ? r - 1 : 0);  // this vector's entry points
        constexpr unsigned o  = MODE == 2 ? 1 : 0;                                       // bw buffer
        unsigned           bw = W;
        T                  base = 0;
        uint32_t           rel  = r * 1024 * SZ;  // the packed rows' place in their buffer
        uint8_t*           pk   = p + pg.off[0] + (uint64_t)r * 1024 * SZ;
        if constexpr (MODE != 0) {
            const unsigned k = wave * run + (v - v0);
            bw   = lane_value(gm.bw, k);
            base = (T)lane_value(gm.base, k);
            rel  = 128u * (uint32_t)(lane_value(gm.bits, k) - pg.b0);
            pk   = p + pg.off[o + 2] + rel;
            if (lane == 0) {
                p[pg.off[o] + r] = (uint8_t)bw;
                st_ua<T>(p + pg.off[o + 1] + (uint64_t)r * SZ, base);
            }
        }
        if (r && lane == 0) {
            if constexpr (MODE == 2) st_ua<uint32_t>(ep, r * 128), ep += 4;
            if constexpr (MODE != 0) st_ua<uint32_t>(ep, r), st_ua<uint32_t>(ep + 4, r * SZ), ep += 8;
            st_ua<uint32_t>(ep, rel);
        }
        T u[16];  // what FFOR packs, in lane order
        static_for<16>([&](auto k) {
            constexpr unsigned c = decltype(k)::value / per, e = decltype(k)::value % per;
            if constexpr (W == 8) u[k] = cur.at(k);
            else u[P::slot(c, e)] = cur.at(k);
        });
        if constexpr (MODE == 2) {
            // lane bases: the lane's first value; then differences in the order of the input
            uint8_t* lb = p + pg.off[0] + (uint64_t)r * 128;
            if constexpr (W == 8) {
                lb[lane] = (uint8_t)u[0], lb[lane + 64] = (uint8_t)u[8];
            } else {
                if (h == 0) st_ua<T>(lb + i * SZ, u[0]);
            }
            if constexpr (W >= 32) {
                // the value before a load's first is the last of the same load in the part before (part 0: of the
                // load before in the last part)
                constexpr unsigned G = W == 64 ? 16 : 32;  // lanes between parts
                T                  before = u[0];          // the segment's start: difference 0
                static_for<SZ>([&](auto c) {
                    const T far = (T)__shfl((C)cur.at(c * per + per - 1), (int)((lane + 64 - G) % 64), 64);
                    T       pv  = h ? far : before;
                    before      = far;
                    static_for<per>([&](auto e) {
                        const T val            = cur.at(c * per + e);
                        u[P::slot(c, e)] = (T)(val - pv);
                        pv                     = val;
                    });
                });
            } else {
                static_for<16>([&](auto k) {
                    constexpr unsigned q = decltype(k)::value;
                    constexpr bool     first = W == 16 ? q == 0 : q % 8 == 0;
                    const T            d = first ? (T)0 : (T)(cur.at(q) - cur.at(q ? q - 1 : 0));
                    if constexpr (W == 8) u[q] = d;
                    else u[P::slot(q / per, q % per)] = d;
                });
            }
        }
        if (bw == 0) continue;
        if constexpr (W >= 32) {
            for (uint32_t c = lane; c < 8 * bw; c += 64) *reinterpret_cast<v4u*>(lr + 16 * c) = v4u {0, 0, 0, 0};
            enc_wave_sync();
            C*       word = reinterpret_cast<C*>(lr) + i;
            uint32_t w = 16 * h * bw / W, nb = 16 * h * bw % W;
            C        acc = 0;
            static_for<16>([&](auto k) {
                const C val = (C)(T)(u[k] - base);
                acc |= val << nb;
                nb += bw;
                if (nb >= W) {
                    atomicOr(word + w * L, acc);
                    nb -= W, ++w;
                    acc = nb ? val >> (bw - nb) : (C)0;
                }
            });
            if (nb) atomicOr(word + w * L, acc);
        } else {
            constexpr unsigned lanes = W == 8 ? 2 : 1;  // lanes per thread
            static_for<lanes>([&](auto q) {
                T*       word = reinterpret_cast<T*>(lr) + lane + 64 * q;
                uint32_t w = 0, nb = 0, acc = 0;
                static_for<16 / lanes>([&](auto k) {
                    acc |= (uint32_t)(T)(u[q * 8 + k] - base) << nb;
                    nb += bw;
                    if (nb >= W) word[w * L] = (T)acc, acc >>= W, nb -= W, ++w;
                });
            });
        }
        enc_wave_sync();
        for (uint32_t c = lane; c < 8 * bw; c += 64)
            *reinterpret_cast<v4u_ua*>(pk + 16 * c) = *reinterpret_cast<const v4u*>(lr + 16 * c);
        enc_wave_sync();
    }
}

// RLE pages: one wave per vector, lane l owning values 16 l .. 16 l + 15, which are one u16 position segment: its run
// flags give the segment's first run index (the lane base) and its packed differences, and the run values it starts.
template <typename T, int VAR>
__global__ __launch_bounds__(64 * kEncMaxWaves) void k_enc_rle_pack(const T* __restrict__ x, EncArgs a, uint8_t* __restrict__ out) {
    constexpr unsigned SZ = sizeof(T);
    extern __shared__ __attribute__((aligned(16))) uint8_t enc_lds[];  // VAR 1: the wave's 1024 transposed positions
    if (a.total->size > a.capacity) return;
    const unsigned lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    // the u16 lane whose segment starts at value 16 * lane: seg_start<16>(i) = 64 (i % 16) + 8 order8(i / 16)
    const unsigned i  = (lane >> 2) + 16 * (((lane & 1) << 1) | ((lane >> 1) & 1));
    uint16_t*      pos = reinterpret_cast<uint16_t*>(enc_lds) + wave * 1024;
    const uint32_t run_v = kEncGroup * 64 / blockDim.x, grp = gridDim.x - 1 - blockIdx.x;
    const uint32_t v0  = grp * kEncGroup + wave * run_v;
    if (v0 >= a.n_vec) return;
    const GroupMeta gm = group_meta<true>(a, grp, lane);
    uint32_t        pi = page_of(a, v0);
    EncPage         pg = a.pages[pi];
    for (uint32_t v = v0; v < v0 + run_v && v < a.n_vec; ++v) {
        if (v - pg.v0 == pg.vec_c) pg = a.pages[++pi];
        const unsigned k_v = wave * run_v + (v - v0);
        const uint32_t r   = v - pg.v0;
        uint8_t*       p  = out + pg.start;
        if (r == 0) page_head(a, pg, p, lane);
        Vals<T>        val;
        const uint32_t f = run_flags(x + (uint64_t)v * 1024, lane, val);
        const uint32_t n = (uint32_t)__builtin_popcount(f);
        uint32_t       inc = n;
        for (unsigned d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(inc, d, 64);
            if (lane >= d) inc += y;
        }
        uint32_t       run = inc - n;  // runs started before this segment
        const uint32_t rel = (uint32_t)((lane_value(gm.runs, k_v) - pg.r0) * SZ);
        uint8_t*       rv  = p + pg.off[0] + rel;
        uint8_t*       ep  = p + 8 + 4 * a.arr_c + 4ull * a.arr_c * (r ? r - 1 : 0);
        const uint32_t first = run + (f & 1u) - 1;  // run index of the segment's first value
        static_for<16>([&](auto k) {
            if ((f >> k) & 1u) st_ua<T>(rv + (uint64_t)run * SZ, val.at(k)), ++run;
            if constexpr (VAR == 1) pos[64 * j_of_p<16>(k) + i] = (uint16_t)(run - 1);
        });
        if constexpr (VAR == 1) {
            enc_wave_sync();
            uint8_t* dst = p + pg.off[1] + (uint64_t)r * 2048;
            static_for<2>([&](auto c) {
                *reinterpret_cast<v4u_ua*>(dst + 1024 * c + 16 * lane) =
                    *reinterpret_cast<const v4u*>(&pos[512 * c + 8 * lane]);
            });
            enc_wave_sync();
            if (r && lane == 0) st_ua<uint32_t>(ep, rel), st_ua<uint32_t>(ep + 4, r * 2048);
        } else {
            const unsigned bw  = lane_value(gm.bw, k_v);
            const uint32_t prl = 128u * (uint32_t)(lane_value(gm.bits, k_v) - pg.b0);
            st_ua<uint16_t>(p + pg.off[1] + (uint64_t)r * 128 + 2 * i, (uint16_t)first);
            if (lane == 0) {
                p[pg.off[2] + r] = (uint8_t)bw;
                st_ua<uint16_t>(p + pg.off[3] + (uint64_t)r * 2, 0);  // base: the minimum difference is 0
                if (r) {
                    st_ua<uint32_t>(ep, rel), st_ua<uint32_t>(ep + 4, r * 128);
                    st_ua<uint32_t>(ep + 8, r), st_ua<uint32_t>(ep + 12, r * 2), st_ua<uint32_t>(ep + 16, prl);
                }
            }
            if (bw) {  // bw 1: the segment's 16 differences form one u16 word, value p at bit j_of_p(p)
                uint32_t word = 0;
                static_for<15>([&](auto k) { word |= ((f >> (k + 1)) & 1u) << j_of_p<16>(k + 1); });
                st_ua<uint16_t>(p + pg.off[4] + prl + 2 * i, (uint16_t)word);
            }
        }
    }
}

template <typename T>
hipError_t launch_enc(const EncArgs& a, const void* x, bool sgn, uint32_t per_pg, uint8_t* out, hipStream_t s) {
    const T*       xv = static_cast<const T*>(x);
    const unsigned waves = enc_waves(a.n_vec);
    const dim3     g((a.n_vec + kEncGroup - 1) / kEncGroup), b(64 * waves);
#define A(M, S) hipLaunchKernelGGL((k_enc_analyze<T, M, S>), g, b, 0, s, xv, a.n_vec, a.bw, a.base, a.sums)
#define P(M) hipLaunchKernelGGL((k_enc_pack<T, M>), g, b, waves * 1024 * sizeof(T), s, xv, a, out)
#define R(V) hipLaunchKernelGGL((k_enc_rle_pack<T, V>), g, b, V == 1 ? waves * 2048 : 0, s, xv, a, out)
    if (a.mode == 1 && sgn) A(1, true);
    else if (a.mode == 1) A(1, false);
    else if (a.mode == 2 && sgn) A(2, true);
    else if (a.mode == 2) A(2, false);
    else if (a.mode >= 3) hipLaunchKernelGGL((k_enc_rle_analyze<T>), g, b, 0, s, xv, a.n_vec, a.bw, a.base, a.sums);
    hipLaunchKernelGGL(k_enc_layout, dim3(1), dim3(1024), 0, s, a, per_pg);
    switch (a.mode) {
    case 0: P(0); break;
    case 1: P(1); break;
    case 2: P(2); break;
    case 3: R(1); break;
    default: R(2); break;
    }
#undef A
#undef P
#undef R
    return hipGetLastError();
}

hipError_t launch_enc_w(unsigned W, const EncArgs& a, const void* x, bool sgn, uint32_t per_pg, uint8_t* out, hipStream_t s) {
    switch (W) {
    case 8: return launch_enc<uint8_t>(a, x, sgn, per_pg, out, s);
    case 16: return launch_enc<uint16_t>(a, x, sgn, per_pg, out, s);
    case 32: return launch_enc<uint32_t>(a, x, sgn, per_pg, out, s);
    default: return launch_enc<uint64_t>(a, x, sgn, per_pg, out, s);
    }
}

}  // namespace
}  // namespace fls

using namespace fls;

// The encoder's device scratch, one region: the total, the page table, per vector its bit width and FFOR base (RLE: run
// count), and the groups' sums. A page holds at least 8192 vectors unless the column ends or
// is split evenly (128 MiB of the widest vectors, below 10.5 KB each, is over 12000), which bounds the page table.
namespace fls {
constexpr uint64_t kEncFixedVec = 16384;  // 2^24 values
constexpr uint64_t enc_pages_max(uint64_t n_vec) { return n_vec / 8192 + (n_vec + kMaxVecPerPage - 1) / kMaxVecPerPage + 2; }
constexpr uint64_t enc_r256(uint64_t n) { return (n + 255) / 256 * 256; }
// offsets of the regions {total, pages, base, sums, bw} and the scratch's size
struct EncScratch {
    uint64_t pages, base, sums, bw, size;
};
constexpr EncScratch enc_scratch(uint64_t n_vec) {
    EncScratch l {};
    l.pages = 256;
    l.base  = l.pages + enc_r256(enc_pages_max(n_vec) * sizeof(EncPage));
    l.sums  = l.base + enc_r256(8 * n_vec);
    l.bw    = l.sums + enc_r256(((n_vec + kEncGroup - 1) / kEncGroup + 1) * sizeof(EncSum));
    l.size  = l.bw + enc_r256(n_vec);
    return l;
}
constexpr size_t kEncFixedBytes = enc_scratch(kEncFixedVec).size;
// Scratch kept for fls_gpu_encode calls of up to kEncSlotVec vectors (2^28 values): a stream allocation, its release and the
// copy of the total cost a call 25 to 45 us, more than its kernels for a small column and a tenth of them at this size (uint32
// FFOR, 490 us, 538 one vector further; 65537 vectors 147 us while slots ended at 65536, 122 now). 2.5 MB a slot; past it
// the share shrinks with the memory growing. A call holds a slot until its stream has completed.
constexpr uint64_t kEncSlotVec   = 262144;
constexpr size_t   kEncSlotBytes = enc_scratch(kEncSlotVec).size;
constexpr unsigned kEncSlots     = 4;
}  // namespace fls

// Device scratch, one copy per GPU for as long as the library is loaded: fls_gpu_encode_noalloc's, and the slots. Host
// code never uses the names as addresses: each device's address comes from hipGetSymbolAddress (EncDevice).
static __device__ __align__(256) uint8_t scratch[fls::kEncFixedBytes];
static __device__ __align__(256) uint8_t enc_slots[fls::kEncSlots * fls::kEncSlotBytes];

namespace {
// A device's scratch addresses, looked up once with that device current, and its slots' owners. Each slot has a place in
// pinned host memory that the layout kernel writes the total to (a copy back of 16 bytes takes 10 us longer); the
// allocation-free encoder has none, because pinned memory is an allocation.
struct EncDevice {
    uint8_t  *fixed = nullptr, *slots = nullptr;
    EncTotal* totals = nullptr;  // kEncSlots
    unsigned  taken  = 0;        // bit k: slot k
};
std::mutex             g_enc_mu;
std::vector<EncDevice> g_enc_dev;

int enc_device(int dev, bool noalloc) {
    hipError_t                  e = hipSuccess;
    std::lock_guard<std::mutex> lock(g_enc_mu);
    if ((size_t)dev >= g_enc_dev.size()) g_enc_dev.resize(dev + 1);
    EncDevice& d = g_enc_dev[dev];
    void*      p = nullptr;
    if (noalloc) {
        if (d.fixed) return FLS_OK;
        if ((e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch))) != hipSuccess) return hip_fail(e, "hipGetSymbolAddress");
        d.fixed = static_cast<uint8_t*>(p);
        return FLS_OK;
    }
    if (d.totals) return FLS_OK;
    if ((e = hipGetSymbolAddress(&p, HIP_SYMBOL(enc_slots))) != hipSuccess) return hip_fail(e, "hipGetSymbolAddress");
    d.slots = static_cast<uint8_t*>(p);
    if ((e = hipHostMalloc(&p, sizeof(EncTotal) * kEncSlots, hipHostMallocPortable | hipHostMallocMapped)) != hipSuccess)
        return hip_fail(e, "hipHostMalloc");
    d.totals = static_cast<EncTotal*>(p);
    return FLS_OK;
}

// The stream's device, made current for as long as this lives: the scratch and the kernels belong to it, whichever device
// the caller has current (the null stream, hipStreamLegacy and hipStreamPerThread are that one's; hipStreamGetDevice takes the
// second of them for a pointer).
struct StreamDevice {
    int        dev = 0, before = 0;
    hipError_t err;
    explicit StreamDevice(hipStream_t s) {
        if ((err = hipGetDevice(&before)) != hipSuccess) return;
        dev = before;
        hipDevice_t d = (hipDevice_t)before;
        if (s && s != hipStreamLegacy && s != hipStreamPerThread && hipStreamGetDevice(s, &d) != hipSuccess) (void)hipGetLastError(), d = (hipDevice_t)before;
        if ((int)d != before && (err = hipSetDevice((int)d)) == hipSuccess) dev = (int)d;
    }
    ~StreamDevice() {
        if (dev != before) (void)hipSetDevice(before);
    }
};

// `noalloc`: the fixed scratch (at most kEncFixedVec vectors); otherwise a slot, or a stream allocation for larger
// columns and when the slots are taken.
int encode_impl(const void* dev_values, uint64_t n, enum data_t type, uint8_t expr_id, uint8_t* dev_out,
                uint64_t capacity, uint64_t* out_size, void* stream, bool noalloc) {
    if (!out_size || !dev_out || (n && !dev_values)) return fail(FLS_E_ARG, "null argument");
    Expr e;
    if (type == STR || !expr_from_id((uint8_t)type, expr_id, e)) return fail(FLS_E_UNSUPPORTED, "unknown expression");
    const int mode = e.exp_t == EXP_UNCOMPRESSED            ? 0
                     : (e.exp_t == EXP_FFOR && e.var == 1)  ? 1
                     : (e.exp_t == EXP_DELTA && e.var == 1) ? 2
                     : (e.exp_t == EXP_RLE && e.var == 1)   ? 3
                     : (e.exp_t == EXP_RLE && e.var == 2)   ? 4
                                                            : -1;
    if (mode < 0) return fail(FLS_E_UNSUPPORTED, "the GPU encoder writes UNCOMPRESSED, FFOR, DELTA and RLE pages (no patches, no chains)");
    // double RLE splits runs by double equality (+0.0 == -0.0, NaN != NaN): the host encoder writes those pages
    if (type == DOUBLE && mode) return fail(FLS_E_UNSUPPORTED, "the GPU encoder writes double columns UNCOMPRESSED only");
    if (n % 1024) return fail(FLS_E_UNSUPPORTED, "value count must be a multiple of 1024");
    const unsigned W = dtype_bits((uint8_t)type);
    const uint64_t n_vec = n / 1024;
    hipStream_t    s     = (hipStream_t)stream;
    hipError_t     err;
    if (n_vec > 0xffffff00ull) return fail(FLS_E_CAPACITY, "column too large");  // 4 TiB and more
    if (!n_vec) {  // one page without vectors: its header, and every buffer at its end
        std::vector<uint8_t> head(8 + 4 * e.arr_c, 0);
        head[0] = e.exp_t, head[1] = e.var;
        for (unsigned b = 0; b < e.arr_c; ++b) head[8 + 4 * b] = (uint8_t)head.size();
        *out_size = head.size();
        if (head.size() > capacity) return fail(FLS_E_CAPACITY, "encoded column exceeds capacity");
        err = hipMemcpyAsync(dev_out, head.data(), head.size(), hipMemcpyHostToDevice, s);
        if (err == hipSuccess) err = hipStreamSynchronize(s);
        return err == hipSuccess ? FLS_OK : hip_fail(err, "hipMemcpyAsync");
    }
    const StreamDevice on(s);
    if (on.err != hipSuccess) return hip_fail(on.err, "stream device");
    const int dev = on.dev;
    if (int rc = enc_device(dev, noalloc)) return rc;
    uint8_t*  d     = nullptr;
    EncTotal* total = nullptr;  // pinned host memory
    unsigned  slot  = kEncSlots;
    {
        std::lock_guard<std::mutex> lock(g_enc_mu);
        EncDevice&                  ed = g_enc_dev[dev];
        if (noalloc) {
            d = ed.fixed;
        } else if (n_vec <= kEncSlotVec) {
            for (slot = 0; slot < kEncSlots && (ed.taken >> slot & 1u);) ++slot;
            if (slot < kEncSlots) ed.taken |= 1u << slot, d = ed.slots + slot * kEncSlotBytes, total = ed.totals + slot;
        }
    }
    const EncScratch at = enc_scratch(n_vec);
    const bool       own = !d;
    if (own && (err = hipMallocAsync((void**)&d, at.size, s)) != hipSuccess) return hip_fail(err, "hipMallocAsync");
    EncArgs a {};
    a.n_vec = (uint32_t)n_vec, a.mode = (uint32_t)mode, a.arr_c = e.arr_c, a.sz = W / 8, a.exp_t = e.exp_t, a.var = e.var;
    a.total = reinterpret_cast<EncTotal*>(d), a.pages = reinterpret_cast<EncPage*>(d + at.pages), a.bw = d + at.bw;
    a.base  = reinterpret_cast<uint64_t*>(d + at.base), a.sums = reinterpret_cast<EncSum*>(d + at.sums);
    a.capacity = capacity, a.host_total = total;
    const uint64_t page_c = (n_vec + kMaxVecPerPage - 1) / kMaxVecPerPage;
    EncTotal       copy {};
    err = launch_enc_w(W, a, dev_values, type == INT64, (uint32_t)((n_vec + page_c - 1) / page_c), dev_out, s);
    if (!total && err == hipSuccess) err = hipMemcpyAsync(&copy, a.total, sizeof copy, hipMemcpyDeviceToHost, s);
    if (own) (void)hipFreeAsync(d, s);
    const hipError_t done = hipStreamSynchronize(s);
    if (err == hipSuccess) err = done;
    if (total) copy = *total;
    if (slot < kEncSlots) {
        std::lock_guard<std::mutex> lock(g_enc_mu);
        g_enc_dev[dev].taken &= ~(1u << slot);
    }
    if (err != hipSuccess) return hip_fail(err, "encode");
    *out_size = copy.size;
    return copy.size > capacity ? fail(FLS_E_CAPACITY, "encoded column exceeds capacity") : FLS_OK;
}
}  // namespace

extern "C" int fls_gpu_encode(const void* dev_values, uint64_t n, enum data_t type, uint8_t expr_id, uint8_t* dev_out,
                              uint64_t capacity, uint64_t* out_size, void* stream) {
    return encode_impl(dev_values, n, type, expr_id, dev_out, capacity, out_size, stream, false);
}

extern "C" int fls_gpu_encode_noalloc(const void* dev_values, uint64_t n, enum data_t type, uint8_t expr_id,
                                      uint8_t* dev_out, uint64_t capacity, uint64_t* out_size, void* stream) {
    if (n / 1024 > kEncFixedVec) return fail(FLS_E_CAPACITY, "the allocation-free encoder takes at most 2^24 values per call");
    return encode_impl(dev_values, n, type, expr_id, dev_out, capacity, out_size, stream, true);
}
