// sort.hip -- LDS-staged radix sort of 30-bit Morton keys into (key, index)
// pairs for gfx950 (the std::sort of LBVH_build, src/renderer/bvh.h:207-208,
// defined stable: equal keys keep index order).
//
// The top digit has between 1 and 11 bits so that a bucket holds ~1K keys
// (10 bits = 1024 buckets at 1M keys).  Three launches, each reading its
// input once:
//   hist     8192-key tiles (1024 threads): LDS histograms of the top digit
//            per 4096-key half; every tile reserves its range inside each
//            bucket with one returning atomic per non-empty digit and hands
//            the halves consecutive sub-ranges.  The atomics make the tile
//            order inside a bucket arbitrary, which is harmless because the
//            last pass orders the full (key, index).
//   scatter  4096-key halves: bucket bases from an LDS scan of the digit
//            totals, LDS-atomic ranks inside the half, 8-byte
//            (key<<32 | index) composites staged in LDS in digit order and
//            written with consecutive lanes on consecutive slots.  The two
//            halves of a histogram tile run on one XCD.
//   local    one block per bucket staged in LDS: MSD split on the next 10 key
//            bits into 1024 sub-buckets (~1 element each), then every
//            composite is placed by its rank among its sub-bucket.  A bucket
//            too large for LDS is cut into pieces of whole sub-buckets, which
//            the blocks take between them (larger ones, local_wide, in sorts
//            of more than kWideMin keys).
// More than kRadixMin keys are sorted by three stable 10-bit passes instead.
// Every bucket block zeroes its digit total once it has read it, so each call
// leaves the totals cleared for the next call in stream order: eager calls and
// replays of captured graphs (of any number of sorts) may interleave freely.
#include "dev_math.h"
#include "gpr_internal.h"

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <string>

namespace gpr {
namespace {

constexpr int kMaxDigits = 2048;    // top-digit buckets (11 bits at most)
constexpr int kSubs = 2;            // scatter sub-tiles per histogram tile
constexpr int kScatterThreads = 1024;
// Reservation groups: tile t reserves its range of each bucket from the
// counter of group t % kGroups, so each counter takes ntiles / kGroups
// returning atomics instead of ntiles (device-scope atomics on one address
// serialise); a bucket holds the groups' ranges one after another.
constexpr int kGroups = 4;
constexpr uint32_t kAccWords = kMaxDigits * kGroups;
// counter of digit d in group g: one group's counters side by side, so the
// reservations of one wave touch two cache lines (64 digits)
GPR_D constexpr uint32_t acc_at(uint32_t d, uint32_t g) { return g * kMaxDigits + d; }
constexpr int kTile = 8192;         // keys per histogram tile
constexpr int kSubTile = kTile / kSubs;  // keys per scatter tile
constexpr int kTileThreads = 1024;
constexpr int kLocalThreads = 512;
constexpr int kFastCap = 1536;      // bucket size of the LDS fast path (A and B)
constexpr int kSub = 1024;          // sub-buckets of the LDS MSD split
constexpr int kSubMax = 48;         // largest sub-bucket of the fast path, where every rank reads its whole sub-bucket
constexpr uint32_t kWin = 4;        // sub-bucket entries a rank reads at once
static_assert(kSub % kLocalThreads == 0, "sub-bucket scan: whole counts per thread");
constexpr uint32_t kWinStep = 1536;   // piece starts fall on sub-bucket starts past multiples of this
constexpr uint32_t kWideStep = 6144;  // the same in sorts of more than kWideMin keys
constexpr int kWideThreads = 512;
constexpr uint32_t kRankMax = 1024;   // largest sub-bucket placed by rank (O(size) LDS reads per entry)
// Pieces of a bucket that are dealt out to all blocks; wide pieces: those after
// the first, which its own block takes.
template <bool WIDE>
GPR_HD constexpr uint32_t pieces_of(uint32_t n) {
    if (WIDE) return n > kWideStep ? (n - 1) / kWideStep : 0u;
    return n > (uint32_t)kFastCap ? (n + kWinStep - 1) / kWinStep : 0u;
}

// Every piece reads its whole bucket, so a bucket of m keys costs m * m / step
// reads.  From kWideMin on most buckets are cut, and with larger pieces a uniform
// bucket is one; from kRadixMin on the passes cost less than the pieces of 1536 did
// for uniform keys, and larger pieces more than one block a bucket did for clustered
// ones.  Us for uniform keys and keys of 64 clusters, with one block a bucket, pieces
// of 1536, of 6144, and the passes:
//          uniform                     clusters
//    3.0M    55    51    60   110     19934    1528    1300   115
//    3.2M    75    76    68   112     25288    1868    1459   119
//    4.2M    88    84    76   124     24499   12175    7770   127
//    8.4M   164   162   140   217     35059   63632   17815   228
//   15.7M   446   417   332   397     61723  211131   62331   412
//   16.8M   492   459   356   413     76482  238898   60209   423
//   67.1M  2258  3022  2080  1758
// 4.2M equal keys: 288 ms, 64 ms, 15.9 ms, 116 us.
constexpr uint32_t kWideMin = 3u << 20, kRadixMin = 15u << 20;

// Top-digit width: ~1K keys per bucket, between 1 and 11 bits.
uint32_t digit_bits(uint32_t n) {
    uint32_t b = 1;
    while (b < 11u && ((uint64_t)n >> b) > 1024u) ++b;
    return b;
}

inline uint32_t div_up(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// Inclusive scan of a wave64: Hillis-Steele inside each row of 16 lanes with
// row_shr DPP moves (1, 2, 4, 8), then the row totals carried across rows with
// row_bcast:15 (rows 1 and 3) and row_bcast:31 (rows 2 and 3).  Lanes a move
// does not reach receive 0.
template <int CTRL, int ROWS>
GPR_D uint32_t dpp_or_zero(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
GPR_D uint32_t wave_scan_incl(uint32_t v) {
    v += dpp_or_zero<0x111, 0xf>(v);  // row_shr:1
    v += dpp_or_zero<0x112, 0xf>(v);  // row_shr:2
    v += dpp_or_zero<0x114, 0xf>(v);  // row_shr:4
    v += dpp_or_zero<0x118, 0xf>(v);  // row_shr:8
    v += dpp_or_zero<0x142, 0xa>(v);  // row_bcast:15 into rows 1, 3
    v += dpp_or_zero<0x143, 0xc>(v);  // row_bcast:31 into rows 2, 3
    return v;
}

// inclusive scan of one value per thread over a block of NT threads (wave64)
template <int NT>
GPR_D uint32_t scan_incl(uint32_t v, uint32_t* sh, uint32_t* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    v = wave_scan_incl(v);
    if (lane == 63) sh[wave] = v;
    __syncthreads();
    uint32_t add = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        const uint32_t s = sh[w];
        add += w < wave ? s : 0u;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return v + add;
}

// inclusive scans of two values per thread over a block of NT threads,
// sharing their barriers
template <int NT>
GPR_D void scan_incl2(uint32_t& a, uint32_t& b, uint32_t* sh /* 2 * NT / 64 */) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    a = wave_scan_incl(a);
    b = wave_scan_incl(b);
    if (lane == 63) {
        sh[2 * wave] = a;
        sh[2 * wave + 1] = b;
    }
    __syncthreads();
    uint32_t adda = 0, addb = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        adda += w < wave ? sh[2 * w] : 0u;
        addb += w < wave ? sh[2 * w + 1] : 0u;
    }
    __syncthreads();
    a += adda;
    b += addb;
}

// ---- hist: 8192-key tiles, per-half histograms, one reservation per digit
__global__ __launch_bounds__(kTileThreads) void k_hist(const uint32_t* __restrict__ keys, uint32_t n,
                                                       uint32_t shift, uint32_t nd,
                                                       uint32_t* __restrict__ acc,
                                                       uint32_t* __restrict__ off) {
    __shared__ uint32_t h[kSubs * kMaxDigits];
    // the keys are requested first (16-byte loads where the array allows,
    // thread t taking keys 4t..4t+3 of each 4096-key round), the LDS histograms
    // cleared while they are in flight
    constexpr int kRound = 4 * kTileThreads;  // keys of one round of 16-byte loads
    static_assert(kRound % kSubTile == 0 || kSubTile % kRound == 0, "load rounds tile the sub-tiles");
    const uint64_t base = (uint64_t)blockIdx.x * kTile;
    const bool vec = (reinterpret_cast<uintptr_t>(keys) & 15u) == 0;
    uint32_t k[kTile / kTileThreads];
#pragma unroll
    for (int x = 0; x < kTile / kRound; ++x) {
        const uint64_t i0 = base + (uint64_t)x * kRound + 4u * threadIdx.x;
        if (vec && i0 + 3 < n) {
            const uint4 v = *reinterpret_cast<const uint4*>(keys + i0);
            k[4 * x] = v.x;
            k[4 * x + 1] = v.y;
            k[4 * x + 2] = v.z;
            k[4 * x + 3] = v.w;
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) k[4 * x + c] = i0 + c < n ? keys[i0 + c] : 0xffffffffu;
        }
    }
    for (uint32_t i = threadIdx.x; i < kSubs * nd; i += kTileThreads) h[i] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kTile / kTileThreads; ++j) {
        // k[4x + c] is key x * kRound + 4 * threadIdx.x + c of the tile
        const uint32_t q = ((uint32_t)(j / 4) * kRound + 4u * threadIdx.x) / kSubTile;
        if (k[j] != 0xffffffffu) atomicAdd(&h[q * nd + ((k[j] >> shift) & (nd - 1))], 1u);
    }
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < nd; d += kTileThreads) {
        uint32_t q[kSubs], tot = 0;
#pragma unroll
        for (int x = 0; x < kSubs; ++x) {
            q[x] = h[x * nd + d];
            tot += q[x];
        }
        uint32_t r = tot ? atomicAdd(&acc[acc_at(d, blockIdx.x % kGroups)], tot) : 0u;
#pragma unroll
        for (int x = 0; x < kSubs; ++x) {
            __hip_atomic_store(&off[((uint64_t)blockIdx.x * kSubs + x) * nd + d], r, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            r += q[x];
        }
    }
}

// ---- scatter: 4096-key sub-tiles, composites into their bucket.
// Workgroups are dispatched round-robin over the 8 XCDs (block b on XCD b%8)
// and the L2 of one XCD is not coherent with the others', so a cache line
// written from two XCDs reaches HBM as two partial writes.  The two halves
// of one histogram tile own consecutive sub-ranges of every bucket; mapping
// them onto one XCD lets its L2 merge their writes into whole lines.
constexpr int kXcds = 8;
GPR_D uint32_t sub_of_block(uint32_t b) {
    const uint32_t g = b / kXcds, x = b % kXcds;
    const uint32_t t = (g / kSubs) * kXcds + x;
    return t * kSubs + g % kSubs;
}

template <bool WIDE>
__global__ __launch_bounds__(kScatterThreads) void k_scatter(const uint32_t* __restrict__ keys, uint32_t n,
                                                             uint32_t shift, uint32_t nd,
                                                             const uint32_t* __restrict__ acc,
                                                             const uint32_t* __restrict__ off,
                                                             uint2* __restrict__ bases,
                                                             unsigned long long* __restrict__ tmp) {
    constexpr int NT = kScatterThreads, KPT = kSubTile / NT;
    constexpr int kPer = kMaxDigits / NT;  // digits per thread at most
    static_assert(kSubTile % NT == 0 && kMaxDigits % NT == 0, "whole keys and digits per thread");
    __shared__ uint32_t gpos[kMaxDigits];  // global slot of digit d's first element, minus its local start
    __shared__ uint32_t lcnt[kMaxDigits];  // digit counts of the sub-tile, then local starts
    __shared__ unsigned long long stage[kSubTile];
    __shared__ uint32_t sh[2 * NT / 64];
    __shared__ uint32_t pieces;
    const uint32_t sub = sub_of_block(blockIdx.x);
    const uint64_t b0 = (uint64_t)sub * kSubTile;
    if (b0 >= n) return;  // padding blocks of the XCD mapping
    // every global load is issued before the first dependent use
    uint32_t k[KPT];
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
        const uint64_t i = b0 + j * NT + threadIdx.x;
        k[j] = i < n ? keys[i] : 0u;
    }
    // thread t owns digits per*t .. per*t + per - 1 (nd is a power of two:
    // either a multiple of NT or below it, then one digit for threads < nd)
    const uint32_t per = nd >= (uint32_t)NT ? nd / NT : 1u;
    const bool owns = threadIdx.x * per < nd;
    const uint32_t d0 = threadIdx.x * per;
    // digit d's total over all groups, and the part of it in groups before
    // this tile's (the tile's range of bucket d follows those groups' ranges)
    const uint32_t grp = (sub / kSubs) % kGroups;
    const uint32_t* offs = off + (uint64_t)sub * nd;
    uint32_t a[kPer], p[kPer], o[kPer];
#pragma unroll
    for (int x = 0; x < kPer; ++x) {
        a[x] = p[x] = o[x] = 0u;
        if (owns && (uint32_t)x < per) {
            uint32_t g[kGroups];
#pragma unroll
            for (int y = 0; y < kGroups; ++y) g[y] = acc[acc_at(d0 + x, y)];
#pragma unroll
            for (int y = 0; y < kGroups; ++y) {
                p[x] += (uint32_t)y < grp ? g[y] : 0u;
                a[x] += g[y];
            }
            o[x] = offs[d0 + x];
        }
    }
    for (uint32_t d = threadIdx.x; d < nd; d += NT) lcnt[d] = 0;
    if (threadIdx.x == 0) pieces = 0;
    __syncthreads();
    // rank of every key among the sub-tile's keys of its digit
    uint32_t r[KPT];
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
        const uint64_t i = b0 + j * NT + threadIdx.x;
        r[j] = i < n ? atomicAdd(&lcnt[(k[j] >> shift) & (nd - 1)], 1u) : 0u;
    }
    __syncthreads();
    uint32_t l[kPer], ex = 0, lex = 0;
#pragma unroll
    for (int x = 0; x < kPer; ++x) {
        l[x] = owns && (uint32_t)x < per ? lcnt[d0 + x] : 0u;
        ex += a[x];
        lex += l[x];
    }
    // bucket bases (exclusive scan of the digit totals) and the sub-tile's
    // digit starts (exclusive scan of its digit counts) in one pass
    const uint32_t ta = ex, tl = lex;
    scan_incl2<NT>(ex, lex, sh);
    ex -= ta;
    lex -= tl;
    if (owns) {
#pragma unroll
        for (int x = 0; x < kPer; ++x) {
            if ((uint32_t)x < per) {
                lcnt[d0 + x] = lex;
                gpos[d0 + x] = ex + p[x] + o[x] - lex;
                if (sub == 0) {
                    bases[d0 + x] = make_uint2(ex, a[x]);
                }
                ex += a[x];
                lex += l[x];
            }
        }
    }
    __syncthreads();
    // stage the composites in digit order, then write them with consecutive
    // lanes on consecutive slots of each digit's run
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
        const uint64_t i = b0 + j * NT + threadIdx.x;
        if (i < n)
            stage[lcnt[(k[j] >> shift) & (nd - 1)] + r[j]] = ((unsigned long long)k[j] << 32) | (unsigned long long)i;
    }
    __syncthreads();
    const uint32_t m = (uint32_t)min<uint64_t>(kSubTile, n - b0);
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
        const uint32_t q = j * NT + threadIdx.x;
        if (q < m) {
            const unsigned long long w = stage[q];
            __hip_atomic_store(&tmp[gpos[(uint32_t)(w >> (32 + shift)) & (nd - 1)] + q], w, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (sub == 0) {
        uint32_t large = 0;
#pragma unroll
        for (int x = 0; x < kPer; ++x) large += pieces_of<WIDE>(a[x]);
        if (large) atomicAdd(&pieces, large);
        __syncthreads();
        if (threadIdx.x == 0) bases[kMaxDigits] = make_uint2(pieces, 0u);
    }
}

// f(entry) for the n entries at src, in 16-byte loads, kBatch of them in
// flight per thread.
template <int NT, class F>
GPR_D void each_entry(const unsigned long long* src, uint32_t n, F&& f) {
    constexpr uint32_t kBatch = 4;
    const uint32_t head = (uint32_t)(reinterpret_cast<uintptr_t>(src) >> 3) & 1u;  // 1: the first pair starts before src
    const ulonglong2* p = reinterpret_cast<const ulonglong2*>(src - head);
    const uint32_t end = n + head, pairs = (end + 1) / 2;
    for (uint32_t base = 0; base < pairs; base += kBatch * NT) {
        ulonglong2 v[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const uint32_t i = base + j * NT + threadIdx.x;
            v[j] = i < pairs ? p[i] : make_ulonglong2(0, 0);
        }
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const uint32_t e = 2 * (base + j * NT + threadIdx.x);
            if (e >= head && e < end) f(v[j].x);
            if (e + 1 < end) f(v[j].y);
        }
    }
}

// A range of a bucket: the entries whose bits under `mask` are `value`, with
// `base` entries of the bucket below them.
struct SortNode {
    unsigned long long mask, value;
    uint32_t base;
};
template <int NT, uint32_t STEP>
struct PieceLds {
    // ranges of a piece yet to do: each of seven levels takes one and adds those of
    // more than kRankMax entries that reach into the piece
    static constexpr uint32_t kMaxTodo = 1 + 7 * (1 + (STEP - 1) / (kRankMax + 1));
    static constexpr uint32_t kMax = STEP + kRankMax;  // entries of a piece at most
    unsigned long long buf[kMax + kSub / 2];           // its entries, then its sub-buckets' places
    uint32_t cnt[kSub], start[kSub];
    // Every scan of a bucket reads the wave sums, 16 bytes at a time if they lie
    // so; four bytes off, as eight 4-byte words, 1M uniform keys took 18.43 us, now 18.29.
    alignas(16) uint32_t sh[NT / 64];
    uint32_t end;                                 // of the last sub-bucket
    SortNode todo[kMaxTodo];
    uint32_t ntodo;
    unsigned long long all, any;  // AND and OR of a range's entries
    uint32_t piece[3];            // of the piece: first slot and size of its bucket, its number in the bucket
};
using LocalLds = PieceLds<kLocalThreads, kWinStep>;
using WideLds = PieceLds<kWideThreads, kWideStep>;
static_assert(offsetof(LocalLds, sh) % 16 == 0 && offsetof(WideLds, sh) % 16 == 0, "the wave sums are read 16 bytes at a time");
// Piece q of a bucket of n composites at src (any order): what belongs at its
// places q * STEP to (q + 1) * STEP, in whole sub-buckets.  The block
// counts a range's sub-buckets, the bucket's own by the key bits below the top
// digit.  Those of up to kRankMax entries that start in the piece it collects
// in LDS and places by rank; larger ones that the piece overlaps are ranges of
// their own, split by the highest 10 bits in which their entries differ
// (composites are all different, so this ends).
// The bucket is read twice for every piece, and three times more for a range
// inside it.  That costs less than a split by one block with its windows one
// after another, which made a bucket take the time of one compute unit, and no
// block waits for another.  One
// block a bucket against this: 1M / 399,952 / 20,000 keys in 64 clusters 11.1 ms /
// 6,861 us / 305 us -> 427 / 266 / 52; 1M equal keys 58.4 -> 2.5 ms; a rebuild of the
// 254K-triangle sphere grid 208 -> 190 us.
template <int NT, uint32_t STEP>
GPR_D void sort_piece(const unsigned long long* src, uint32_t n, uint32_t q, uint32_t sub_shift, uint32_t nsub,
                      uint32_t* __restrict__ skeys, uint32_t* __restrict__ sidx, PieceLds<NT, STEP>& L) {
    const uint32_t p0 = q * STEP, p1 = p0 + STEP;
    uint32_t* at_of = reinterpret_cast<uint32_t*>(L.buf + L.kMax);  // a sub-bucket's place in the buffer
    __syncthreads();  // the LDS is free
    if (threadIdx.x == 0) {
        L.todo[0] = SortNode{0ull, 0ull, 0u};
        L.ntodo = 1;
    }
    __syncthreads();
    for (bool whole = true;; whole = false) {
        const uint32_t left = L.ntodo;
        if (left == 0) break;
        const SortNode node = L.todo[left - 1];
        __syncthreads();
        for (uint32_t s = threadIdx.x; s < kSub; s += NT) L.cnt[s] = 0;
        if (threadIdx.x == 0) {
            L.ntodo = left - 1;
            L.all = ~0ull;
            L.any = 0ull;
        }
        __syncthreads();
        const auto inside = [&](unsigned long long v) { return (v & node.mask) == node.value; };
        uint32_t shift = sub_shift, nd = nsub;
        if (!whole) {
            unsigned long long all = ~0ull, any = 0ull;
            each_entry<NT>(src, n, [&](unsigned long long v) {
                all &= inside(v) ? v : ~0ull;
                any |= inside(v) ? v : 0ull;
            });
            atomicAnd(&L.all, all);
            atomicOr(&L.any, any);
            __syncthreads();
            const uint32_t top = 63u - (uint32_t)__clzll((long long)(L.all ^ L.any));
            shift = top > 9u ? top - 9u : 0u;
            nd = 2u << (top - shift);
        }
        const auto digit = [&](unsigned long long v) { return (uint32_t)(v >> shift) & (nd - 1); };
        each_entry<NT>(src, n, [&](unsigned long long v) {
            if (!inside(v)) return;
            // equal digits in a whole wave: one atomic
            const uint32_t d = digit(v), d0 = __builtin_amdgcn_readfirstlane(d);
            const unsigned long long here = __ballot(true);
            if (__ballot(d == d0) != here) atomicAdd(&L.cnt[d], 1u);
            else if ((threadIdx.x & 63) == (uint32_t)__builtin_ctzll(here)) atomicAdd(&L.cnt[d], (uint32_t)__popcll(here));
        });
        __syncthreads();
        constexpr int kQ = kSub / NT;
        uint32_t c[kQ], sum = 0, tot;
#pragma unroll
        for (int k = 0; k < kQ; ++k) sum += c[k] = L.cnt[kQ * threadIdx.x + k];
        const uint32_t size_end = scan_incl<NT>(sum, L.sh, &tot);
        // the sub-buckets that start in the piece, and the large ones that reach into it
        uint32_t first = node.base + size_end - sum, mine = 0, at[kQ];
#pragma unroll
        for (int k = 0; k < kQ; ++k) {
            const uint32_t d = kQ * threadIdx.x + k;
            L.start[d] = first;
            at[k] = ~0u;
            if (c[k] > kRankMax) {
                if (first < p1 && first + c[k] > p0)
                    L.todo[atomicAdd(&L.ntodo, 1u)] =
                        SortNode{node.mask | (unsigned long long)(nd - 1) << shift,
                                 node.value | (unsigned long long)d << shift, first};
            } else if (c[k] != 0 && first >= p0 && first < p1) {
                at[k] = mine;
                mine += c[k];
            }
            first += c[k];
        }
        if (threadIdx.x == NT - 1) L.end = first;
        const uint32_t mine_end = scan_incl<NT>(mine, L.sh, &tot);
#pragma unroll
        for (int k = 0; k < kQ; ++k) at_of[kQ * threadIdx.x + k] = at[k] == ~0u ? ~0u : at[k] + mine_end - mine;
        const uint32_t m = tot;
        __syncthreads();
        if (m == 0) continue;
        each_entry<NT>(src, n, [&](unsigned long long v) {
            const uint32_t d = digit(v);
            if (inside(v) && at_of[d] != ~0u) L.buf[at_of[d] + atomicSub(&L.cnt[d], 1u) - 1u] = v;
        });
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < m; j += NT) {
            const unsigned long long v = L.buf[j];
            const uint32_t d = digit(v), b = at_of[d];
            // 8 independent LDS reads per step: the loop is bound by LDS
            // latency, not by the compares
            const uint32_t e = (d + 1 < (uint32_t)kSub ? L.start[d + 1] : L.end) - L.start[d];
            uint32_t rank = 0, x = 0;
            for (; x + 8 <= e; x += 8) {
                unsigned long long a[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) a[u] = L.buf[b + x + u];
#pragma unroll
                for (int u = 0; u < 8; ++u) rank += a[u] < v ? 1u : 0u;
            }
            for (; x < e; ++x) rank += L.buf[b + x] < v ? 1u : 0u;
            __hip_atomic_store(&skeys[L.start[d] + rank], (uint32_t)(v >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&sidx[L.start[d] + rank], (uint32_t)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
    }
}

// The pieces dealt out: block takes every nd-th.
template <bool WIDE, int NT, uint32_t STEP>
GPR_D void deal_pieces(uint32_t pieces, uint32_t block, uint32_t nd, uint32_t sub_shift, uint32_t nsub,
                       const uint2* __restrict__ bases, const unsigned long long* __restrict__ tmp,
                       uint32_t* __restrict__ skeys, uint32_t* __restrict__ sidx, PieceLds<NT, STEP>& L) {
    constexpr int kDigits = kMaxDigits / NT;  // digits per thread at most
    const uint32_t per = nd >= (uint32_t)NT ? nd / NT : 1u;
    for (uint32_t w = block; w < pieces; w += nd) {
        uint2 l[kDigits];
        uint32_t sum = 0, tot;
#pragma unroll
        for (int x = 0; x < kDigits; ++x) {
            const uint32_t i = threadIdx.x * per + x;
            l[x] = (uint32_t)x < per && i < nd ? bases[i] : make_uint2(0u, 0u);
            sum += pieces_of<WIDE>(l[x].y);
        }
        __syncthreads();  // the LDS is free
        uint32_t first = scan_incl<NT>(sum, L.sh, &tot) - sum;
#pragma unroll
        for (int x = 0; x < kDigits; ++x) {
            const uint32_t k = pieces_of<WIDE>(l[x].y);
            if (w - first < k) {
                L.piece[0] = l[x].x;
                L.piece[1] = l[x].y;
                L.piece[2] = w - first + (WIDE ? 1u : 0u);
            }
            first += k;
        }
        __syncthreads();
        const uint32_t p0 = L.piece[0];
        sort_piece(tmp + p0, L.piece[1], L.piece[2], sub_shift, nsub, skeys + p0, sidx + p0, L);
    }
}

// ---- local: one bucket per block, LDS MSD split + rank inside each
// sub-bucket; then the block's share of the pieces of the large buckets
__global__ __launch_bounds__(kLocalThreads, 8) void k_local(uint32_t shift, uint32_t nd, uint32_t* __restrict__ acc,
                                                         const uint2* __restrict__ bases,
                                                         const unsigned long long* __restrict__ tmp,
                                                         uint32_t* __restrict__ skeys,
                                                         uint32_t* __restrict__ sidx) {
    __shared__ LocalLds L;
    unsigned long long* buf = L.buf;  // A | B
    uint32_t* cnt = L.cnt;
    uint32_t* start = L.start;
    uint32_t* sh = L.sh;
    __shared__ uint32_t crowded;
    const uint32_t d = blockIdx.x;
    // the bucket's base and size, as the scatter pass computed them
    const uint2 bn = bases[d];
    const uint32_t b0 = bn.x, n = bn.y;
    const uint32_t pieces = bases[kMaxDigits].x;  // of all buckets
    // the reservation counters start from zero in the next call
    if (threadIdx.x < kGroups) acc[acc_at(d, threadIdx.x)] = 0u;
    if (n == 0 && __builtin_expect(pieces == 0, 1)) return;
    const unsigned long long* src = tmp + b0;
    const uint32_t sub_bits = min(10u, shift);
    const uint32_t nsub = 1u << sub_bits;
    const uint32_t sub_shift = 32 + shift - sub_bits;
    if (n != 0 && n <= (uint32_t)kFastCap) {
        unsigned long long* A = buf;
        unsigned long long* B = buf + kFastCap;
        // all loads in flight before the first LDS use
        constexpr int kPer = (kFastCap + kLocalThreads - 1) / kLocalThreads;
        unsigned long long v[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const uint32_t i = j * kLocalThreads + threadIdx.x;
            v[j] = i < n ? src[i] : 0ull;
        }
        for (uint32_t s = threadIdx.x; s < kSub; s += kLocalThreads) cnt[s] = 0;
        if (threadIdx.x == 0) crowded = 0;
        __syncthreads();
        uint32_t r[kPer], sb[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const uint32_t i = j * kLocalThreads + threadIdx.x;
            sb[j] = (uint32_t)(v[j] >> sub_shift) & (nsub - 1);
            r[j] = i < n ? atomicAdd(&cnt[sb[j]], 1u) : 0u;
        }
        __syncthreads();
        constexpr int kQ = kSub / kLocalThreads;  // sub-bucket counts scanned per thread
        uint32_t cq[kQ], sq = 0;
#pragma unroll
        for (int k = 0; k < kQ; ++k) {
            cq[k] = cnt[kQ * threadIdx.x + k];
            sq += cq[k];
            if (cq[k] > kSubMax) crowded = 1;
        }
        uint32_t tot;
        uint32_t run = scan_incl<kLocalThreads>(sq, sh, &tot) - sq;
#pragma unroll
        for (int k = 0; k < kQ; ++k) {
            start[kQ * threadIdx.x + k] = run;
            run += cq[k];
        }
        __syncthreads();
        if (!crowded) {
            // sub-bucket order (arrival order inside each sub-bucket) ...
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const uint32_t i = j * kLocalThreads + threadIdx.x;
                if (i < n) A[start[sb[j]] + r[j]] = v[j];
            }
            __syncthreads();
            // ... then every composite's rank among its sub-bucket (all distinct)
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const uint32_t i = j * kLocalThreads + threadIdx.x;
                if (i < n) {
                    // rank among the sub-bucket: its first kWin entries are read
                    // together (independent LDS loads); longer sub-buckets continue
                    const uint32_t b = start[sb[j]], c = cnt[sb[j]];
                    uint32_t rank = 0;
#pragma unroll
                    for (uint32_t x = 0; x < kWin; ++x) {
                        const unsigned long long a = A[min(b + x, (uint32_t)kFastCap - 1)];
                        rank += (x < c && a < v[j]) ? 1u : 0u;
                    }
                    for (uint32_t x = kWin; x < c; ++x) rank += A[b + x] < v[j] ? 1u : 0u;
                    B[b + rank] = v[j];
                }
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const uint32_t i = j * kLocalThreads + threadIdx.x;
                if (i < n) {
                    const unsigned long long w = B[i];
                    __hip_atomic_store(&skeys[b0 + i], (uint32_t)(w >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(&sidx[b0 + i], (uint32_t)w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            if (__builtin_expect(pieces == 0, 1)) return;
        } else {
            sort_piece(src, n, 0, sub_shift, nsub, skeys + b0, sidx + b0, L);
        }
    }
    deal_pieces<false, kLocalThreads, kWinStep>(pieces, d, nd, sub_shift, nsub, bases, tmp, skeys, sidx, L);
}

// ---- the same for buckets that are large as a rule
__global__ __launch_bounds__(kWideThreads, 4) void k_local_wide(uint32_t shift, uint32_t nd, uint32_t* __restrict__ acc,
                                                             const uint2* __restrict__ bases,
                                                             const unsigned long long* __restrict__ tmp,
                                                             uint32_t* __restrict__ skeys,
                                                             uint32_t* __restrict__ sidx) {
    __shared__ WideLds L;
    const uint32_t d = blockIdx.x;
    const uint2 bn = bases[d];
    const uint32_t pieces = bases[kMaxDigits].x;
    if (threadIdx.x < kGroups) acc[acc_at(d, threadIdx.x)] = 0u;
    const uint32_t sub_bits = min(10u, shift), nsub = 1u << sub_bits, sub_shift = 32 + shift - sub_bits;
    if (bn.y) sort_piece(tmp + bn.x, bn.y, 0, sub_shift, nsub, skeys + bn.x, sidx + bn.x, L);
    deal_pieces<true>(pieces, d, nd, sub_shift, nsub, bases, tmp, skeys, sidx, L);
}

// ---- the sort of many keys: three stable passes over 10 bits each, low bits
// first, so its cost does not depend on how the keys are spread.
// Every pass counts the digits of its tiles, turns the counts into starts (a
// block takes 16 digits over all tiles), and scatters: a wave ranks its 64 keys
// against each other with ballots and against its earlier ones with a count per
// wave and digit, so equal digits keep their order.  The tile is then put into
// digit order in LDS and leaves in runs of 64 bytes at 8 keys a digit; tiles
// that follow each other run on one XCD, whose L2 joins their runs.  16.8M keys
// take 409 us, three times a scatter of 100, a count of 21 and starts of 14; the
// traffic of 64 bytes a key would take 250: a scatter block has a compute unit to
// itself (two, with 64 registers, spill: 514 us).
constexpr int kRadix = 1024;
constexpr int kRadixBits = 10;
constexpr int kRadixPasses = 3;
constexpr int kRadixThreads = 1024;
constexpr int kRadixWaves = kRadixThreads / 64;
constexpr int kRadixKeys = kTile / kRadixThreads;  // keys per thread
constexpr int kStartDigits = 16, kStartChunks = 1024 / kStartDigits;
static_assert(kRadix == kRadixThreads, "a thread owns a digit");

template <bool FIRST>
__global__ __launch_bounds__(kRadixThreads) void k_radix_count(const uint32_t* __restrict__ keys,
                                                               const unsigned long long* __restrict__ src, uint32_t n,
                                                               uint32_t shift, uint32_t* __restrict__ cnt) {
    __shared__ uint32_t h[kRadix];
    const uint64_t b0 = (uint64_t)blockIdx.x * kTile;
    h[threadIdx.x] = 0;
    uint32_t k[kRadixKeys];
#pragma unroll
    for (int j = 0; j < kRadixKeys; ++j) {
        const uint64_t i = b0 + j * kRadixThreads + threadIdx.x;
        k[j] = i >= n ? 0u : FIRST ? keys[i] : (uint32_t)(src[i] >> 32);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRadixKeys; ++j) {
        if (b0 + j * kRadixThreads + threadIdx.x >= n) continue;
        const uint32_t d = (k[j] >> shift) & (kRadix - 1), d0 = __builtin_amdgcn_readfirstlane(d);
        const unsigned long long here = __ballot(true);  // equal digits in a whole wave: one atomic
        if (__ballot(d == d0) != here) atomicAdd(&h[d], 1u);
        else if ((threadIdx.x & 63) == (uint32_t)__builtin_ctzll(here)) atomicAdd(&h[d], (uint32_t)__popcll(here));
    }
    __syncthreads();
    cnt[(uint64_t)blockIdx.x * kRadix + threadIdx.x] = h[threadIdx.x];
}

// Counts to starts inside their digit, and every digit's total.
__global__ __launch_bounds__(1024) void k_radix_starts(uint32_t* __restrict__ cnt, uint32_t ntiles,
                                                       uint32_t* __restrict__ total) {
    __shared__ uint32_t sums[kStartChunks][kStartDigits];
    const uint32_t dd = threadIdx.x % kStartDigits, d = blockIdx.x * kStartDigits + dd;
    const uint32_t chunk = threadIdx.x / kStartDigits, per = (ntiles + kStartChunks - 1) / kStartChunks;
    const uint32_t t0 = min(chunk * per, ntiles), t1 = min(t0 + per, ntiles);
    uint32_t sum = 0;
    constexpr uint32_t kBatch = 8;  // reads in flight per thread
    for (uint32_t t = t0; t < t1; t += kBatch) {
        uint32_t c[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) c[j] = t + j < t1 ? cnt[(uint64_t)(t + j) * kRadix + d] : 0u;
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) sum += c[j];
    }
    sums[chunk][dd] = sum;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (uint32_t c = 0; c < kStartChunks; ++c) {
        const uint32_t x = sums[c][dd];
        before += c < chunk ? x : 0u;
        all += x;
    }
    if (chunk == 0) total[d] = all;
    for (uint32_t t = t0; t < t1; t += kBatch) {
        uint32_t c[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) c[j] = t + j < t1 ? cnt[(uint64_t)(t + j) * kRadix + d] : 0u;
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            if (t + j < t1) cnt[(uint64_t)(t + j) * kRadix + d] = before;
            before += c[j];
        }
    }
}

template <bool FIRST, bool LAST>
__global__ __launch_bounds__(kRadixThreads) void k_radix_scatter(
    const uint32_t* __restrict__ keys, const unsigned long long* __restrict__ src, uint32_t n, uint32_t shift,
    uint32_t ntiles, const uint32_t* __restrict__ starts, const uint32_t* __restrict__ total,
    unsigned long long* __restrict__ dst, uint32_t* __restrict__ skeys, uint32_t* __restrict__ sidx) {
    // the waves' counts are read before the tile takes their place
    __shared__ union {
        uint16_t wave[kRadixWaves][kRadix];
        unsigned long long tile[kTile];
    } L;
    __shared__ uint32_t lstart[kRadix], gpos[kRadix];
    __shared__ uint32_t sh[2 * kRadixWaves];
    const uint32_t per = (ntiles + kXcds - 1) / kXcds, t = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (t >= ntiles) return;  // a whole block: the grid is padded to kXcds * per
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    const uint64_t b0 = (uint64_t)t * kTile;
    const uint32_t m = (uint32_t)min<uint64_t>(kTile, n - b0), at = wave * (64 * kRadixKeys) + lane;
    unsigned long long v[kRadixKeys];
#pragma unroll
    for (int j = 0; j < kRadixKeys; ++j) {
        const uint32_t q = at + 64 * j;
        v[j] = q >= m ? 0ull : FIRST ? (unsigned long long)keys[b0 + q] << 32 | (b0 + q) : src[b0 + q];
    }
    const uint32_t tot = total[threadIdx.x], start = starts[(uint64_t)t * kRadix + threadIdx.x];
    for (uint32_t i = threadIdx.x; i < kRadixWaves * kRadix / 2; i += kRadixThreads)
        reinterpret_cast<uint32_t*>(&L.wave[0][0])[i] = 0u;
    __syncthreads();
    uint32_t r[kRadixKeys];
#pragma unroll
    for (int j = 0; j < kRadixKeys; ++j) {
        const uint32_t d = (uint32_t)(v[j] >> (32 + shift)) & (kRadix - 1);
        const bool valid = at + 64 * j < m;
        const unsigned long long live = __ballot(valid);
        uint32_t lo = (uint32_t)live, hi = (uint32_t)(live >> 32);  // lanes with this lane's digit
#pragma unroll
        for (int b = 0; b < kRadixBits; ++b) {
            const uint32_t bit = 0u - (d >> b & 1u);
            const unsigned long long ones = __ballot(bit != 0);
            lo &= ~((uint32_t)ones ^ bit);
            hi &= ~((uint32_t)(ones >> 32) ^ bit);
        }
        const uint32_t before = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
        const uint32_t had = L.wave[wave][d];
        r[j] = had + before;
        // other lanes' counts are read before they change and seen after
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid && before == 0) L.wave[wave][d] = (uint16_t)(had + __popc(lo) + __popc(hi));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);  // a round's masks are not kept beside the next one's
    }
    __syncthreads();
    // digit threadIdx.x: where each wave's keys start among the tile's
    uint32_t mine = 0;
#pragma unroll
    for (int w = 0; w < kRadixWaves; ++w) {
        const uint32_t c = L.wave[w][threadIdx.x];
        L.wave[w][threadIdx.x] = (uint16_t)mine;
        mine += c;
    }
    uint32_t first = mine, base = tot;
    scan_incl2<kRadixThreads>(first, base, sh);
    first -= mine;
    lstart[threadIdx.x] = first;
    gpos[threadIdx.x] = base - tot + start - first;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRadixKeys; ++j) {
        const uint32_t d = (uint32_t)(v[j] >> (32 + shift)) & (kRadix - 1);
        r[j] += lstart[d] + L.wave[wave][d];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRadixKeys; ++j)
        if (at + 64 * j < m) L.tile[r[j]] = v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRadixKeys; ++j) {
        const uint32_t q = j * kRadixThreads + threadIdx.x;
        if (q >= m) continue;
        const unsigned long long w = L.tile[q];
        const uint32_t to = gpos[(uint32_t)(w >> (32 + shift)) & (kRadix - 1)] + q;
        if constexpr (LAST) {
            skeys[to] = (uint32_t)(w >> 32);
            sidx[to] = (uint32_t)w;
        } else {
            dst[to] = w;
        }
    }
}

struct Layout {
    uint32_t* acc;
    uint2* bases;     // per bucket: first slot, size; then the pieces of all large buckets
    uint32_t* off;    // radix passes: the tiles' counts and starts
    unsigned long long* tmp;
    unsigned long long* alt;  // radix passes only
};
// Byte offsets of the scratch arrays for n keys, each on a 256-B boundary
// (constexpr: the no-allocation entry point sizes its fixed array with it).
struct Offsets {
    size_t acc, bases, off, tmp, alt, total;
};
constexpr size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }
constexpr Offsets offsets(uint32_t n) {
    const uint64_t ntiles = n > (uint32_t)kTile ? ((uint64_t)n + kTile - 1) / kTile : 1;
    const uint64_t nk = n ? n : 1;
    Offsets o{};
    o.acc = 0;
    o.bases = align256(o.acc + 4ull * kAccWords);
    o.off = align256(o.bases + 8ull * (kMaxDigits + 1));
    o.tmp = align256(o.off + 4ull * kMaxDigits * kSubs * ntiles);
    o.alt = align256(o.tmp + 8ull * nk);
    o.total = o.alt + (n > kRadixMin ? 8ull * nk : 0ull) + 256;
    return o;
}
size_t layout(uint32_t n, char* base, Layout* L) {
    const Offsets o = offsets(n);
    if (L) {
        L->acc = reinterpret_cast<uint32_t*>(base + o.acc);
        L->bases = reinterpret_cast<uint2*>(base + o.bases);
        L->off = reinterpret_cast<uint32_t*>(base + o.off);
        L->tmp = reinterpret_cast<unsigned long long*>(base + o.tmp);
        L->alt = reinterpret_cast<unsigned long long*>(base + o.alt);
    }
    return o.total;
}

// zero fill of n words (graph-capturable, unlike a memset node)
__global__ __launch_bounds__(1024) void k_clear_words(uint32_t* __restrict__ p, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

}  // namespace

size_t sort_scratch_bytes(uint32_t n) { return layout(n, nullptr, nullptr); }

int sort_prepare(void* scratch, size_t bytes, hipStream_t st) {
    // the digit totals (the first array of the layout) start cleared; afterwards
    // every call clears them after use
    GPR_HIP(hipMemsetAsync(scratch, 0, std::min<size_t>(bytes, 4ull * kAccWords), st));
    return GPR_OK;
}

namespace {
void radix_sort(const uint32_t* keys, uint32_t* skeys, uint32_t* sidx, uint32_t n, const Layout& L, hipStream_t st) {
    const uint32_t ntiles = div_up(n, kTile), blocks = div_up(ntiles, kXcds) * kXcds;
    uint32_t* total = reinterpret_cast<uint32_t*>(L.bases);
    static_assert(4 * kRadix <= 8 * kMaxDigits && kRadix <= kMaxDigits * kSubs, "totals and counts fit the MSD sort's arrays");
    const auto pass = [&](auto count, auto scatter, const unsigned long long* src, uint32_t shift, unsigned long long* dst) {
        hipLaunchKernelGGL(count, dim3(ntiles), dim3(kRadixThreads), 0, st, keys, src, n, shift, L.off);
        hipLaunchKernelGGL(k_radix_starts, dim3(kRadix / kStartDigits), dim3(1024), 0, st, L.off, ntiles, total);
        hipLaunchKernelGGL(scatter, dim3(blocks), dim3(kRadixThreads), 0, st, keys, src, n, shift, ntiles, L.off, total,
                           dst, skeys, sidx);
    };
    pass(k_radix_count<true>, k_radix_scatter<true, false>, nullptr, 0, L.tmp);
    pass(k_radix_count<false>, k_radix_scatter<false, false>, L.tmp, kRadixBits, L.alt);
    pass(k_radix_count<false>, k_radix_scatter<false, true>, L.alt, 2 * kRadixBits, nullptr);
    static_assert(kRadixPasses * kRadixBits == 30, "the passes cover a key");
}
}  // namespace

int sort_pairs(const uint32_t* keys, uint32_t* skeys, uint32_t* sidx, uint32_t n, void* scratch,
               size_t scratch_bytes, hipStream_t st) {
    if (n == 0) return GPR_OK;
    if (scratch_bytes < sort_scratch_bytes(n)) return fail(GPR_ERR_INVALID, "sort scratch too small");
    Layout L;
    layout(n, reinterpret_cast<char*>(scratch), &L);
    if (n > kRadixMin) {
        radix_sort(keys, skeys, sidx, n, L, st);
        GPR_HIP(hipGetLastError());
        return GPR_OK;
    }
    const uint32_t dbits = digit_bits(n);
    const uint32_t nd = 1u << dbits, shift = 30 - dbits;
    const uint32_t ntiles = div_up(n, kTile);
    hipLaunchKernelGGL(k_hist, dim3(ntiles), dim3(kTileThreads), 0, st, keys, n, shift, nd, L.acc, L.off);
    // grid padded to whole groups of kXcds tiles for the XCD mapping
    const uint32_t nsub_blocks = div_up(ntiles, kXcds) * kXcds * kSubs;
    const bool wide = n > kWideMin;
    hipLaunchKernelGGL(wide ? k_scatter<true> : k_scatter<false>, dim3(nsub_blocks), dim3(kScatterThreads), 0, st, keys, n,
                       shift, nd, L.acc, L.off, L.bases, L.tmp);
    hipLaunchKernelGGL(wide ? k_local_wide : k_local, dim3(nd), dim3(wide ? kWideThreads : kLocalThreads), 0, st, shift, nd,
                       L.acc, L.bases, L.tmp, skeys, sidx);
    GPR_HIP(hipGetLastError());
    return GPR_OK;
}

}  // namespace gpr

// ---- the sort without allocation ------------------------------------------
// A fixed device array holds the scratch of sorts of up to kNoAllocMaxKeys
// keys, so gpr_sort_pairs_device_noalloc calls neither hipMalloc nor hipFree.
// Each GPU holds its own copy of the array until the process ends (10.5 MB);
// every call on a GPU shares it.
namespace {
constexpr uint32_t kNoAllocMaxKeys = 1u << 20;
constexpr size_t kNoAllocBytes = gpr::offsets(kNoAllocMaxKeys).total;
constexpr int kMaxDevices = 16;
std::mutex g_noalloc_mu;
void* g_noalloc_ptr[kMaxDevices] = {};
}  // namespace

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

namespace {
// The array's device address on the current device, looked up once per device
// with that device current.  In host code `scratch` names a host-side stand-in,
// never the device memory: only this address is passed to kernels.
int noalloc_scratch(void** out) {
    int dev = 0;
    GPR_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices)
        return gpr::fail(GPR_ERR_INVALID, "gpr_sort_pairs_device_noalloc: device index outside 0..15");
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        void* p = nullptr;
        GPR_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return gpr::fail(GPR_ERR_HIP, "gpr_sort_pairs_device_noalloc: no device address for the scratch array");
        g_noalloc_ptr[dev] = p;
    }
    *out = g_noalloc_ptr[dev];
    return GPR_OK;
}
}  // namespace

int gpr_sort_pairs_device_noalloc(const uint32_t* keys, uint32_t* sk, uint32_t* si, uint32_t n) {
    using namespace gpr;
    if (n == 0) return GPR_OK;
    if (!keys || !sk || !si) return fail(GPR_ERR_INVALID, "gpr_sort_pairs_device_noalloc: null pointer");
    if (n > kNoAllocMaxKeys)
        return fail(GPR_ERR_INVALID, "gpr_sort_pairs_device_noalloc: n = " + std::to_string(n) +
                                         " exceeds the fixed scratch's maximum of " +
                                         std::to_string(kNoAllocMaxKeys) + " keys");
    if (sort_scratch_bytes(n) > kNoAllocBytes)
        return fail(GPR_ERR_INVALID, "gpr_sort_pairs_device_noalloc: scratch layout exceeds the fixed array");
    void* p = nullptr;
    GPR_TRY(noalloc_scratch(&p));
    // the digit totals start at zero whatever an earlier call left in the array
    hipLaunchKernelGGL(k_clear_words, dim3(2), dim3(1024), 0, stream(), reinterpret_cast<uint32_t*>(p),
                       (uint32_t)kAccWords);
    GPR_HIP(hipGetLastError());
    return sort_pairs(keys, sk, si, n, p, kNoAllocBytes, stream());
}
