// bvh_build.hip -- device LBVH construction for gfx950.
//
// Replaces the reference's single-threaded host builder LBVH_build
// (src/renderer/bvh.h:186-221) with an all-device pipeline that produces the
// same tree:
//   1. centroid bounds            (bvh.h:192-196)           two-level block reduction
//   2. 30-bit Morton keys         (bvh.h:12-32, 199-204)    one thread per triangle
//   3. (key, index) sort          (bvh.h:207-208)           LDS-staged MSD radix sort
//   4. split weights              (bvh.h:161-176)           adjacent-pair common prefix;
//      equal-key runs get 32 + the split depth of the reference's midpoint
//      rule ((l+r)>>1)-1, so the radix tree reproduces that rule exactly
//   5. tree + refit               (bvh.h:143-184)           bottom-up agglomerative build
//      (parent = deeper of the two boundary splits) fused with the box union,
//      in LDS for the subtrees inside 512 consecutive leaves
//   6. layouts                    (bvh.h:121-141)           reference DFS order via
//      pre-order index = 2*first_leaf + number_of_left_steps, and packed 128-B
//      BVH4 nodes (binary nodes at even depth) for the traversal kernels.
#include "dev_math.h"
#include "gpr_internal.h"

#include <algorithm>

namespace gpr {
namespace {

constexpr int kB = 256;              // threads per block
constexpr int kMaxDepth = 256;       // > 30 radix levels + 32 midpoint levels
constexpr int kTreeB = 512;          // leaves whose subtrees one block builds

inline uint32_t div_up(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// What a build leaves for the host, and the root for its later kernels.
struct BuildState {
    uint32_t nbvh4;  // BVH4 nodes numbered so far (the root is number 0)
    uint32_t ntop;   // published nodes listed by k_top
    uint32_t err;    // bit 0 inconsistent publication, 1 box mismatch, 2 node out of range
    uint32_t root;   // node id of the root
};

// Triangle::worldBound (src/renderer/triangle.h:96-101): Union(AABB(p0,p1), p2)
GPR_D void tri_bounds(const float* p, v3& lo, v3& hi) {
    const v3 p0 = load3(p), p1 = load3(p + 3), p2 = load3(p + 6);
    const v3 a = vmin3(p0, p1), b = vmax3(p0, p1);
    lo = vmin3(a, p2);
    hi = vmax3(b, p2);
}

// ------------------------------------------------------------ bounds ----
template <int NT>
GPR_D void block_minmax(v3& lo, v3& hi, float* sh) {
    const int t = threadIdx.x;
    sh[t * 6 + 0] = lo.x; sh[t * 6 + 1] = lo.y; sh[t * 6 + 2] = lo.z;
    sh[t * 6 + 3] = hi.x; sh[t * 6 + 4] = hi.y; sh[t * 6 + 5] = hi.z;
    __syncthreads();
    for (int s = NT / 2; s > 0; s >>= 1) {
        if (t < s) {
            for (int k = 0; k < 3; ++k) sh[t * 6 + k] = fmin_h(sh[t * 6 + k], sh[(t + s) * 6 + k]);
            for (int k = 3; k < 6; ++k) sh[t * 6 + k] = fmax_h(sh[t * 6 + k], sh[(t + s) * 6 + k]);
        }
        __syncthreads();
    }
    lo = V(sh[0], sh[1], sh[2]);
    hi = V(sh[3], sh[4], sh[5]);
}

__global__ __launch_bounds__(kB) void k_centroid_partial(const float* __restrict__ pos, uint32_t n,
                                                         float* __restrict__ part) {
    __shared__ float sh[kB * 6];
    v3 lo = V(INFINITY, INFINITY, INFINITY), hi = V(-INFINITY, -INFINITY, -INFINITY);
    for (uint32_t i = blockIdx.x * kB + threadIdx.x; i < n; i += gridDim.x * kB) {
        v3 a, b;
        tri_bounds(pos + 9ull * i, a, b);
        const v3 c = (a + b) * 0.5f;  // AABB::centroid (aabb.h:23)
        lo = vmin3(lo, c);
        hi = vmax3(hi, c);
    }
    block_minmax<kB>(lo, hi, sh);
    if (threadIdx.x == 0) {
        float* o = part + 6 * blockIdx.x;
        o[0] = lo.x; o[1] = lo.y; o[2] = lo.z; o[3] = hi.x; o[4] = hi.y; o[5] = hi.z;
    }
}

__global__ __launch_bounds__(kB) void k_centroid_final(const float* __restrict__ part, uint32_t np,
                                                       float* __restrict__ out, uint32_t first4,
                                                       BuildState* __restrict__ bs) {
    __shared__ float sh[kB * 6];
    v3 lo = V(INFINITY, INFINITY, INFINITY), hi = V(-INFINITY, -INFINITY, -INFINITY);
    for (uint32_t i = threadIdx.x; i < np; i += kB) {
        lo = vmin3(lo, load3(part + 6 * i));
        hi = vmax3(hi, load3(part + 6 * i + 3));
    }
    block_minmax<kB>(lo, hi, sh);
    if (threadIdx.x == 0) {
        *bs = BuildState{first4, 0u, 0u, 0u};
        out[0] = lo.x; out[1] = lo.y; out[2] = lo.z; out[3] = hi.x; out[4] = hi.y; out[5] = hi.z;
    }
}

// ------------------------------------------------------------ Morton ----
// LeftShift3 (bvh.h:12-25): 10 bits to every third bit, 1024 -> 1023.
GPR_D uint32_t spread3(uint32_t x) {
    x = x == 1024u ? 1023u : x;
    x = (x | (x << 16)) & 0x030000ffu;
    x = (x | (x << 8)) & 0x0300f00fu;
    x = (x | (x << 4)) & 0x030c30c3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}
// float -> uint truncation; NaN (flat axis, 0/0) -> 0.
GPR_D uint32_t quant(float v) {
    if (!(v == v) || v <= 0.0f) return 0u;
    return v >= 4294967040.0f ? 0xffffffffu : (uint32_t)v;
}

__global__ __launch_bounds__(kB) void k_morton(const float* __restrict__ pos, uint32_t n,
                                               const float* __restrict__ bounds,
                                               uint32_t* __restrict__ keys, uint32_t* __restrict__ arrive) {
    const uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= n) return;
    arrive[i] = 0u;
    const v3 lo = load3(bounds), hi = load3(bounds + 3);
    v3 a, b;
    tri_bounds(pos + 9ull * i, a, b);
    const v3 c = (a + b) * 0.5f;
    const v3 q = (c - lo) / (hi - lo) * 1024.f;  // EncodeMorton3 input (bvh.h:203)
    keys[i] = (spread3(quant(q.z)) << 2) | (spread3(quant(q.y)) << 1) | spread3(quant(q.x));
}

// ---------------------------------------------------------- weights -----
// Split depth of adjacent pair j in the reference's midpoint tree over a run
// of m equal keys: root split after floor(m/2) leaves (bvh.h:162-165).
GPR_D uint32_t midpoint_depth(uint32_t j, uint32_t m) {
    uint32_t d = 0;
    while (m > 1) {
        const uint32_t h = m >> 1;
        if (j == h - 1) return d;
        if (j < h - 1) {
            m = h;
        } else {
            j -= h;
            m -= h;
        }
        ++d;
    }
    return d;
}

// First index in [lo, hi) whose key is not below / is above a.
template <bool ABOVE>
GPR_D uint32_t key_bound(const uint32_t* k, uint32_t lo, uint32_t hi, uint32_t a) {
    while (lo < hi) {
        const uint32_t m = (lo + hi) >> 1;
        if (ABOVE ? k[m] <= a : k[m] < a) lo = m + 1;
        else hi = m;
    }
    return lo;
}

// Weight of the split between sorted leaves k and k + 1, 0 <= k < n - 1: the
// deeper split has the larger weight.  keys[0 .. m] are sk[s .. s + m] and
// s <= k < s + m: a run of equal keys is searched there first, and in all of sk
// only where it goes on past an end.
GPR_D int32_t split_weight(const uint32_t* __restrict__ sk, uint32_t n, const uint32_t* keys, uint32_t s, uint32_t m,
                           uint32_t k) {
    const uint32_t i = k - s, a = keys[i], b = keys[i + 1];
    if (a != b) return __clz(a ^ b);
    uint32_t first = s + key_bound<false>(keys, 0, i, a);
    if (first == s && s > 0) first = key_bound<false>(sk, 0, s, a);
    uint32_t end = s + key_bound<true>(keys, i + 1, m + 1, a);
    if (end == s + m + 1 && end < n) end = key_bound<true>(sk, end, n, a);
    return 32 + (int32_t)midpoint_depth(k - first, end - first);
}

// ------------------------------------------------------ tree + refit ----
// Node ids: internal node k (split between sorted leaves k and k+1) = k,
// leaf i = (n-1)+i.  A node covering [l, r] has parent r (as left child) if
// the split after r is deeper than the split before l, else parent l-1 (as
// right child).  The second child to arrive at a parent forms its box.
//
// Everything one thread publishes for another (boxes, child ids, range
// bounds) is written with device-scope relaxed atomic stores, which gfx950
// issues as write-through stores (sc1) to the device-coherent level; the
// writer waits for their completion (vmcnt(0)) before it bumps the arrival
// counter (a device-scope RMW, performed at the coherent level), and the
// reader loads with device-scope atomic loads (sc1, served from the coherent
// level) only after that RMW has returned.  So no L2 write-back (buffer_wbl2)
// or invalidate is needed although the eight XCD L2 caches are not coherent
// with each other; device-scope release / acquire on the RMW would add both
// on every arrival (measured 16x slower at 1M triangles).  Values read back
// are range-checked, and the layout kernels check every parent box against the
// union of its children's (k_layout inside a block, and that a block's own
// subtrees have the boxes that were published; k_layout_top above), so a protocol
// failure raises the error word instead of indexing out of bounds or producing a
// wrong tree silently.
GPR_D void pub(uint32_t* p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
GPR_D uint32_t get(uint32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
GPR_D void pub8(uint64_t* p, uint64_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
GPR_D uint64_t get8(uint64_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
GPR_D void pub2(uint64_t* p, float a, float b) {
    pub8(p, (uint64_t)__float_as_uint(a) | ((uint64_t)__float_as_uint(b) << 32));
}
GPR_D void get2(uint64_t* p, float& a, float& b) {
    const uint64_t v = get8(p);
    a = __uint_as_float((uint32_t)v);
    b = __uint_as_float((uint32_t)(v >> 32));
}

// Most of a tree lies inside short runs of leaves: a block builds the subtrees
// inside its kTreeB consecutive leaves in LDS, and only the nodes whose range
// crosses a run's edge (1-2 % of them) go through the published protocol above.
// The layout pass builds the same subtrees again from the triangle records
// rather than reading 60 bytes a node back.  Both passes are bound by memory:
// random reads of the positions in the first, 180 MB of layouts written in the
// second.  Tree, refit and layouts of a 1M-triangle soup take 168 us
// instead of the 559 of one published climb per leaf and a kernel per layout.
// Weights fit 16 bits; with 32 a block of k_layout took 41,008 bytes of LDS, three
// to a CU instead of four: 80.7 us without its checks, 82.6 with them, now 75.8.
constexpr uint16_t kNoNode = 0xffff;
// Node codes inside a block: internal node of split j is j, leaf i is kTreeB + i.
struct TreeShared {
    float box[6][2 * kTreeB];
    uint16_t par[2 * kTreeB];  // local parent; kNoNode at the roots of local subtrees
    uint16_t ch[2][kTreeB];
    uint16_t lo[kTreeB], hi[kTreeB];  // leaf range
    uint32_t cnt[kTreeB];             // arrivals: 2 = built here
    int16_t w[kTreeB + 1];            // w[j]: weight of the split before leaf j, -1 before the first and after the last
};
// Where a thread's climb ended: the local subtree it holds, and whether that
// subtree is a root of its block's forest.
struct Climb {
    uint32_t code, l, r;  // node and its leaf range (block-local)
    v3 lo, hi;
    bool root;       // nothing above it was built here
    bool whole;      // it is the whole tree
    bool as_left;    // side on its parent
    int32_t parent;  // its parent's split, block-local (-1 .. kTreeB - 1)
};

GPR_D void put_box(TreeShared& S, uint32_t code, v3 lo, v3 hi) {
    S.box[0][code] = lo.x; S.box[1][code] = lo.y; S.box[2][code] = lo.z;
    S.box[3][code] = hi.x; S.box[4][code] = hi.y; S.box[5][code] = hi.z;
}

// Builds the subtrees inside leaves [s, s + m); (lo, hi) is leaf threadIdx.x's
// box, S.w holds the weights (its writes need no barrier before the call).
GPR_D Climb local_tree(TreeShared& S, uint32_t n, uint32_t s, uint32_t m, v3 lo, v3 hi) {
    const uint32_t i = threadIdx.x;
    Climb c;
    c.code = kTreeB + i;
    c.l = c.r = i;
    c.lo = lo;
    c.hi = hi;
    c.root = c.whole = c.as_left = false;
    c.parent = -1;
    S.cnt[i] = 0;
    S.par[i] = S.par[kTreeB + i] = kNoNode;
    __syncthreads();
    if (i < m) {
        while (true) {
            put_box(S, c.code, c.lo, c.hi);
            if (s + c.l == 0 && s + c.r == n - 1) {
                c.root = c.whole = true;
                break;
            }
            c.as_left = S.w[c.r + 1] > S.w[c.l];
            c.parent = c.as_left ? (int32_t)c.r : (int32_t)c.l - 1;
            if (c.parent < 0 || c.parent + 1 >= (int32_t)m) {  // the split is another block's, or between two blocks
                c.root = true;
                break;
            }
            const uint32_t p = (uint32_t)c.parent;
            S.par[c.code] = (uint16_t)p;
            S.ch[c.as_left ? 0 : 1][p] = (uint16_t)c.code;
            if (c.as_left) S.lo[p] = (uint16_t)c.l;
            else S.hi[p] = (uint16_t)c.r;
            // everything above is in LDS before the arrival is counted
            __threadfence_block();
            if (atomicAdd(&S.cnt[p], 1u) == 0) break;
            __threadfence_block();
            const uint32_t sib = S.ch[c.as_left ? 1 : 0][p];
            const v3 slo = V(S.box[0][sib], S.box[1][sib], S.box[2][sib]);
            const v3 shi = V(S.box[3][sib], S.box[4][sib], S.box[5][sib]);
            // Union(l_child, r_child) (aabb.h:37-46, bvh.h:182)
            if (c.as_left) {
                c.r = S.hi[p];
                c.lo = vmin3(c.lo, slo);
                c.hi = vmax3(c.hi, shi);
            } else {
                c.l = S.lo[p];
                c.lo = vmin3(slo, c.lo);
                c.hi = vmax3(shi, c.hi);
            }
            c.code = p;
        }
    }
    __syncthreads();
    // the first to arrive at a node whose other child reaches out of the block
    if (i < m && !c.root && S.cnt[c.parent] == 1) {
        c.root = true;
        S.par[c.code] = kNoNode;
    }
    return c;
}
GPR_D uint32_t node_id(uint32_t code, uint32_t s, uint32_t n) {
    return code < kTreeB ? s + code : (n - 1) + s + (code - kTreeB);
}

__global__ __launch_bounds__(kTreeB) void k_tree(const float* __restrict__ pos, uint32_t n,
                                                 const uint32_t* __restrict__ sidx,
                                                 const uint32_t* __restrict__ sk, TriRec* __restrict__ tris,
                                                 int32_t* __restrict__ w, uint32_t* __restrict__ parent,
                                                 uint32_t* __restrict__ child, uint64_t* __restrict__ ends,
                                                 uint32_t* __restrict__ arrive,
                                                 float* __restrict__ box,  // (2n-1)*6
                                                 BuildState* __restrict__ bs) {
    __shared__ TreeShared S;
    __shared__ uint32_t keys[kTreeB + 2];  // of leaves s - 1 .. s + m, as far as they exist
    const uint32_t s = blockIdx.x * kTreeB, m = min((uint32_t)kTreeB, n - s);
    const uint32_t before = s > 0 ? 1u : 0u, after = s + m < n ? 1u : 0u, nkeys = before + m + after;
    v3 lo = V(0, 0, 0), hi = V(0, 0, 0);
    for (uint32_t k = threadIdx.x; k < nkeys; k += kTreeB) keys[k] = sk[s - before + k];
    if (threadIdx.x < m) {
        const uint32_t t = sidx[s + threadIdx.x];
        float q[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) q[k] = pos[9ull * t + k];
        TriRec rec;
        rec.a = make_float4(q[0], q[1], q[2], q[3]);
        rec.b = make_float4(q[4], q[5], q[6], q[7]);
        rec.c = make_float4(q[8], __uint_as_float(t), 0.f, 0.f);
        tris[s + threadIdx.x] = rec;
        tri_bounds(q, lo, hi);
    }
    __syncthreads();
    // splits s - 1 .. s + m - 1
    for (uint32_t j = threadIdx.x; j <= m; j += kTreeB) {
        const bool inside = (j > 0 || before) && (j < m || after);
        const int32_t v = inside ? split_weight(sk, n, keys, s - before, nkeys - 1, s + j - 1) : -1;
        S.w[j] = (int16_t)v;
        if (j > 0) w[s + j - 1] = v;
    }
    const Climb c = local_tree(S, n, s, m, lo, hi);
    if (!c.root) return;
    uint32_t node = node_id(c.code, s, n);
    lo = c.lo;
    hi = c.hi;
    // a node's box is 24 B at 6*node floats: three 8-byte words
    uint64_t* bx = reinterpret_cast<uint64_t*>(box);
    uint32_t l = s + c.l, r = s + c.r;
    // weights of the splits before and after the node; an end travels with its
    // weight (weight << 32 | leaf), so no step waits for keys
    int32_t wl = S.w[c.l], wr = S.w[c.r + 1];
    for (int guard = 0; guard < kMaxDepth; ++guard) {
        uint64_t* b = bx + 3ull * node;
        pub2(b + 0, lo.x, lo.y);
        pub2(b + 1, lo.z, hi.x);
        pub2(b + 2, hi.y, hi.z);
        if (l == 0 && r == n - 1) {
            bs->root = node;
            break;
        }
        const bool as_left = wr > wl;
        const uint32_t p = as_left ? r : l - 1;
        parent[node] = p << 1 | (as_left ? 1u : 0u);
        pub(&child[2 * p + (as_left ? 0 : 1)], node);
        pub8(&ends[2ull * p + (as_left ? 0 : 1)], (uint64_t)(uint32_t)(as_left ? wl : wr) << 32 | (as_left ? l : r));
        // every publish above has completed (s_waitcnt vmcnt(0)) before the
        // arrival RMW is issued; the fence keeps the compiler from moving the
        // publishing stores past the wait
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        if (__hip_atomic_fetch_add(&arrive[p], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) break;
        // second arrival: the sibling's publishes completed before its
        // increment; the loads below are issued after this RMW returned
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        const uint64_t e = get8(&ends[2ull * p + (as_left ? 1 : 0)]);
        if (as_left) {
            r = (uint32_t)e;
            wr = (int32_t)(e >> 32);
        } else {
            l = (uint32_t)e;
            wl = (int32_t)(e >> 32);
        }
        const uint32_t sib = get(&child[2 * p + (as_left ? 1 : 0)]);
        if (r >= n || l > p || (as_left && r <= p) || sib >= 2 * n - 1) {
            atomicOr(&bs->err, 1u);
            break;
        }
        uint64_t* sb = bx + 3ull * sib;
        v3 slo, shi;
        get2(sb + 0, slo.x, slo.y);
        get2(sb + 1, slo.z, shi.x);
        get2(sb + 2, shi.y, shi.z);
        // Union(l_child, r_child) (aabb.h:37-46, bvh.h:182)
        if (as_left) {
            lo = vmin3(lo, slo);
            hi = vmax3(hi, shi);
        } else {
            lo = vmin3(slo, lo);
            hi = vmax3(shi, hi);
        }
        node = p;
    }
}

// Exclusive rank of the threads with `mine` in a block of NT and their count.
template <int NT>
GPR_D uint32_t block_rank(bool mine, uint32_t* sh /* NT / 64 */, uint32_t* total) {
    const unsigned long long b = __ballot(mine);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) sh[wave] = (uint32_t)__popcll(b);
    __syncthreads();
    uint32_t before = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        before += w < wave ? sh[w] : 0u;
        tot += sh[w];
    }
    *total = tot;
    return before + __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
}

// The nodes k_tree published (arrive == 2): left steps and depth from the root,
// a BVH4 number for those at even depth (the top of the tree first), and a list
// of them.  They are few and far between, so a block gathers those of kTopSpan
// splits in LDS, walks them up with full waves and reserves their numbers and
// list entries with one atomic.
constexpr int kTopB = 1024, kTopSpan = 4096;
__global__ __launch_bounds__(kTopB) void k_top(uint32_t n, const uint32_t* __restrict__ arrive,
                                               const uint32_t* __restrict__ parent,  // split << 1 | as left child
                                               uint32_t* __restrict__ left, uint32_t* __restrict__ depth,
                                               uint32_t* __restrict__ id4, uint32_t* __restrict__ list,
                                               BuildState* __restrict__ bs) {
    __shared__ uint32_t node[kTopSpan];
    __shared__ uint16_t rank[kTopSpan];  // among the block's even-depth nodes; kNoNode at odd depth
    __shared__ uint32_t ntop, neven, base[2];
    if (threadIdx.x == 0) ntop = neven = 0;
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < kTopSpan; j += kTopB) {
        const uint32_t k = blockIdx.x * kTopSpan + j;
        if (k + 1 < n && arrive[k] == 2u) node[atomicAdd(&ntop, 1u)] = k;
    }
    __syncthreads();
    const uint32_t rt = bs->root;
    for (uint32_t e = threadIdx.x; e < ntop; e += kTopB) {
        const uint32_t k = node[e];
        uint32_t dep = 0, lf = 0, y = k;
        while (y != rt && dep < kMaxDepth) {
            const uint32_t p = parent[y];
            if (p >> 1 >= n - 1) break;  // only reachable through a malformed tree
            lf += p & 1u;
            ++dep;
            y = p >> 1;
        }
        if (y != rt) atomicOr(&bs->err, 4u);
        left[k] = lf;
        depth[k] = dep;
        if (dep == 0) id4[k] = 0;
        rank[e] = dep != 0 && (dep & 1u) == 0 ? (uint16_t)atomicAdd(&neven, 1u) : kNoNode;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long at = 0;  // nbvh4 and ntop side by side
        if (ntop) at = atomicAdd(reinterpret_cast<unsigned long long*>(bs), (unsigned long long)ntop << 32 | neven);
        base[0] = (uint32_t)at;
        base[1] = (uint32_t)(at >> 32);
    }
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < ntop; e += kTopB) {
        if (rank[e] != kNoNode) id4[node[e]] = base[0] + rank[e];
        list[base[1] + e] = node[e];
    }
}

GPR_D void put_ref(gpr_ref_node* __restrict__ ref, uint32_t nn, uint32_t at, const float b[6], uint32_t idx,
                   uint32_t leaf, BuildState* __restrict__ bs) {
    if (at >= nn) {
        atomicOr(&bs->err, 4u);
        return;
    }
    float4* o = reinterpret_cast<float4*>(ref + at);
    o[0] = make_float4(b[0], b[1], b[2], b[3]);
    o[1] = make_float4(b[4], b[5], __uint_as_float(idx), __uint_as_float(leaf));
}

// Bound `q` (lox loy loz hix hiy hiz) of the union of a left and a right child.
GPR_D float union_of(int q, float l, float r) { return q < 3 ? fmin_h(l, r) : fmax_h(l, r); }
GPR_D bool same_bits(float a, float b) { return __float_as_uint(a) == __float_as_uint(b); }

// Layouts of the nodes built inside blocks: reference nodes, BVH4 nodes, and
// for the published nodes above what they need of the subtrees below them.
__global__ __launch_bounds__(kTreeB) void k_layout(uint32_t n, const TriRec* __restrict__ tris,
                                                   const int32_t* __restrict__ w,
                                                   const uint32_t* __restrict__ left,
                                                   const uint32_t* __restrict__ depth,
                                                   uint32_t* __restrict__ child, float* __restrict__ box,
                                                   uint32_t* __restrict__ id4, gpr_ref_node* __restrict__ ref,
                                                   Bvh4Node* __restrict__ out, BuildState* __restrict__ bs) {
    __shared__ TreeShared S;
    __shared__ uint16_t s_left[2 * kTreeB];   // left steps and depth from the root
    __shared__ uint16_t s_depth[2 * kTreeB];
    __shared__ uint16_t s_rank[kTreeB];       // BVH4 number minus the block's first, even depth only
    __shared__ uint16_t s_even[kTreeB];       // splits of the block's BVH4 nodes
    __shared__ uint32_t sh[kTreeB / 64];
    __shared__ uint32_t s_base;
    __shared__ uint32_t s_whole;  // split of the root when the block holds the whole tree
    const uint32_t s = blockIdx.x * kTreeB, m = min((uint32_t)kTreeB, n - s), nn = 2 * n - 1;
    const uint32_t i = threadIdx.x;
    v3 lo = V(0, 0, 0), hi = V(0, 0, 0);
    uint32_t tri = 0;
    if (i < m) {
        const float4* t = reinterpret_cast<const float4*>(tris + s + i);
        const float4 a = t[0], b = t[1], c = t[2];
        const float q[9] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x};
        tri = __float_as_uint(c.y);
        tri_bounds(q, lo, hi);
    }
    for (uint32_t j = i; j <= m; j += kTreeB) S.w[j] = (int16_t)(s + j > 0 ? w[s + j - 1] : -1);
    const Climb c = local_tree(S, n, s, m, lo, hi);
    if (c.root) {
        uint32_t l = 0, d = 0;
        if (!c.whole) {
            const uint32_t p = (uint32_t)((int64_t)s + c.parent);
            l = left[p] + (c.as_left ? 1u : 0u);
            d = depth[p] + 1;
            // the box that k_tree published is this build's
            const float2* b = reinterpret_cast<const float2*>(box + 6ull * node_id(c.code, s, n));
            const float2 x = b[0], y = b[1], z = b[2];
            if (!(same_bits(x.x, c.lo.x) && same_bits(x.y, c.lo.y) && same_bits(y.x, c.lo.z) && same_bits(y.y, c.hi.x) &&
                  same_bits(z.x, c.hi.y) && same_bits(z.y, c.hi.z)))
                atomicOr(&bs->err, 2u);
        }
        s_left[c.code] = (uint16_t)l;
        s_depth[c.code] = (uint16_t)d;
        if (c.whole) s_whole = c.code;
    }
    if (i == 0 && n > kTreeB) s_whole = 0;  // no node moves in front of split 0
    __syncthreads();
    // from its root to each of the thread's two nodes
    const bool inner = i + 1 < m && S.cnt[i] == 2u;
    uint32_t lf[2] = {0, 0}, dp[2] = {0, 0};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        if (k == 0 ? !inner : i >= m) continue;
        uint32_t y = k == 0 ? i : kTreeB + i;
        for (uint32_t p = S.par[y]; p != kNoNode; p = S.par[y]) {
            lf[k] += S.ch[0][p] == y ? 1u : 0u;
            ++dp[k];
            y = p;
        }
        lf[k] += s_left[y];
        dp[k] += s_depth[y];
    }
    const bool even = inner && (dp[0] & 1u) == 0;
    uint32_t count;
    uint32_t rank = block_rank<kTreeB>(even, sh, &count);
    // a whole tree's root is number 0
    if (i == s_whole && n <= kTreeB) rank = 0;
    else if (i < s_whole) ++rank;
    if (i == 0) s_base = count ? atomicAdd(&bs->nbvh4, count) : 0u;
    if (even) {
        s_rank[i] = (uint16_t)rank;
        s_even[rank] = (uint16_t)i;
    }
    if (i < m) {
        const float b[6] = {lo.x, lo.y, lo.z, hi.x, hi.y, hi.z};
        put_ref(ref, nn, 2 * (s + i) + lf[1], b, tri, 1u, bs);
    }
    if (inner) {
        const float b[6] = {S.box[0][i], S.box[1][i], S.box[2][i], S.box[3][i], S.box[4][i], S.box[5][i]};
        // the right child starts at leaf split + 1 and is reached without a left step
        put_ref(ref, nn, 2 * (s + S.lo[i]) + lf[0], b, 2 * (s + i + 1) + lf[0], 0u, bs);
    }
    __syncthreads();
    const uint32_t base = s_base;
    const auto ref4 = [&](uint32_t code) -> int32_t {
        return code >= kTreeB ? ~(int32_t)(s + code - kTreeB) : (int32_t)(base + s_rank[code]);
    };
    if (base + count > n - 1 && count) {
        if (i == 0) atomicOr(&bs->err, 4u);
        return;
    }
    // BVH4 nodes, eight lanes each: lane j writes the j-th 16 bytes of the line
    for (uint32_t w = i; w < count * 8; w += kTreeB) {
        const uint32_t x = s_even[w >> 3], piece = w & 7;
        // slots: the children, an inner child replaced by its two
        const uint32_t c0 = S.ch[0][x], c1 = S.ch[1][x];
        const bool in0 = c0 < kTreeB, in1 = c1 < kTreeB;
        const uint32_t r0 = in1 ? S.ch[0][c1] : c1, r1 = in1 ? S.ch[1][c1] : 0u;
        const uint32_t slot[4] = {in0 ? S.ch[0][c0] : c0, in0 ? S.ch[1][c0] : r0, in0 ? r0 : r1, r1};
        const int k = 2 + (in0 ? 1 : 0) + (in1 ? 1 : 0);
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // planes: lox hix loy hiy loz hiz
            if (piece < 6) v[q] = q < k ? S.box[(piece >> 1) + (piece & 1) * 3][slot[q]] : INFINITY;
            else if (piece == 6) v[q] = __int_as_float(q < k ? ref4(slot[q]) : kEmptyChild);
            else v[q] = __uint_as_float(q == 0 ? s + x : 0u);
        }
        reinterpret_cast<float4*>(out + base + (w >> 3))[piece] = make_float4(v[0], v[1], v[2], v[3]);
    }
    // every parent's box against its children's
    if (inner) {
        const uint32_t c0 = S.ch[0][i], c1 = S.ch[1][i];
        bool same = c0 < 2 * kTreeB && c1 < 2 * kTreeB;
#pragma unroll
        for (int q = 0; q < 6; ++q) same = same && same_bits(union_of(q, S.box[q][c0], S.box[q][c1]), S.box[q][i]);
        if (!same) atomicOr(&bs->err, 2u);
    }
    if (c.root && c.code < kTreeB) {
        const uint32_t id = s + c.code;
        if ((s_depth[c.code] & 1u) == 0) {
            id4[id] = (uint32_t)ref4(c.code);
        } else {
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const uint32_t a = S.ch[side][c.code], aid = node_id(a, s, n);
                child[2 * id + side] = aid;
                for (int q = 0; q < 6; ++q) box[6ull * aid + q] = S.box[q][a];
                if (a < kTreeB) id4[aid] = (uint32_t)ref4(a);
            }
        }
    }
}

// Layouts of the published nodes, eight lanes each.  Their boxes are checked
// against their children's as they stand now (a stale box read in k_tree would
// break the equality).
__global__ __launch_bounds__(kB) void k_layout_top(uint32_t n, const uint32_t* __restrict__ list,
                                                   const uint32_t* __restrict__ child,
                                                   const uint64_t* __restrict__ ends,
                                                   const float* __restrict__ box,
                                                   const uint32_t* __restrict__ left,
                                                   const uint32_t* __restrict__ depth,
                                                   const uint32_t* __restrict__ id4,
                                                   gpr_ref_node* __restrict__ ref, Bvh4Node* __restrict__ out,
                                                   BuildState* __restrict__ bs) {
    const uint32_t nn = 2 * n - 1, ntop = min(bs->ntop, n - 1), piece = threadIdx.x & 7;
    for (uint32_t k = (blockIdx.x * kB + threadIdx.x) >> 3; k < ntop; k += gridDim.x * kB / 8) {
        const uint32_t x = list[k];
        const uint32_t c[2] = {child[2 * x], child[2 * x + 1]};
        const uint32_t lf = left[x], dep = depth[x];
        if (c[0] >= nn || c[1] >= nn) {
            atomicOr(&bs->err, 2u);
            continue;
        }
        if (piece < 6) {
            const float u = union_of(piece, box[6ull * c[0] + piece], box[6ull * c[1] + piece]);
            if (!same_bits(u, box[6ull * x + piece])) atomicOr(&bs->err, 2u);
        } else if (piece == 6) {
            put_ref(ref, nn, 2 * (uint32_t)ends[2ull * x] + lf, box + 6ull * x, 2 * (x + 1) + lf, 0u, bs);
        }
        if (dep & 1u) continue;
        const bool in0 = c[0] < n - 1, in1 = c[1] < n - 1;
        uint32_t g[4] = {0, 0, 0, 0};  // grandchildren
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (q < 2 ? in0 : in1) g[q] = child[2 * c[q >> 1] + (q & 1)];
        const uint32_t id = id4[x];
        if (g[0] >= nn || g[1] >= nn || g[2] >= nn || g[3] >= nn || id >= n - 1) {
            atomicOr(&bs->err, 2u);
            continue;
        }
        const uint32_t r0 = in1 ? g[2] : c[1], r1 = in1 ? g[3] : 0u;
        const uint32_t slot[4] = {in0 ? g[0] : c[0], in0 ? g[1] : r0, in0 ? r0 : r1, r1};
        const int cnt = 2 + (in0 ? 1 : 0) + (in1 ? 1 : 0);
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (piece < 6) v[q] = q < cnt ? box[6ull * slot[q] + (piece >> 1) + (piece & 1) * 3] : INFINITY;
            else if (piece == 6)
                v[q] = __int_as_float(q >= cnt ? kEmptyChild
                                      : slot[q] >= n - 1 ? ~(int32_t)(slot[q] - (n - 1)) : (int32_t)id4[slot[q]]);
            else v[q] = __uint_as_float(q == 0 ? x : 0u);
        }
        reinterpret_cast<float4*>(out + id)[piece] = make_float4(v[0], v[1], v[2], v[3]);
    }
}

struct Carve {
    char* base;
    size_t off;
    template <class T>
    T* take(size_t count) {
        off = (off + 255) & ~(size_t)255;
        T* p = reinterpret_cast<T*>(base + off);
        off += count * sizeof(T);
        return p;
    }
};

}  // namespace

int build_bvh(gpr_scene* s) {
    BvhDev& B = s->bvh;
    const uint32_t n = (uint32_t)s->mat.size();
    B.n = n;
    if (n == 0) {
        B.nbvh4 = 0;
        return GPR_OK;
    }
    hipStream_t st = stream();
    const uint32_t nn = 2 * n - 1;
    const uint32_t npart = std::min(1024u, div_up(n, kB));
    // ---- carve the arena
    size_t need = 0;
    for (int pass = 0; pass < 2; ++pass) {
        Carve c{pass ? B.arena.as<char>() : nullptr, 0};
        float* part = c.take<float>(6ull * npart);
        float* bounds = c.take<float>(8);
        uint32_t* keys = c.take<uint32_t>(n);
        uint32_t* skeys = c.take<uint32_t>(n);
        uint32_t* sidx = c.take<uint32_t>(n);
        uint32_t* parent = c.take<uint32_t>(nn);
        uint32_t* child = c.take<uint32_t>(2ull * n);
        uint64_t* ends = c.take<uint64_t>(2ull * n);
        int32_t* w = c.take<int32_t>(n);
        uint32_t* list = c.take<uint32_t>(n);
        uint32_t* arrive = c.take<uint32_t>(n);
        float* box = c.take<float>(6ull * nn);
        uint32_t* left = c.take<uint32_t>(n);
        uint32_t* depth = c.take<uint32_t>(n);
        uint32_t* id4 = c.take<uint32_t>(n);
        BuildState* state = c.take<BuildState>(1);  // 256-aligned, as its 64-bit atomic needs
        gpr_ref_node* ref = c.take<gpr_ref_node>(nn);
        Bvh4Node* bvh4 = c.take<Bvh4Node>(std::max(1u, n - 1));
        TriRec* tris = c.take<TriRec>(n);
        if (pass == 0) {
            need = c.off + 256;
            GPR_TRY(B.arena.alloc(need));
            const size_t sb = sort_scratch_bytes(n);
            if (B.sort_scratch.bytes < sb || !B.sort_scratch.p) {
                GPR_TRY(B.sort_scratch.alloc(sb));
                GPR_TRY(sort_prepare(B.sort_scratch.p, B.sort_scratch.bytes, st));
            }
            continue;
        }
        B.keys = keys;
        B.skeys = skeys;
        B.sidx = sidx;
        B.ref = ref;
        B.bvh4 = bvh4;
        B.tris = tris;
        const float* pos = s->d_pos.as<float>();
        for (hipEvent_t& e : B.ev)
            if (!e) GPR_HIP(hipEventCreate(&e));
        hipEvent_t* ev = B.ev;
        GPR_HIP(hipEventRecord(ev[0], st));
        hipLaunchKernelGGL(k_centroid_partial, dim3(npart), dim3(kB), 0, st, pos, n, part);
        hipLaunchKernelGGL(k_centroid_final, dim3(1), dim3(kB), 0, st, part, npart, bounds, n > kTreeB ? 1u : 0u, state);
        hipLaunchKernelGGL(k_morton, dim3(div_up(n, kB)), dim3(kB), 0, st, pos, n, bounds, keys, arrive);
        GPR_HIP(hipEventRecord(ev[1], st));
        GPR_TRY(sort_pairs(keys, skeys, sidx, n, B.sort_scratch.p, B.sort_scratch.bytes, st));
        GPR_HIP(hipEventRecord(ev[2], st));
        const dim3 tree(div_up(n, kTreeB));
        hipLaunchKernelGGL(k_tree, tree, dim3(kTreeB), 0, st, pos, n, sidx, skeys, tris, w, parent, child, ends,
                           arrive, box, state);
        GPR_HIP(hipEventRecord(ev[3], st));
        if (n > kTreeB)  // otherwise one block builds the whole tree
            hipLaunchKernelGGL(k_top, dim3(div_up(n, kTopSpan)), dim3(kTopB), 0, st, n, arrive, parent, left, depth, id4,
                               list, state);
        hipLaunchKernelGGL(k_layout, tree, dim3(kTreeB), 0, st, n, tris, w, left, depth, child, box, id4, ref,
                           bvh4, state);
        if (n > kTreeB)
            hipLaunchKernelGGL(k_layout_top, dim3(std::min(1024u, div_up(n, kB))), dim3(kB), 0, st, n, list, child,
                               ends, box, left, depth, id4, ref, bvh4, state);
        GPR_HIP(hipEventRecord(ev[4], st));
        GPR_HIP(hipGetLastError());
        BuildState bs{};
        GPR_HIP(hipMemcpyAsync(&bs, state, sizeof bs, hipMemcpyDeviceToHost, st));
        GPR_HIP(hipStreamSynchronize(st));
        const uint32_t nb4 = bs.nbvh4, tree_err = bs.err;
        if (tree_err)
            return fail(GPR_ERR_INVALID, std::string("LBVH build: ") +
                                             ((tree_err & 1u) ? "inconsistent node publication " : "") +
                                             ((tree_err & 2u) ? "parent box differs from the union of its children " : "") +
                                             ((tree_err & 4u) ? "node unreachable from the root" : ""));
        B.nbvh4 = nb4;
        if (n > 1 && (nb4 == 0 || nb4 > n - 1))
            return fail(GPR_ERR_INVALID, "LBVH build produced an invalid BVH4 node count");
        B.root4 = n == 1 ? ~(int32_t)0 : 0;
        float ms;
        for (int k = 0; k < 4; ++k) {
            GPR_HIP(hipEventElapsedTime(&ms, ev[k], ev[k + 1]));
            B.timing[k] = ms;
        }
        GPR_HIP(hipEventElapsedTime(&ms, ev[0], ev[4]));
        B.timing[4] = ms;
    }
    return GPR_OK;
}

}  // namespace gpr
