// traverse.h -- closest-hit and any-hit traversal device code for gfx950.
//
// Two traversals share one triangle test:
//   * ref_*  : the reference's visit order on its DFS layout (BVHLinearNode),
//              its slab test and its per-thread 64-entry stack
//              (src/renderer/pathtracer_kernel.h:154-308).  Used for exact
//              reference semantics and for the traversal statistics.
//   * fast_* : packed 128-B BVH4 nodes (one cache line per node), a robust slab
//              test on all four children, nearest-first descent, leaf triangles
//              tested as soon as their parent is visited (the persistent any-hit
//              kernel instead parks them for wave-wide leaf rounds, TravD), and a
//              short per-lane stack in LDS whose youngest entries go to a global
//              overflow area when it is full.  Closest-hit results equal the reference's up
//              to ties of t.
#pragma once

#include "dev_math.h"
#include "gpr_internal.h"

namespace gpr {

constexpr int kStackGlobal = 96;   // global overflow entries per lane

struct Ray3 {
    v3 o, d;
    float tmin, tmax;
};

// triangle_intersect (pathtracer_kernel.h:119-152): float dots widened to
// double, double 1/det; rejects det==0, u<0|u>1, v<0|u+v>1, t<tmin|t>tmax.
GPR_D bool tri_hit_wide(v3 p0, v3 p1, v3 p2, v3 o, v3 d, float tmin, float tmax, double& th,
                        float& uh, float& vh) {
    const v3 e1 = p1 - p0;
    const v3 e2 = p2 - p0;
    const v3 P = cross3(d, e2);
    const double det = (double)dot3(P, e1);
    if (det == 0) return false;
    const double inv_det = 1.0 / det;
    const v3 T = o - p0;
    const double u = (double)dot3(P, T) * inv_det;
    if (u < 0.0 || u > 1.0) return false;
    const v3 Q = cross3(T, e1);
    const double v = (double)dot3(Q, d) * inv_det;
    if (v < 0.0 || u + v > 1.0) return false;
    const double t = (double)dot3(Q, e2) * inv_det;
    if (t < (double)tmin || t > (double)tmax) return false;
    th = t;
    uh = (float)u;
    vh = (float)v;
    return true;
}
GPR_D bool tri_hit_ref(v3 p0, v3 p1, v3 p2, v3 o, v3 d, float tmin, float tmax, float& th,
                       float& uh, float& vh) {
    double t;
    if (!tri_hit_wide(p0, p1, p2, o, d, tmin, tmax, t, uh, vh)) return false;
    th = (float)t;
    return true;
}

// ------------------------------------------------- reference traversal ---
// aabb_intersect (pathtracer_kernel.h:154-173)
GPR_D bool ref_box(const gpr_ref_node& nd, v3 o, float tmin_r, float tmax_r, v3 inv, int nx, int ny,
                   int nz) {
    const float bx0 = nx ? nd.bmax[0] : nd.bmin[0], bx1 = nx ? nd.bmin[0] : nd.bmax[0];
    const float by0 = ny ? nd.bmax[1] : nd.bmin[1], by1 = ny ? nd.bmin[1] : nd.bmax[1];
    const float bz0 = nz ? nd.bmax[2] : nd.bmin[2], bz1 = nz ? nd.bmin[2] : nd.bmax[2];
    float t0 = (bx0 - o.x) * inv.x;
    float t1 = (bx1 - o.x) * inv.x;
    const float ty0 = (by0 - o.y) * inv.y;
    const float ty1 = (by1 - o.y) * inv.y;
    if (t0 > ty1 || ty0 > t1) return false;
    t0 = fmax_h(t0, ty0);
    t1 = fmin_h(t1, ty1);
    const float tz0 = (bz0 - o.z) * inv.z;
    const float tz1 = (bz1 - o.z) * inv.z;
    if (t0 > tz1 || tz0 > t1) return false;
    t0 = fmax_h(t0, tz0);
    t1 = fmin_h(t1, tz1);
    return (t0 < tmax_r) && (t1 > tmin_r);
}

// trace_kernel / trace_shadow_kernel bodies (pathtracer_kernel.h:175-308).
template <bool ANY>
GPR_D gpr_hit ref_trace(const SceneView& sv, Ray3 r, uint32_t* nvisit, uint32_t* ntest) {
    gpr_hit hit{INFINITY, -1, 0.f, 0.f};
    const v3 inv = V(1 / r.d.x, 1 / r.d.y, 1 / r.d.z);
    const int nx = inv.x < 0, ny = inv.y < 0, nz = inv.z < 0;
    int cur = 0, sp = 0;
    int stack[64];
    uint32_t visits = 0, tests = 0;
    while (true) {
        // every node is visited at most once; both checks only trip on a malformed layout
        if ((uint32_t)cur >= sv.nref || visits > sv.nref) break;
        const gpr_ref_node nd = ldg(sv.ref + cur);
        ++visits;
        if (ref_box(nd, r.o, r.tmin, r.tmax, inv, nx, ny, nz)) {
            if (nd.leaf & 0xffu) {
                if (nd.idx >= sv.ntri) break;
                const float* p = sv.pos + 9ull * nd.idx;
                float t, u, v;
                ++tests;
                const v3 p0 = V(ldg(p), ldg(p + 1), ldg(p + 2)), p1 = V(ldg(p + 3), ldg(p + 4), ldg(p + 5));
                const v3 p2 = V(ldg(p + 6), ldg(p + 7), ldg(p + 8));
                if (tri_hit_ref(p0, p1, p2, r.o, r.d, r.tmin, r.tmax, t, u, v)) {
                    r.tmax = t;
                    hit = gpr_hit{t, (int32_t)nd.idx, u, v};
                    if (ANY) break;
                }
                if (sp == 0) break;
                cur = stack[--sp];
            } else {
                if (sp >= 64) break;  // unreachable for 30-bit keys; never write past the stack
                stack[sp++] = cur + 1;
                cur = (int)nd.idx;
            }
        } else {
            if (sp == 0) break;
            cur = stack[--sp];
        }
    }
    *nvisit += visits;
    *ntest += tests;
    return hit;
}

// ------------------------------------------------------ BVH4 traversal ---
// Per-lane traversal stack: the oldest SL entries in an LDS column of the wave's
// own part of the block's LDS (entry k at lds[k * 64]), the rest in a per-lane
// global slab of kStackGlobal entries (walks rarely reach it).  Entry 0 is a sentinel that
// every pop accepts and that ends the walk, so popping needs no empty test.
// Closest hit keeps 8 bytes per entry (the order key and the child), any hit
// only the child.
template <class E, int SL>
struct LaneStackT {
    using Entry = E;
    static constexpr int kStride = 64;
    E* lds;    // this lane's column
    E* spill;  // this lane's overflow area (kStackGlobal entries)
    int sp;
    // block_lds: SL entries a lane; overflow: kStackGlobal int2 a lane of the grid
    template <int NT>
    GPR_D void place(void* block_lds, int2* overflow) {
        lds = static_cast<E*>(block_lds) + (threadIdx.x / 64) * (SL * 64) + (threadIdx.x & 63);
        spill = reinterpret_cast<E*>(overflow + (uint64_t)(blockIdx.x * NT + threadIdx.x) * kStackGlobal);
    }
    GPR_D void reset(E sentinel) {
        lds[0] = sentinel;
        sp = 1;
    }
    GPR_D void put(int at, E e) {
        if (at < SL) lds[at * kStride] = e;
        else spill[at - SL] = e;
    }
    GPR_D E pop() {
        --sp;
        if (sp >= SL) return spill[sp - SL];
        return lds[sp * kStride];
    }
    // true when no active lane of the wave could leave the LDS part by pushing k entries
    GPR_D bool roomy(int k) const { return __ballot(sp + k > SL) == 0ull; }
    GPR_D bool full(int k) const { return sp + k > SL + kStackGlobal; }
};
// Stack entry of a walk: closest hit (order key, child << 2 | low bits of the
// entry distance), any hit (child).
template <bool ANY>
struct StackEntry {
    using type = uint2;
};
template <>
struct StackEntry<true> {
    using type = int32_t;
};
template <bool ANY, int SL>
using LaneStack = LaneStackT<typename StackEntry<ANY>::type, SL>;

GPR_D void tri_rec_hit(const TriRec* tris, uint32_t ntri, int32_t leaf, const Ray3& r, float& tmax,
                       gpr_hit& hit, bool& found) {
    if ((uint32_t)leaf >= ntri) return;
    const TriRec* t = tris + leaf;
    const float4 a = ldg(&t->a), b = ldg(&t->b), c = ldg(&t->c);
    float th, uh, vh;
    if (tri_hit_ref(V(a.x, a.y, a.z), V(a.w, b.x, b.y), V(b.z, b.w, c.x), r.o, r.d, r.tmin, tmax, th,
                    uh, vh)) {
        tmax = th;
        hit = gpr_hit{th, (int32_t)__float_as_uint(c.y), uh, vh};
        found = true;
    }
}

// BVH4 traversal as an explicit state machine: trav_begin sets a ray up,
// each trav_step visits one node (its leaf children are tested first, they
// tighten tmax before the descent decision), so a caller can either run a ray
// to completion (fast_trace) or interleave the steps of many rays and give a
// lane a new ray as soon as its ray is done.  The walk goes on while
// trav_live(); node is then kTravDone, or anything else outside the tree when
// the stack ran out (or the tree is malformed).
struct Trav {
    Ray3 r;
    v3 inv;
    uint32_t ox, oy, oz;  // byte offset of each axis' near planes in a node (far planes: offset ^ 16)
    float tmax;
    gpr_hit hit;
    int32_t node;
    uint32_t fetched;
    uint32_t tested;  // triangle tests (read only by the statistics kernel; dead code elsewhere)
    bool found;
};
constexpr float kSlabCons = 1.0f + 2.0f * 1.7881394e-07f;  // 1 + 2*gamma(3)
enum : int32_t { kTravDone = 0x3fffffff, kTravOverflow = -1 };  // no node: a tree holds fewer than 2^30 - 1 nodes (137 GB)
constexpr uint32_t kKeyNone = 0x7fefffffu;  // order key of a child not taken: above every key, and no NaN as a double's high word

template <bool ANY, class Stack>
GPR_D void trav_begin(const SceneView& sv, const Ray3& r, Stack& st, Trav& t) {
    t.r = r;
    t.hit = gpr_hit{INFINITY, -1, 0.f, 0.f};
    t.tmax = r.tmax;
    t.found = false;
    t.fetched = 0;
    t.tested = 0;
    // the sentinel's entry distance is -inf: no limit culls it
    if constexpr (ANY) st.reset(kTravDone);
    else st.reset(make_uint2((uint32_t)kTravDone << 2, 0xff800000u));
    t.inv = V(1 / r.d.x, 1 / r.d.y, 1 / r.d.z);
    t.ox = __builtin_signbit(t.inv.x) ? 16u : 0u;
    t.oy = __builtin_signbit(t.inv.y) ? 48u : 32u;
    t.oz = __builtin_signbit(t.inv.z) ? 80u : 64u;
    t.node = sv.root4;
    if (sv.root4 < 0) {  // single-triangle scene: finished at once
        tri_rec_hit(sv.tris, sv.ntri, ~sv.root4, r, t.tmax, t.hit, t.found);
        t.node = kTravDone;
    }
}

// Whether the walk goes on.  A depth-first walk fetches every node at most
// once: the second bound only trips on a malformed tree.
GPR_D bool trav_live(const SceneView& sv, const Trav& t) {
    return (uint32_t)t.node < sv.nbvh4 && t.fetched <= sv.nbvh4;
}

// 64-bit minimum / maximum of two (order key, payload) pairs as doubles: keys
// are float bit patterns below 0x7ff00000, so the pairs are non-negative
// doubles that order by key; one instruction each instead of a compare and
// two selects, and the payload travels with its key.
GPR_D void key_sort2(double& a, double& b) {
    double lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
}
GPR_D double key_pair(uint32_t key, uint32_t payload) { return __hiloint2double((int)key, (int)payload); }
GPR_D uint32_t key_of(double e) { return (uint32_t)__double2hiint(e); }

// One node's box tests: leaf children in leaf_mask (slot order), inner
// children that the ray meets in hitc, entry distances in tn.
struct NodeHits {
    float tn[4];
    int32_t ch[4];
    bool hitc[4];
    uint32_t leaf_mask;
};
GPR_D void trav_boxes(const SceneView& sv, const Trav& t, NodeHits& h) {
    // the ray enters each slab at the plane its direction meets first: near
    // and far planes are loaded by the direction's signs, so no per-axis min
    // / max.  A 0 * inf (ray in a slab plane) gives NaN, which fmaxf / fminf
    // ignore: that axis then does not cull the child.
    const char* np = reinterpret_cast<const char*>(sv.bvh4) + ((uint64_t)(uint32_t)t.node << 7);
    const auto plane = [&](uint32_t off) { return ldg(reinterpret_cast<const float4*>(np + off)); };
    const float4 nx = plane(t.ox), fx = plane(t.ox ^ 16u), ny = plane(t.oy), fy = plane(t.oy ^ 16u);
    const float4 nz = plane(t.oz), fz = plane(t.oz ^ 16u);
    const int4 ch = ldg(reinterpret_cast<const int4*>(np + 96));
    const float nxa[4] = {nx.x, nx.y, nx.z, nx.w}, fxa[4] = {fx.x, fx.y, fx.z, fx.w};
    const float nya[4] = {ny.x, ny.y, ny.z, ny.w}, fya[4] = {fy.x, fy.y, fy.z, fy.w};
    const float nza[4] = {nz.x, nz.y, nz.z, nz.w}, fza[4] = {fz.x, fz.y, fz.z, fz.w};
    h.ch[0] = ch.x;
    h.ch[1] = ch.y;
    h.ch[2] = ch.z;
    h.ch[3] = ch.w;
    h.leaf_mask = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float x0 = (nxa[c] - t.r.o.x) * t.inv.x, x1 = (fxa[c] - t.r.o.x) * t.inv.x;
        const float y0 = (nya[c] - t.r.o.y) * t.inv.y, y1 = (fya[c] - t.r.o.y) * t.inv.y;
        const float z0 = (nza[c] - t.r.o.z) * t.inv.z, z1 = (fza[c] - t.r.o.z) * t.inv.z;
        const float tnear = fmaxf(fmaxf(x0, y0), fmaxf(z0, t.r.tmin));
        const float tfar = fminf(fminf(x1, y1), fminf(z1, t.tmax));
        h.tn[c] = tnear;
        const bool in = tnear <= tfar * kSlabCons;
        h.hitc[c] = in && h.ch[c] >= 0;
        h.leaf_mask |= (in && (uint32_t)h.ch[c] > (uint32_t)kEmptyChild) ? 1u << c : 0u;
    }
}
// child reference of the lowest slot set in m (m != 0)
GPR_D int32_t lowest_child(const NodeHits& h, uint32_t m) {
    const int c = __builtin_ctz(m);
    const int32_t lo = (c & 1) ? h.ch[1] : h.ch[0], hi = (c & 1) ? h.ch[3] : h.ch[2];
    return (c & 2) ? hi : lo;
}

// Descends after a closest-hit node's leaves: the nearest inner child next,
// the others pushed far to near, or the nearest pending node that can still
// hold a closer hit.  Children order by their entry distance with the slot in
// its two low bits; those bits travel with the child, so a pop compares the
// distance as computed.  The walk is bound by instruction issue as much as by
// the cache (a wave runs ~490 vector instructions per node it steps), so the
// pushes carry no loop and no branch: against a push loop over a sorted key
// list with child selects, 4M incoherent rays at 1M triangles take 3.47 ms
// instead of 3.97 wave-synchronous and 2.78 instead of 2.82 refilled, 700K
// any-hit rays at 262K triangles 0.69 ms instead of 0.79.
template <class Stack>
GPR_D void trav_descend(Stack& st, Trav& t, const NodeHits& h) {
    const float lim = t.tmax * kSlabCons;
    double e[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const bool go = h.hitc[c] && h.tn[c] <= lim;
        const uint32_t tb = __float_as_uint(h.tn[c]);
        const uint32_t key = go ? ((__float_as_uint(fmaxf(h.tn[c], 0.f)) & ~3u) | (uint32_t)c) : kKeyNone;
        e[c] = key_pair(key, ((uint32_t)h.ch[c] << 2) | (tb & 3u));
    }
    key_sort2(e[0], e[1]);
    key_sort2(e[2], e[3]);
    key_sort2(e[0], e[2]);
    key_sort2(e[1], e[3]);
    key_sort2(e[1], e[2]);
    ++t.fetched;
    using E = typename Stack::Entry;
    const auto entry = [](double v) { return make_uint2((uint32_t)__double2loint(v), (uint32_t)__double2hiint(v)); };
    if (st.roomy(3)) {
        // written without a branch: a slot whose child is not taken is
        // overwritten by the next entry (or left above the top)
#pragma unroll
        for (int k = 3; k >= 1; --k) {
            st.lds[st.sp * Stack::kStride] = entry(e[k]);
            st.sp += key_of(e[k]) != kKeyNone ? 1 : 0;
        }
    } else {
        if (st.full(3)) {
            t.node = kTravOverflow;
            return;
        }
#pragma unroll
        for (int k = 3; k >= 1; --k)
            if (key_of(e[k]) != kKeyNone) st.put(st.sp++, entry(e[k]));
    }
    uint32_t next = (uint32_t)__double2loint(e[0]);
    if (key_of(e[0]) == kKeyNone) {
        // distances below 0 (rays with tmin < 0) order and compare as 0
        const float plim = fmaxf(lim, __uint_as_float(4u));
        E p;
        do {
            p = st.pop();
        } while (__uint_as_float((p.y & ~3u) | (p.x & 3u)) > plim);
        next = p.x;
    }
    t.node = (int32_t)(next >> 2);
}

// Any hit needs no near-to-far order (any occluder ends the walk): the lowest
// hit slot is visited first and the others pushed, with no sorting network.
template <class Stack>
GPR_D void trav_descend_any(Stack& st, Trav& t, const NodeHits& h) {
    ++t.fetched;
    int32_t next = -1;
    if (st.roomy(3)) {
#pragma unroll
        for (int c = 3; c >= 0; --c) {
            if (c < 3) st.lds[st.sp * Stack::kStride] = next;
            st.sp += (c < 3 && h.hitc[c] && next >= 0) ? 1 : 0;
            next = h.hitc[c] ? h.ch[c] : next;
        }
    } else {
        if (st.full(3)) {
            t.node = kTravOverflow;
            return;
        }
#pragma unroll
        for (int c = 3; c >= 0; --c) {
            if (c < 3 && h.hitc[c] && next >= 0) st.put(st.sp++, next);
            next = h.hitc[c] ? h.ch[c] : next;
        }
    }
    t.node = next >= 0 ? next : st.pop();
}

// One node of a live walk.
template <bool ANY, class Stack>
GPR_D void trav_step(const SceneView& sv, Stack& st, Trav& t) {
    NodeHits h;
    trav_boxes(sv, t, h);
    // leaf children in ascending slot order, as a loop over this lane's own
    // leaves: a wave runs the triangle test as often as its busiest lane
    // needs it, not once per slot that any lane has a leaf in
    uint32_t leaves = h.leaf_mask;
    while (leaves != 0) {
        const int32_t leaf = lowest_child(h, leaves);
        leaves &= leaves - 1;
        tri_rec_hit(sv.tris, sv.ntri, ~leaf, t.r, t.tmax, t.hit, t.found);
        ++t.tested;
        if (ANY && t.found) leaves = 0;
    }
    if constexpr (ANY) {
        if (t.found) t.node = kTravDone;
        else trav_descend_any(st, t, h);
    } else {
        trav_descend(st, t, h);
    }
}

// Postponed-leaf form of the any-hit walk, used by the persistent kernel.  A
// node step does not test its leaf children: it parks them (slot mask +
// references) and the lane pauses; the wave tests the parked leaves of its
// lanes together in one leaf round, so the (double precision) triangle test
// runs with many lanes active instead of the few whose node held leaves.  A
// lane descends before its leaves are tested, and visits the next node only
// after them: the walk and its occluder are those of trav_step.
struct TravD : Trav {
    uint32_t pmask;  // parked leaf slots of the last visited node
    NodeHits h;      // that node's children
};
template <class Stack>
GPR_D void travd_step(const SceneView& sv, Stack& st, TravD& t) {
    trav_boxes(sv, t, t.h);
    t.pmask = t.h.leaf_mask;
    trav_descend_any(st, t, t.h);
}
// Tests the parked leaves in slot order.
GPR_D void travd_leaves(const SceneView& sv, TravD& t) {
    while (t.pmask != 0) {
        const int32_t leaf = lowest_child(t.h, t.pmask);
        t.pmask &= t.pmask - 1;
        tri_rec_hit(sv.tris, sv.ntri, ~leaf, t.r, t.tmax, t.hit, t.found);
        if (t.found) t.pmask = 0;
    }
}

// Closest hit (ANY=false) or any hit (ANY=true) against the BVH4.  Returns
// false only if the stack capacity was exceeded (the ray is then reported
// with the hits found so far and the caller raises an error flag).
template <bool ANY, class Stack>
GPR_D bool fast_trace(const SceneView& sv, const Ray3& r, Stack& st, gpr_hit& hit) {
    Trav t;
    trav_begin<ANY>(sv, r, st, t);
    while (trav_live(sv, t)) trav_step<ANY>(sv, st, t);
    hit = t.hit;
    return t.node == kTravDone;
}

// ------------------------------------------- four lanes to a ray (BVH4) ---
// A short batch leaves most lanes of the chip idle, and its time is that of one
// long walk: a chain of node loads and of the ~190 instructions a lane runs
// between two of them.  Here four lanes walk one ray: each tests one child's
// box, or its triangle if the child is a leaf, the children order by comparing
// keys across the four lanes, and each pushed child is stored by its own lane,
// about half the instructions.  Boxes, keys, stack entries and the order of the
// triangle tests are those of trav_step, so hits are bit-identical.
template <int CTRL>
GPR_D uint32_t quad_dpp(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, CTRL, 0xf, 0xf, true);
}
enum : int { kQuadRot1 = 0x39, kQuadRot2 = 0x4e, kQuadRot3 = 0x93 };  // lane i reads lane i + 1, 2, 3 of its four
template <int FROM>
GPR_D double quad_from(double x) {
    constexpr int ctrl = FROM * 0x55;
    return __hiloint2double((int)quad_dpp<ctrl>((uint32_t)__double2hiint(x)),
                            (int)quad_dpp<ctrl>((uint32_t)__double2loint(x)));
}
GPR_D uint32_t quad_or(uint32_t x) {
    x |= quad_dpp<kQuadRot2>(x);
    return x | quad_dpp<kQuadRot1>(x);
}
// the four lanes' bits, slot 0 lowest
GPR_D uint32_t quad_mask(bool b) { return quad_or(b ? 1u << (threadIdx.x & 3) : 0u); }

// A ray's stack, shared by its four lanes: SL entries in LDS, the rest in the overflow area.
template <class E, int SL>
struct QuadStack {
    static constexpr int kStride = 16;
    E* lds;
    E* spill;
    int sp;
    template <int NT>
    GPR_D void place(void* block_lds, int2* overflow) {
        const uint32_t wave = threadIdx.x / 64, quad = (threadIdx.x & 63) / 4;
        lds = static_cast<E*>(block_lds) + wave * (SL * 16) + quad;
        spill = reinterpret_cast<E*>(overflow + ((uint64_t)(blockIdx.x * (NT / 64) + wave) * 16 + quad) * kStackGlobal);
    }
    GPR_D void put(int at, E e) {
        if (at < SL) lds[at * kStride] = e;
        else spill[at - SL] = e;
    }
    GPR_D E get(int at) const { return at < SL ? lds[at * kStride] : spill[at - SL]; }
    GPR_D bool full(int k) const { return sp + k > SL + kStackGlobal; }
    // entries that one lane wrote are read by the others
    GPR_D void publish() const {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
};

// The walk of fast_trace<ANY>.  All four lanes hold the ray, tmax, node and
// stack height; lane c of the four holds child c, and `hit` belongs to the lane
// that `own` names (the first one for a miss).  Returns false where fast_trace does.
template <bool ANY, class Stack>
GPR_D bool quad_trace(const SceneView& sv, const Ray3& r, Stack& st, gpr_hit& hit, uint32_t& own) {
    using E = typename StackEntry<ANY>::type;
    const uint32_t c = threadIdx.x & 3;
    float tmax = r.tmax;
    hit = gpr_hit{INFINITY, -1, 0.f, 0.f};
    own = 0;
    if (sv.root4 < 0) {  // single-triangle scene
        bool found = false;
        tri_rec_hit(sv.tris, sv.ntri, ~sv.root4, r, tmax, hit, found);
        return true;
    }
    if constexpr (ANY) st.put(0, kTravDone);
    else st.put(0, make_uint2((uint32_t)kTravDone << 2, 0xff800000u));
    st.sp = 1;
    const v3 inv = V(1 / r.d.x, 1 / r.d.y, 1 / r.d.z);
    const uint32_t nxo = (__builtin_signbit(inv.x) ? 16u : 0u) + 4 * c, fxo = nxo ^ 16u;
    const uint32_t nyo = (__builtin_signbit(inv.y) ? 48u : 32u) + 4 * c, fyo = nyo ^ 16u;
    const uint32_t nzo = (__builtin_signbit(inv.z) ? 80u : 64u) + 4 * c, fzo = nzo ^ 16u;
    int32_t node = sv.root4;
    uint32_t fetched = 0;
    while ((uint32_t)node < sv.nbvh4 && fetched <= sv.nbvh4) {
        const char* np = reinterpret_cast<const char*>(sv.bvh4) + ((uint64_t)(uint32_t)node << 7);
        const auto plane = [&](uint32_t off) { return ldg(reinterpret_cast<const float*>(np + off)); };
        const float nx = plane(nxo), fx = plane(fxo), ny = plane(nyo), fy = plane(fyo), nz = plane(nzo), fz = plane(fzo);
        const int32_t ch = ldg(reinterpret_cast<const int32_t*>(np + 96 + 4 * c));
        const float x0 = (nx - r.o.x) * inv.x, x1 = (fx - r.o.x) * inv.x;
        const float y0 = (ny - r.o.y) * inv.y, y1 = (fy - r.o.y) * inv.y;
        const float z0 = (nz - r.o.z) * inv.z, z1 = (fz - r.o.z) * inv.z;
        const float tn = fmaxf(fmaxf(x0, y0), fmaxf(z0, r.tmin));
        const float tf = fminf(fminf(x1, y1), fminf(z1, tmax));
        const bool in = tn <= tf * kSlabCons;
        ++fetched;
        // leaf children, all at once
        bool ok = false;
        double td = 0.0;
        gpr_hit h{};
        if (in && (uint32_t)ch > (uint32_t)kEmptyChild && (uint32_t)~ch < sv.ntri) {
            const TriRec* t = sv.tris + (uint32_t)~ch;
            const float4 a = ldg(&t->a), b = ldg(&t->b), e = ldg(&t->c);
            ok = tri_hit_wide(V(a.x, a.y, a.z), V(a.w, b.x, b.y), V(b.z, b.w, e.x), r.o, r.d, r.tmin, tmax, td, h.u, h.v);
            h.t = (float)td;
            h.id = (int32_t)__float_as_uint(e.y);
        }
        if (__ballot(ok) != 0ull) {
            const uint32_t m = quad_mask(ok);
            if constexpr (ANY) {
                if (m) {  // the first in slot order ends the walk
                    own = __builtin_ctz(m);
                    if (c == own) hit = h;
                    return true;
                }
            } else {
                // in slot order, each against what the ones before it left of the ray
                uint32_t best = 4;
                const auto take = [&](uint32_t s, double t) {
                    const bool nearer = (m >> s & 1u) && !(t > (double)tmax);
                    tmax = nearer ? (float)t : tmax;
                    best = nearer ? s : best;
                };
                take(0, quad_from<0>(td));
                take(1, quad_from<1>(td));
                take(2, quad_from<2>(td));
                take(3, quad_from<3>(td));
                if (best != 4) own = best;
                if (c == best) hit = h;
            }
        }
        // inner children: the first one next, the others pushed
        bool go = in && ch >= 0;
        uint32_t key, payload;
        E e;
        if constexpr (ANY) {
            key = go ? c : kKeyNone;
            payload = (uint32_t)ch;
            e = ch;
        } else {
            go = go && tn <= tmax * kSlabCons;
            key = go ? ((__float_as_uint(fmaxf(tn, 0.f)) & ~3u) | c) : kKeyNone;
            payload = ((uint32_t)ch << 2) | (__float_as_uint(tn) & 3u);
            e = make_uint2(payload, key);
        }
        const uint32_t before = (quad_dpp<kQuadRot1>(key) < key ? 1u : 0u) + (quad_dpp<kQuadRot2>(key) < key ? 1u : 0u) +
                                (quad_dpp<kQuadRot3>(key) < key ? 1u : 0u);
        const int n = __popc(quad_mask(go));
        if (n == 0) {
            if constexpr (ANY) {
                node = st.get(--st.sp);
            } else {
                const float plim = fmaxf(tmax * kSlabCons, __uint_as_float(4u));
                E p;
                do {
                    p = st.get(--st.sp);
                } while (__uint_as_float((p.y & ~3u) | (p.x & 3u)) > plim);
                node = (int32_t)(p.x >> 2);
            }
        } else {
            if (st.full(3)) return false;
            if (go && before > 0) st.put(st.sp + n - 1 - (int)before, e);
            st.sp += n - 1;
            const uint32_t next = quad_or(go && before == 0 ? payload : 0u);
            node = ANY ? (int32_t)next : (int32_t)(next >> 2);
        }
        st.publish();
    }
    return node == kTravDone;
}

// Rays a wave takes a turn: `chunk` (a power of two, at least 64) of them, or
// fewer than a wave has lanes when kSpreadWaves waves of 32 lanes (or the whole
// grid, if smaller) hold all n.  Log2.
constexpr uint32_t kSpreadWaves = 4096;
template <class I>
GPR_D uint32_t turn_log(I n, uint32_t waves, uint32_t chunk_log) {
    const uint32_t spread = waves < kSpreadWaves ? waves : kSpreadWaves;
    if (n > (I)32 * spread) return chunk_log;
    uint32_t w = 0;
    while (((I)spread << w) < n) ++w;
    return w;
}

// Hands turns 0 .. n-1 to the waves of the grid and calls f(turn) for each.
//  - Every wave is dealt its first turn and claims the others as it comes free.
//    Claims are atomics that serialise at ~12 ns on one address, 131 us for the
//    11,000 claims of a million rays; so there are kClaimSets counters, each
//    for every kClaimSets-th turn and wave.  Neighbouring turns lie in
//    different sets, so the sets run out together, and a wave ends with its own:
//    looking through the others cost more than it evened out.
//  - A short queue is spread thin over kSpreadWaves waves (four to a SIMD): a
//    wave takes the union of its lanes' node steps and leaf tests, so thin
//    waves finish sooner and the chip has room for them (turn_log): one sample
//    of an 803x451 textured scene 1.85 ms unspread, 1.60 / 1.51 / 1.48 over 1024
//    / 2048 / 4096 waves.
// One counter with half of the turns dealt out beforehand, then 4 / 8 / 16 sets:
// 16 samples of the 256x256 Cornell box 1319, then 734 / 685 / 688 us; 8 of the
// 803x451 textured scene 2842, then 2525 / 2521 / 2523; 8 of a 500x300 sphere grid
// 2256, then 2146 / 2125 / 2132; the batch of 12 scenes 40.5 ms, then 39.1 / 39.4
// / 39.3.  8 sets with a search through the others' turns at the end: 1038,
// 2875, 2327 us and 41.0 ms.
constexpr uint32_t kClaimSets = 8;
constexpr uint32_t kClaimLine = 128;  // bytes between two counters
template <class C>
GPR_HD constexpr uint32_t claim_stride() { return kClaimLine / sizeof(C); }
// sets that `waves` waves claim from: every one needs a wave
GPR_D uint32_t claim_sets(uint32_t waves) { return waves >= kClaimSets ? kClaimSets : 1u; }
template <int NT, class I, class C, class F>
GPR_D void for_each_turn(C* cursor, I n, F&& f) {
    const uint32_t waves = gridDim.x * (NT / 64);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (NT / 64) + threadIdx.x / 64);
    const uint32_t sets = claim_sets(waves), set = wave % sets;
    C* mine = cursor + set * claim_stride<C>();
    for (I t = wave; t < n;) {
        f(t);
        if (n <= waves) break;
        C got = 0;
        if ((threadIdx.x & 63) == 0) got = atomicAdd(mine, (C)1);
        if constexpr (sizeof(I) == 4) t = waves + __builtin_amdgcn_readfirstlane(got) * sets + set;
        else t = waves + (I)__shfl(got, 0, 64) * sets + set;
    }
}

}  // namespace gpr
