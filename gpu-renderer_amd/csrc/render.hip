// render.hip -- wavefront path tracer on gfx950 (PathTracer::render,
// src/renderer/pathtracer.cu:41-150, kernels of src/renderer/pathtracer_kernel.h).
//
// A pass of 1 to 64 samples of every pixel is a fixed launch sequence with no host
// round trip:  gen -> extend(primary) -> max_depth x { shade -> trace } -> flush
// -> accum (several samples) -> finish, as two such chains side by side where it is
// large.  Queue sizes live on the device; each kernel reads the size it
// consumes and early-exits, so the whole pass can be replayed as a hipGraph.
//
//   gen     primary rays (InitRandom/NextRandom jitter or PCG32), queue A
//   extend  closest hit of the primary queue
//   shade   shade_hit_with_MIS: emission, NEE shadow append, BSDF scatter
//           append.  Appends are compacted: a wave ballot and mbcnt give lane
//           offsets, LDS gives wave offsets, and one atomic on the counter of
//           the block's queue segment gives the block's place.  In reference
//           RNG mode, where slot order must equal the serial order of the
//           reference's host loop, a decoupled look-back over tiles (one 64-bit
//           status word per tile) gives it instead.
//   trace   any hit of the shadow queue + accumulate_light_sampling_contribution;
//           closest hit of the scatter queue, its BSDF-sampling MIS term
//           (accumulate_BSDF_sampling_contribution), left in the entry, and, in
//           reference RNG mode, its roulette (pathtracer_kernel.h:684-749)
//   flush   the MIS terms of the last bounce; those of the others are added by
//           the next shade
//
// Per pixel the frame buffer receives emission, NEE and BSDF terms in the
// same order as the reference kernels (in every kernel one thread adds to a
// path, so the read-modify-write needs no atomics).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "dev_bsdf.h"
#include "dev_texture.h"
#include "engine.h"
#include "traverse.h"

namespace gpr {
namespace {

constexpr int kShadeBlock = 256;
constexpr uint32_t kMaxBounce = 64;
constexpr uint32_t kMaxSegs = 4;  // a power of two
constexpr uint32_t kLastSpread = 16;

// Queue of path vertices / rays (SoA, capacity = paths per sample or pass).
struct QueueView {
    float4* o_tmin;   // origin, tmin
    float4* d_tmax;   // direction, tmax
    float4* hit;      // t, id bits, u, v
    float4* w_pdf;    // throughput rgb, BSDF pdf
    uint32_t* pix;    // frame-buffer pixel, or path id of a multi-sample pass | specular << 31
    unsigned long long* rng;  // PCG32 state (pcg mode)
    uint32_t* seed = nullptr;  // slot-indexed LCG seed (reference mode, persists across samples)
    uint32_t* job;    // multi-job passes: the entry's scene << kJobBits | pass job
};

constexpr uint32_t kClaimWords = kClaimSets * claim_stride<uint32_t>();

// Per-sample control block (counters cleared by k_gen).
struct alignas(kClaimLine) Ctrl {
    uint32_t sample;         // current sample index (single-scene; advanced by k_finish)
    uint32_t error;          // bit0: traversal stack overflow, bit1: look-back timeout
    uint32_t tile_counter[kMaxBounce];
    uint32_t sh_cursor[kMaxBounce];
    alignas(kClaimLine) uint32_t claims[kMaxBounce + 1][kClaimWords];  // turns: [0] primary queue, [b+1] queues of bounce b
};

// Segments of the shadow and scatter queues of an unordered pass: appends take
// their place from one of several counters (shadow << 32 | scatter) on lines of
// their own, since returning atomics on one address serialise.  Block b of
// k_shade appends to segment (b / kSegGroup) % nseg, which holds at most cap
// entries.  4 samples of the 1920x1080 sphere grid take 13.2 ms with four
// segments, 14.5 with one, 13.2 with sixteen (15.2 with ordered appends: a
// ticket, also one address, and a look-back per block).  A segment's slack is
// memory: with `tight` (the engine, whose queues count against its caller's
// budget) slack and counters stay below 2 bytes a path.
struct Segs {
    uint32_t nseg, cap;
};
constexpr uint32_t kSegGroup = 4;
constexpr uint32_t shade_blocks(uint32_t paths, uint32_t nseg) {
    return (paths + kShadeBlock - 1) / kShadeBlock + (nseg > 1 ? nseg : 0);  // a segment's last tile may be partial
}
Segs segs_for(uint32_t paths, bool tight) {
    Segs s;
    s.nseg = paths >= (tight ? 5u << 17 : 1u << 16) ? kMaxSegs : 1u;
    const uint32_t groups = (shade_blocks(paths, s.nseg) + kSegGroup - 1) / kSegGroup;
    s.cap = s.nseg == 1 ? paths : (groups + s.nseg - 1) / s.nseg * kSegGroup * kShadeBlock;
    return s;
}
// A large pass runs as two parts, each a chain of launches of its own over half
// of the paths, side by side.  The traversal kernels hold the whole chip until
// their queue is dealt out and then wait for their longest walks (CUs were busy
// 79 % of a launch); the other part's next kernel takes the blocks that come
// free.  One part against two: a batch of 12 scenes 45.6 -> 41.9 ms, 16 server
// requests 154 -> 137 ms (passes of 2^22 paths); 4 samples of the 1920x1080
// sphere grid 13.9 -> 13.5 ms in all, 8 of the textured scene (2.9M paths) 3.29
// -> 3.20.  A pass of 2^20 paths is too short: 16 samples of the 256x256 Cornell
// box 1.39 -> 1.43 ms.  In the engine (`tight`) parts also take queue slack of
// their own, below 2 bytes a path from the size given.
constexpr uint32_t kMaxParts = 2;
constexpr uint32_t parts_for(uint32_t paths, bool tight) { return paths >= (tight ? 5u << 18 : 1u << 21) ? kMaxParts : 1u; }
// 64-bit words between two segments' counters, and of all counters
GPR_HD constexpr uint32_t seg_stride(uint32_t nseg) { return nseg > 1 ? 16u : 1u; }
constexpr uint32_t seg_words(uint32_t nseg) { return kMaxBounce * nseg * seg_stride(nseg); }

// Jobs of one multi-job pass (device copy of EngineJob[] plus the path offsets).
struct PassJob {
    EngineJob j;
    uint32_t path_off;  // first path of the job in the pass
    uint32_t pix_off;   // its first pixel among the pass's pixels
    uint32_t pad[2];
};
struct PassBuf {
    uint32_t npaths;
    uint32_t njobs;
    uint32_t npixels;
    uint32_t pad[61];
    PassJob jobs[kMaxPassJobs];
};

struct RenderArgs {
    SceneView sv;              // single-scene renders
    const SceneView* scenes;   // multi-job passes: scene table
    const PassBuf* pass;       // multi-job passes: jobs of this pass
    QueueView q[3];            // A, B (in/scatter alternate), S (shadow)
    float4* fb;
    Ctrl* ctrl;                // cursors of this part of the pass
    Ctrl* base;                // sample and error flags of the pass
    unsigned long long* status;  // [kMaxBounce][ntiles] look-back words
    int2* spill;
    uint32_t paths;            // single-scene: paths of the pass
    uint32_t parts, part;      // the pass runs as one chain of launches or as two, this is one of them
    uint32_t ntiles;           // look-back words per bounce (capacity / kShadeBlock)
    uint32_t nseg, seg_cap;    // segments of the shadow and scatter queues
    unsigned long long* seg;   // [bounce][segment] entries appended: shadow << 32 | scatter
    unsigned long long* last;  // multi-sample passes, [bounce][kLastSpread]: those of the last sample, spread
    uint32_t depth;            // bounces of the sample / pass
    uint32_t chunk_log;        // log2 of the entries a wave takes a turn in extend / shadow
    uint32_t rng_mode;
    uint32_t rr_start;
    unsigned long long seed;
    // multi-sample passes (null: one sample a pass, terms added to fb at once)
    float4* terms;             // [plane][path]: k-th radiance term of a path
    uint8_t* nterm;            // terms of each path so far
    uint32_t tstride;          // paths per plane
    uint32_t log_s;            // single-scene: log2 of the samples of the pass
};

GPR_D unsigned long long* seg_at(const RenderArgs& a, uint32_t bounce, uint32_t g) {
    return a.seg + (bounce * a.nseg + g) * seg_stride(a.nseg);
}
// Paths of a pass before part `part` of `parts`.
GPR_HD constexpr uint32_t part_begin(uint32_t n, uint32_t parts, uint32_t part) {
    if (part == 0) return 0;
    const uint32_t half = ((n + 1) / 2 + kShadeBlock - 1) / kShadeBlock * kShadeBlock;  // no later part is larger
    return part < parts && half < n ? half : n;
}
template <bool MULTI>
GPR_D uint32_t first_path_of(const RenderArgs& a) {
    if constexpr (MULTI) return part_begin(a.pass->npaths, a.parts, a.part);
    else return part_begin(a.paths, a.parts, a.part);
}
template <bool MULTI>
GPR_D uint32_t npaths_of(const RenderArgs& a) {
    uint32_t n;
    if constexpr (MULTI) n = a.pass->npaths;
    else n = a.paths;
    return part_begin(n, a.parts, a.part + 1) - part_begin(n, a.parts, a.part);
}
// Multi-job queue entries carry scene << kJobBits | pass job, so the kernels
// that only need the scene (traversal) index the scene table directly.
constexpr uint32_t kJobBits = 10;
static_assert(kMaxPassJobs <= (1u << kJobBits), "pass job index must fit its bits");
template <bool MULTI>
GPR_D SceneView scene_of(const RenderArgs& a, const QueueView& q, uint32_t i) {
    if constexpr (MULTI) return ldg(a.scenes + (q.job[i] >> kJobBits));
    else return a.sv;
}

// One radiance term of the path `pix` (a queue entry's pix word without its
// flag).  A pass of one sample adds it to the pixel.  A pass of several samples
// holds several paths of a pixel in flight, and a float sum depends on its
// order: each path lists its terms in its own order, and k_accum adds them
// sample by sample, so the image has the bits of passes of one sample.
GPR_D void add_term(const RenderArgs& a, uint32_t pix, c3 v) {
    if (a.terms) {
        const uint32_t k = a.nterm[pix];
        a.terms[(uint64_t)k * a.tstride + pix] = make_float4(v.r, v.g, v.b, 0.f);
        a.nterm[pix] = (uint8_t)(k + 1);
        return;
    }
    float4 x = a.fb[pix];
    x.x = x.x + v.r;
    x.y = x.y + v.g;
    x.z = x.z + v.b;
    a.fb[pix] = x;
}
// Terms a path of `depth` bounces can list: one per vertex on the path
// (emission, environment or the BSDF-sampling term that replaces emission
// after a non-specular bounce) and one light sample per bounce.
constexpr uint32_t max_terms(uint32_t depth) { return 2 * depth + 1; }
static_assert(max_terms(kMaxBounce) < 256, "term counts are bytes");

// Pixel of position p in the slot order of an image: 8-row bands walked column
// by column, so the 64 rays of a wave cover an 8x8 block instead of a 64-pixel
// row and meet fewer different nodes and materials (a sample of the 1920x1080
// sphere grid: 6.48 ms against 6.60 by rows).  Random numbers depend on
// (sample, pixel) only, so the order is free (PCG mode).
GPR_D uint32_t slot_pixel(uint32_t p, uint32_t w, uint32_t npix) {
    const uint32_t band = p / (8 * w), r = p - band * 8 * w;
    const uint32_t left = npix / w - 8 * band, bh = left < 8 ? left : 8u;
    const uint32_t x = r / bh;
    return (8 * band + (r - x * bh)) * w + x;
}

// Camera::generateRay (camera.h:86-119), Mitsuba raster mode.
GPR_D void camera_ray(const float* m, const float* c, float px, float py, v3& o, v3& d) {
    float x = m[0] * px + m[1] * py + m[2] * 0.f + m[3];
    float y = m[4] * px + m[5] * py + m[6] * 0.f + m[7];
    float z = m[8] * px + m[9] * py + m[10] * 0.f + m[11];
    const float w = m[12] * px + m[13] * py + m[14] * 0.f + m[15];
    v3 pc = V(x, y, z);
    if (!(w == 1)) pc = pc / w;
    x = c[0] * 0.f + c[1] * 0.f + c[2] * 0.f + c[3];
    y = c[4] * 0.f + c[5] * 0.f + c[6] * 0.f + c[7];
    z = c[8] * 0.f + c[9] * 0.f + c[10] * 0.f + c[11];
    const float ow = c[12] * 0.f + c[13] * 0.f + c[14] * 0.f + c[15];
    o = V(x, y, z);
    if (!(ow == 1)) o = o / ow;
    const v3 n = norm3(pc);
    d = norm3(V(c[0] * n.x + c[1] * n.y + c[2] * n.z, c[4] * n.x + c[5] * n.y + c[6] * n.z,
                c[8] * n.x + c[9] * n.y + c[10] * n.z));
}

// Camera::generateRay (camera.h:89-107), free mode: film frame precomputed on the host.
GPR_D void camera_ray_free(const SceneView& sv, float px, float py, v3& o, v3& d) {
    const float sx = 2.f * (px / (float)sv.width) - 1.f;
    const float sy = 2.f * (py / (float)sv.height) - 1.f;
    const v3 p = load3(sv.cam_mid) + load3(sv.cam_h) * sx + load3(sv.cam_v) * sy;
    o = load3(sv.cam_eye);
    d = norm3(p - o);
}

template <bool MULTI>
__global__ __launch_bounds__(256) void k_gen(RenderArgs a) {
    const uint32_t tid = blockIdx.x * 256 + threadIdx.x;
    const uint32_t gsz = gridDim.x * 256;
    const uint32_t n = npaths_of<MULTI>(a);
    const uint32_t path = first_path_of<MULTI>(a) + tid;  // in the slot order of the pass
    // clear the per-sample counters, cursors and the look-back words this sample uses
    Ctrl* c = a.ctrl;
    for (uint32_t i = tid; i < kMaxBounce; i += gsz) {
        c->tile_counter[i] = 0u;
        c->sh_cursor[i] = 0u;
    }
    if constexpr (!MULTI) {
        if (a.log_s)
            for (uint32_t i = tid; i < kMaxBounce * kLastSpread; i += gsz) a.last[i] = 0ull;
    }
    for (uint32_t i = tid; i < kMaxBounce * a.nseg; i += gsz) a.seg[i * seg_stride(a.nseg)] = 0ull;
    for (uint32_t i = tid; i < (kMaxBounce + 1) * kClaimSets; i += gsz)
        (&c->claims[0][0])[i * claim_stride<uint32_t>()] = 0u;
    if (!MULTI && a.rng_mode == GPR_RNG_REFERENCE) {
        const uint32_t used_tiles = (n + kShadeBlock - 1) / kShadeBlock;
        const uint64_t nstat = (uint64_t)a.depth * used_tiles;
        for (uint64_t i = tid; i < nstat; i += gsz) a.status[(i / used_tiles) * a.ntiles + i % used_tiles] = 0ull;
    }
    if (tid >= n) return;
    const QueueView& q = a.q[0];
    if constexpr (MULTI) {
        // the job holding the path: last job whose path_off <= path
        const PassBuf* pb = a.pass;
        uint32_t lo = 0, hi = pb->njobs;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (pb->jobs[mid].path_off <= path) lo = mid;
            else hi = mid;
        }
        const EngineJob& jb = pb->jobs[lo].j;
        const uint32_t off = pb->jobs[lo].path_off;
        const uint32_t lp = slot_pixel((path - off) >> jb.log_s, jb.width, jb.npix);
        const uint32_t sub = (path - off) & ((1u << jb.log_s) - 1u);
        uint32_t word = jb.fb_off + lp;
        if (a.terms) {
            word = off + (lp << jb.log_s | sub);
            a.nterm[word] = 0;
        } else if (jb.sample == 0) {
            a.fb[word] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        const uint64_t inc = pcg_inc(jb.sample + sub, lp);
        uint64_t st = pcg_init(jb.seed, inc);
        const float jx = pcg_unit(st, inc);
        const float jy = pcg_unit(st, inc);
        v3 o, d;
        camera_ray(jb.r2c, jb.c2w, (float)(lp % jb.width) + jx, (float)(lp / jb.width) + jy, o, d);
        q.rng[tid] = st;
        q.o_tmin[tid] = make_float4(o.x, o.y, o.z, 0.f);
        q.d_tmax[tid] = make_float4(d.x, d.y, d.z, 1e34f);
        q.w_pdf[tid] = make_float4(1.f, 1.f, 1.f, 0.f);
        q.pix[tid] = word;
        q.job[tid] = (jb.scene << kJobBits) | lo;
    } else {
        const uint32_t W = a.sv.width;
        // reference RNG mode indexes its seeds by slot: slot order = pixel order
        const uint32_t lpix = a.rng_mode == GPR_RNG_REFERENCE ? tid : slot_pixel(path >> a.log_s, W, a.paths >> a.log_s);
        const uint32_t sub = path & ((1u << a.log_s) - 1u);
        const uint32_t sample = a.base->sample + sub;
        const uint32_t x = lpix % W, y = lpix / W;
        float jx, jy;
        if (a.rng_mode == GPR_RNG_REFERENCE) {
            uint32_t s = tea16(tid, sample);  // InitRandom(idx, sample) (pathtracer_kernel.h:92)
            jx = lcg_next(s);
            jy = lcg_next(s);
            q.seed[tid] = s;
        } else {
            const uint64_t inc = pcg_inc(sample, lpix);
            uint64_t st = pcg_init(a.seed, inc);
            jx = pcg_unit(st, inc);
            jy = pcg_unit(st, inc);
            q.rng[tid] = st;
        }
        v3 o, d;
        if (a.sv.cam_free) camera_ray_free(a.sv, (float)x + jx, (float)y + jy, o, d);
        else camera_ray(a.sv.r2c, a.sv.c2w, (float)x + jx, (float)y + jy, o, d);
        q.o_tmin[tid] = make_float4(o.x, o.y, o.z, 0.f);
        q.d_tmax[tid] = make_float4(d.x, d.y, d.z, 1e34f);
        q.w_pdf[tid] = make_float4(1.f, 1.f, 1.f, 0.f);
        const uint32_t word = (lpix << a.log_s) | sub;
        q.pix[tid] = word;
        if (a.terms) a.nterm[word] = 0;
    }
}

template <bool ANY, bool REF_ORDER, class Stack>
GPR_D gpr_hit trace_one(const RenderArgs& a, const SceneView& sv, const Ray3& r, Stack& st) {
    gpr_hit h;
    if constexpr (REF_ORDER) {
        uint32_t nv = 0, nt = 0;
        h = ref_trace<ANY>(sv, r, &nv, &nt);
    } else {
        if (!fast_trace<ANY>(sv, r, st, h)) atomicOr(&a.base->error, 1u);
    }
    return h;
}

// One triangle's shading record, read as five 16-byte loads from its line
// (its corner uvs, needed only for textured hits, are read by resolve_textures).
struct Shade {
    v3 p0, p1, p2, n0, n1, n2;
    uint32_t flags, mat;
};
GPR_D Shade load_shade(const SceneView& sv, uint32_t t) {
    const float4* r = reinterpret_cast<const float4*>(sv.shade + t);
    const float4 a = ldg(r), b = ldg(r + 1), c = ldg(r + 2), d = ldg(r + 3), e = ldg(r + 4);
    Shade s;
    s.p0 = V(a.x, a.y, a.z);
    s.p1 = V(a.w, b.x, b.y);
    s.p2 = V(b.z, b.w, c.x);
    s.n0 = V(c.y, c.z, c.w);
    s.n1 = V(d.x, d.y, d.z);
    s.n2 = V(d.w, e.x, e.y);
    s.flags = __float_as_uint(e.z);
    s.mat = __float_as_uint(e.w);
    return s;
}
// Light pdf (Triangle::pdf + pdf_lights, triangle.h:156-175, pathtracer_kernel.h:338-348)
GPR_D float tri_area(const Shade& s) { return len3(cross3(s.p1 - s.p0, s.p2 - s.p0)) * 0.5f; }
struct Geom {
    v3 p, ns;
};
// Triangle::setupDifferential (triangle.h:104-138)
GPR_D Geom setup_geom(const Shade& s, float u, float v) {
    Geom g;
    g.p = s.p0 * (1 - u - v) + s.p1 * u + s.p2 * v;
    if (s.flags & 1u) g.ns = norm3(s.n0 * (1 - u - v) + s.n1 * u + s.n2 * v);
    else g.ns = norm3(cross3(s.p0 - s.p2, s.p1 - s.p2));
    return g;
}
GPR_D c3 emission_of(const SceneView& sv, const Shade& s) {
    const float* e = sv.mats[s.mat].emission;
    return C(ldg(e), ldg(e + 1), ldg(e + 2));
}
GPR_D float power_heur(float a, float b) {
    a *= a;
    b *= b;
    return a / (a + b);
}

// Walks a segmented queue in turns of 2^lg entries.  Uniform: written member by
// member and chosen from as scalars.  With arrays the compiler kept the walk in each
// lane's scratch memory (44 B; 92 in k_trace) or, in k_shade and the 32-entry shapes,
// in 11 KB of LDS: 16 samples of the 256x256 Cornell box 753 us, now 701; 8 of the
// 803x451 textured scene 2610 and 2521; the batch 40.0 ms and 38.0, 16 served jobs
// 150 and 138.
struct SegWalk {
    uint32_t n0, n1, n2, n3;  // entries of the segments
    uint32_t f1, f2, f3;      // the turns that they start at (the first one at 0)
    uint32_t turns, cap, lg;
    GPR_D uint32_t turns_of(uint32_t n) const { return (n + (1u << lg) - 1) >> lg; }
    GPR_D void init(uint32_t seg_cap, uint32_t log_turn) {
        cap = seg_cap;
        lg = log_turn;
        f1 = turns_of(n0);
        f2 = f1 + turns_of(n1);
        f3 = f2 + turns_of(n2);
        turns = f3 + turns_of(n3);
    }
    GPR_D uint32_t total() const { return n0 + n1 + n2 + n3; }
    GPR_D void range(uint32_t turn, uint32_t& begin, uint32_t& end) const {
        // the last segment that starts at or before the turn (empty ones before it start there too)
        const auto uni = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane(v); };
        const uint32_t s1 = uni(f1), s2 = uni(f2), s3 = uni(f3), m0 = uni(n0), m1 = uni(n1), m2 = uni(n2), m3 = uni(n3);
        const bool after1 = turn >= s1, after2 = turn >= s2, after3 = turn >= s3;
        const uint32_t g = after3 ? 3u : after2 ? 2u : after1 ? 1u : 0u;
        const uint32_t f = after3 ? s3 : after2 ? s2 : after1 ? s1 : 0u;
        const uint32_t m = after3 ? m3 : after2 ? m2 : after1 ? m1 : m0;
        const uint32_t off = (turn - f) << lg;
        begin = g * cap + off;
        end = g * cap + min(off + (1u << lg), m);
    }
};
static_assert(kMaxSegs == 4, "a walk has four segments");
// Entries of the primary queue (one segment of all paths), or of what bounce
// `bounce` appended.
enum QueueKind { kPrimary, kScatter, kShadow };
template <QueueKind KIND, bool MULTI>
GPR_D uint32_t seg_count(const RenderArgs& a, uint32_t bounce, uint32_t g) {
    if constexpr (KIND == kPrimary) return g == 0 ? npaths_of<MULTI>(a) : 0u;
    if (g >= a.nseg) return 0u;
    const unsigned long long v = *seg_at(a, bounce, g);
    return __builtin_amdgcn_readfirstlane(KIND == kShadow ? (uint32_t)(v >> 32) : (uint32_t)v);
}
template <QueueKind KIND, bool MULTI>
GPR_D void seg_counts(const RenderArgs& a, uint32_t bounce, SegWalk& w) {
    w.n0 = seg_count<KIND, MULTI>(a, bounce, 0);
    w.n1 = seg_count<KIND, MULTI>(a, bounce, 1);
    w.n2 = seg_count<KIND, MULTI>(a, bounce, 2);
    w.n3 = seg_count<KIND, MULTI>(a, bounce, 3);
}
// Calls f(i) for the entries of a queue, a turn's lanes together.
template <QueueKind KIND, bool MULTI, int NT, class F>
GPR_D void for_each_entry(const RenderArgs& a, uint32_t bounce, uint32_t* cursor, F&& f) {
    SegWalk w;
    seg_counts<KIND, MULTI>(a, bounce, w);
    w.init(a.seg_cap, turn_log(w.total(), gridDim.x * (NT / 64), a.chunk_log));
    for_each_turn<NT>(cursor, w.turns, [&](uint32_t turn) {
        uint32_t begin, end;
        w.range(turn, begin, end);
        for (uint32_t i = begin + (threadIdx.x & 63); i < end; i += 64) f(i);
    });
}

// Per-lane ray refill over queue entries: a lane whose ray is done takes the
// next entry from a wave-local pool of a turn's entries (one atomic a turn).
// begin(i) sets entry i up and returns true if it finished at once; step()
// advances the lane's ray one node and returns true when it is done.
template <QueueKind KIND, bool MULTI, class Begin, class Step>
GPR_D void refill_loop(const RenderArgs& a, uint32_t bounce, uint32_t* cursor, Begin&& begin, Step&& step) {
    const int lane = threadIdx.x & 63;
    // whole turns only: a pool feeds all lanes of its wave
    SegWalk w;
    seg_counts<KIND, MULTI>(a, bounce, w);
    w.init(a.seg_cap, a.chunk_log);
    uint32_t pb = 0, pe = 0;  // wave-local pool of entries (wave-uniform)
    bool drained = false;
    bool active = false;
    while (true) {
        const unsigned long long need = __ballot(!active);
        if (need != 0ull && !(drained && pb == pe)) {
            const uint32_t cnt = (uint32_t)__popcll(need);
            const uint32_t rank =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(need >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)need, 0u));
            const uint32_t avail = pe - pb;
            uint32_t nb = pe, ne = pe;
            if (avail < cnt && !drained) {
                uint32_t b = 0;
                if (lane == 0) b = atomicAdd(cursor, 1u);
                b = __builtin_amdgcn_readfirstlane(b);
                drained = b + 1 >= w.turns;
                if (b < w.turns) w.range(b, nb, ne);
            }
            if (!active) {
                const bool from_old = rank < avail;
                const uint32_t idx = from_old ? pb + rank : nb + (rank - avail);
                if (from_old || idx < ne) active = !begin(idx);
            }
            if (avail >= cnt) {
                pb += cnt;
            } else {
                const uint32_t taken = nb + (cnt - avail);
                pb = taken < ne ? taken : ne;
                pe = ne;
            }
        }
        if (__ballot(active) == 0ull) {
            if (drained && pb == pe) break;
            continue;
        }
        if (active) active = !step();
    }
}

GPR_D Ray3 queue_ray(const QueueView& q, uint32_t i) {
    const float4 ot = q.o_tmin[i], dt = q.d_tmax[i];
    Ray3 r;
    r.o = V(ot.x, ot.y, ot.z);
    r.d = V(dt.x, dt.y, dt.z);
    r.tmin = ot.w;
    r.tmax = dt.w;
    return r;
}

// After the closest hit of entry i: for scattered rays the BSDF-sampling MIS
// term and, in reference RNG mode, its roulette (pathtracer_kernel.h:684-749).
// The term waits in the entry for the next bounce's shading or k_flush
// (tmin = kMisTerm marks it): the shadow rays of the same bounce add theirs
// meanwhile, and a path's terms keep the order light sample, BSDF sample.  It
// replaces the origin, which only a miss reads, or the t, u, v of a miss that
// the roulette made of a hit.
constexpr float kMisTerm = -1.f;
GPR_D c3 mis_term(const float4& o_tmin, const float4& hit) {
    return __float_as_int(hit.y) != -1 ? C(o_tmin.x, o_tmin.y, o_tmin.z) : C(hit.x, hit.z, hit.w);
}
template <bool PRIMARY, bool MULTI>
GPR_D void extend_finish(const RenderArgs& a, const QueueView& q, uint32_t i, const SceneView& sv, const Ray3& r,
                         gpr_hit h, uint32_t bounce) {
    if (!PRIMARY) {
        const float4 wp = q.w_pdf[i];
        const bool spec = (q.pix[i] >> 31) != 0;
        const c3 w = C(wp.x, wp.y, wp.z);
        bool dropped = false;
        if (!MULTI && a.rng_mode == GPR_RNG_REFERENCE) {
            // roulette without reweighting; a terminated path is a miss (pathtracer_kernel.h:738-748)
            const float u_rr = lcg_next(q.seed[i]);
            dropped = cmax(w) < 1 && bounce > 3 && u_rr < fmax_h(0.05f, 1 - cmax(w));
        }
        if (h.id != -1 && !spec) {
            const Shade ts = load_shade(sv, (uint32_t)h.id);
            const c3 le = emission_of(sv, ts);
            if (!black(le)) {
                const Geom lg = setup_geom(ts, h.u, h.v);
                float lpdf = 1.f / tri_area(ts);
                lpdf /= sv.nlights;
                const float d = h.t;
                lpdf *= d * d / fabsf(dot3(r.d, lg.ns));
                const c3 fl = dot3(-r.d, lg.ns) > 0 ? le : C(0.f);
                const float wgt = power_heur(wp.w, lpdf);
                const c3 v = w * fl * wgt;
                if (dropped) {
                    h.t = v.r;
                    h.u = v.g;
                    h.v = v.b;
                    q.o_tmin[i].w = kMisTerm;
                } else {
                    q.o_tmin[i] = make_float4(v.r, v.g, v.b, kMisTerm);
                }
            }
        }
        if (dropped) h.id = -1;
    }
    q.hit[i] = make_float4(h.t, __int_as_float(h.id), h.u, h.v);
}

// After the any-hit test of shadow entry i (pathtracer_kernel.h:642-664).
GPR_D void shadow_finish(const RenderArgs& a, const QueueView& q, uint32_t i, const gpr_hit& h) {
    if (h.id == -1) {
        const float4 wp = q.w_pdf[i];
        add_term(a, q.pix[i] & 0x7fffffffu, C(wp.x, wp.y, wp.z));
    }
}

// A queue this short walks its rays with four lanes each (quad_trace): a launch
// then takes as long as its longest walk.  Never / up to 2^16 / 2^17 entries: 57,000
// paths of the textured scene 1000 / 845 / 800 us, 60,000 of the sphere grid 1232 /
// 1018 / 980, a 300x200 frame 746 / 620 / 593; 12-job batch 41.1 / 40.6 ms, then
// with cheaper turns 39.4 / 39.0; 16 served jobs 141 / 137 ms.  3 * 2^15 entries:
// 802, 1022, 620 us; 3 * 2^16: 801, 974, 594 us, but served jobs 138 ms for 136.5.
constexpr uint32_t kQuadEntries = 1u << 17;
// log2 of the entries of a turn: turn_log, or at most 16 where four lanes take one
GPR_D uint32_t entries_log(uint32_t total, uint32_t waves, uint32_t chunk_log, bool quads) {
    const uint32_t lg = turn_log(total, waves, chunk_log);
    return quads && total <= kQuadEntries ? min(lg, 4u) : lg;
}
// One entry's walk by four lanes; finish(hit) runs in the lane that holds the hit.
template <bool ANY, int NT, int STACK, class F>
GPR_D void quad_entry(const RenderArgs& a, void* lds, const SceneView& sv, const Ray3& r, F&& finish) {
    QuadStack<typename StackEntry<ANY>::type, STACK> st;
    st.template place<NT>(lds, a.spill);
    gpr_hit h;
    uint32_t own;
    const bool ok = quad_trace<ANY>(sv, r, st, h, own);
    if ((threadIdx.x & 3) != own) return;
    if (!ok) atomicOr(&a.base->error, 1u);
    finish(h);
}

// extend: closest hit; for scattered rays also the BSDF-sampling MIS term.
// REFILL: per-lane ray refill (BVH4 traversal only).
template <bool PRIMARY, bool REF_ORDER, bool MULTI, int NT, int SL, bool REFILL = false>
__global__ __launch_bounds__(NT) void k_extend(RenderArgs a, uint32_t bounce) {
    using Stack = LaneStack<false, SL>;
    __shared__ typename Stack::Entry lds[SL * NT];
    Stack st;
    st.template place<NT>(lds, a.spill);
    // queue: primary = A; at bounce b the scatter queue is q[(b+1)&1]
    const QueueView& q = a.q[PRIMARY ? 0 : ((bounce + 1) & 1)];
    constexpr QueueKind kKind = PRIMARY ? kPrimary : kScatter;
    uint32_t* cur = a.ctrl->claims[PRIMARY ? 0 : bounce + 1];
    if constexpr (REFILL && !REF_ORDER) {
        uint32_t ei = 0;
        SceneView sv;
        Trav t;
        refill_loop<kKind, MULTI>(
            a, bounce, cur,
            [&](uint32_t i) {
                ei = i;
                sv = scene_of<MULTI>(a, q, i);
                trav_begin<false>(sv, queue_ray(q, i), st, t);
                if (trav_live(sv, t)) return false;
                extend_finish<PRIMARY, MULTI>(a, q, i, sv, t.r, t.hit, bounce);
                return true;
            },
            [&]() {
                trav_step<false>(sv, st, t);
                if (trav_live(sv, t)) return false;
                if (t.node != kTravDone) atomicOr(&a.base->error, 1u);
                extend_finish<PRIMARY, MULTI>(a, q, ei, sv, t.r, t.hit, bounce);
                return true;
            });
    } else {
        if constexpr (!REF_ORDER) {
            SegWalk w;
            seg_counts<kKind, MULTI>(a, bounce, w);
            const uint32_t total = w.total();
            if (total <= kQuadEntries) {
                w.init(a.seg_cap, entries_log(total, gridDim.x * (NT / 64), a.chunk_log, true));
                for_each_turn<NT>(cur, w.turns, [&](uint32_t turn) {
                    uint32_t begin, end;
                    w.range(turn, begin, end);
                    const uint32_t i = begin + (threadIdx.x & 63) / 4;
                    if (i >= end) return;
                    const SceneView sv = scene_of<MULTI>(a, q, i);
                    const Ray3 r = queue_ray(q, i);
                    quad_entry<false, NT, 4 * SL>(a, lds, sv, r, [&](const gpr_hit& h) {
                        extend_finish<PRIMARY, MULTI>(a, q, i, sv, r, h, bounce);
                    });
                });
                return;
            }
        }
        for_each_entry<kKind, MULTI, NT>(a, bounce, cur, [&](uint32_t i) {
            const SceneView sv = scene_of<MULTI>(a, q, i);
            const Ray3 r = queue_ray(q, i);
            const gpr_hit h = trace_one<false, REF_ORDER>(a, sv, r, st);
            extend_finish<PRIMARY, MULTI>(a, q, i, sv, r, h, bounce);
        });
    }
}

// shadow: any hit + accumulate_light_sampling_contribution
// (pathtracer_kernel.h:642-664), with per-lane ray refill.
template <int NT, int SL>
__global__ __launch_bounds__(NT) void k_shadow(RenderArgs a, uint32_t bounce) {
    using Stack = LaneStack<true, SL>;
    __shared__ typename Stack::Entry lds[SL * NT];
    Stack st;
    st.template place<NT>(lds, a.spill);
    const QueueView& q = a.q[2];
    uint32_t ei = 0;
    SceneView sv;
    Trav t;
    refill_loop<kShadow, true>(
        a, bounce, &a.ctrl->sh_cursor[bounce],
        [&](uint32_t i) {
            ei = i;
            sv = scene_of<true>(a, q, i);
            trav_begin<true>(sv, queue_ray(q, i), st, t);
            if (trav_live(sv, t)) return false;
            shadow_finish(a, q, i, t.hit);
            return true;
        },
        [&]() {
            trav_step<true>(sv, st, t);
            if (trav_live(sv, t)) return false;
            if (t.node != kTravDone) atomicOr(&a.base->error, 1u);
            shadow_finish(a, q, ei, t.hit);
            return true;
        });
}

// The scattered rays of a bounce (closest hit) and its shadow rays (any hit) in
// one launch: bound by the latency of the walks, and each launch ends in a tail
// of a few long ones; here the tails overlap, and a bounce has one boundary
// less.  Scattered rays come first, their walks are longer.  Two kernels
// against one: a 1280x720 reference-RNG frame of depth 8 2332 -> 2082 us, 16
// samples of the textured scene (362,000 pixels) 3.80 -> 3.55 ms, a 12-job batch
// 55.6 -> 48.6 ms, 16 served jobs 177 -> 158 ms.
template <bool REF_ORDER, bool MULTI, int NT, int SL>
__global__ __launch_bounds__(NT) void k_trace(RenderArgs a, uint32_t bounce) {
    __shared__ uint2 lds[SL * NT];
    const QueueView& qx = a.q[(bounce + 1) & 1];
    const QueueView& qs = a.q[2];
    SegWalk wx, ws;
    seg_counts<kScatter, MULTI>(a, bounce, wx);
    seg_counts<kShadow, MULTI>(a, bounce, ws);
    const uint32_t total = wx.total() + ws.total();
    const uint32_t lg = entries_log(total, gridDim.x * (NT / 64), a.chunk_log, !REF_ORDER);
    wx.init(a.seg_cap, lg);
    ws.init(a.seg_cap, lg);
    if (!REF_ORDER && total <= kQuadEntries) {
        for_each_turn<NT>(a.ctrl->claims[bounce + 1], wx.turns + ws.turns, [&](uint32_t turn) {
            const uint32_t quad = (threadIdx.x & 63) / 4;
            uint32_t begin, end;
            if (turn < wx.turns) {
                wx.range(turn, begin, end);
                const uint32_t i = begin + quad;
                if (i >= end) return;
                const SceneView sv = scene_of<MULTI>(a, qx, i);
                const Ray3 r = queue_ray(qx, i);
                quad_entry<false, NT, 4 * SL>(a, lds, sv, r, [&](const gpr_hit& h) {
                    extend_finish<false, MULTI>(a, qx, i, sv, r, h, bounce);
                });
            } else {
                ws.range(turn - wx.turns, begin, end);
                const uint32_t i = begin + quad;
                if (i >= end) return;
                const SceneView sv = scene_of<MULTI>(a, qs, i);
                // half the entry, twice the entries: every wave keeps to its own part of the LDS
                quad_entry<true, NT, 8 * SL>(a, lds, sv, queue_ray(qs, i),
                                             [&](const gpr_hit& h) { shadow_finish(a, qs, i, h); });
            }
        });
        return;
    }
    for_each_turn<NT>(a.ctrl->claims[bounce + 1], wx.turns + ws.turns, [&](uint32_t turn) {
        uint32_t begin, end;
        if (turn < wx.turns) {
            LaneStack<false, SL> st;
            st.template place<NT>(lds, a.spill);
            wx.range(turn, begin, end);
            for (uint32_t i = begin + (threadIdx.x & 63); i < end; i += 64) {
                const SceneView sv = scene_of<MULTI>(a, qx, i);
                const Ray3 r = queue_ray(qx, i);
                const gpr_hit h = trace_one<false, REF_ORDER>(a, sv, r, st);
                extend_finish<false, MULTI>(a, qx, i, sv, r, h, bounce);
            }
        } else {
            LaneStack<true, 2 * SL> st;  // half the entry, twice the entries
            st.template place<NT>(lds, a.spill);
            ws.range(turn - wx.turns, begin, end);
            for (uint32_t i = begin + (threadIdx.x & 63); i < end; i += 64) {
                const SceneView sv = scene_of<MULTI>(a, qs, i);
                const gpr_hit h = trace_one<true, REF_ORDER>(a, sv, queue_ray(qs, i), st);
                shadow_finish(a, qs, i, h);
            }
        }
    });
}

// Adds the BSDF-sampling terms that the last bounce's scattered rays left.
template <bool MULTI>
__global__ __launch_bounds__(256) void k_flush(RenderArgs a) {
    const uint32_t bounce = a.depth - 1;
    const QueueView& q = a.q[a.depth & 1];
    SegWalk w;
    seg_counts<kScatter, MULTI>(a, bounce, w);
    w.init(a.seg_cap, 8);
    for (uint32_t turn = blockIdx.x; turn < w.turns; turn += gridDim.x) {
        uint32_t begin, end;
        w.range(turn, begin, end);
        const uint32_t i = begin + threadIdx.x;
        if (i >= end) continue;
        const float4 o = q.o_tmin[i];
        if (o.w == kMisTerm) add_term(a, q.pix[i] & 0x7fffffffu, mis_term(o, q.hit[i]));
    }
}

// ------------------------------------------------------------- shade ----
struct Out {
    v3 o, d;
    float tmin, tmax;
    c3 w;
    float pdf;
    bool spec;
};

// 64-bit look-back word: [63:62] flag (1 aggregate, 2 inclusive) [61:31] shadow [30:0] scatter
GPR_D unsigned long long pack_status(uint32_t flag, uint32_t sh, uint32_t sc) {
    return ((unsigned long long)flag << 62) | ((unsigned long long)sh << 31) | (unsigned long long)sc;
}

// Publishes a tile's counts and returns the sum of those before it (without the
// flag), by the 64 lanes of one wave: a step back reads 64 tiles.
GPR_D unsigned long long look_back(unsigned long long* st, uint32_t tile, unsigned long long mine, uint32_t* error) {
    const uint32_t lane = threadIdx.x & 63;
    constexpr unsigned long long kCounts = (1ull << 62) - 1;
    unsigned long long sum = 0;
    if (tile > 0) {
        if (lane == 0) __hip_atomic_store(st + tile, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        uint32_t spins = 0;
        for (uint32_t end = tile;;) {  // tiles from end on are summed
            unsigned long long v = 2ull << 62;  // nothing before the first tile
            if (lane < end) v = __hip_atomic_load(st + (end - 1 - lane), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long open = __ballot((v >> 62) == 0), whole = __ballot((v >> 62) == 2);
            const int stop = whole ? __builtin_ctzll(whole) : 63;  // the lane whose tile ends the step
            if (open & (2ull << stop) - 1) {
                // predecessor tiles took their ids earlier and are resident: this wait ends
                if (++spins > (1u << 26)) {
                    if (lane == 0) atomicOr(error, 2u);
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
                continue;
            }
            v = (int)lane <= stop ? v & kCounts : 0ull;
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
            sum += v;
            if (whole) break;
            end -= 64;
        }
    }
    if (lane == 0)
        __hip_atomic_store(st + tile, (2ull << 62) | (sum + (mine & kCounts)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return sum;
}

// ORDERED: appends keep the queue order (reference RNG mode: seeds belong to
// slots), by tickets and a decoupled look-back over one segment.  Otherwise a
// block takes its place in its segment with one atomic.
// Ordered tiles take a ticket each, an atomic on one address (~12 ns, one after
// the other), so they are larger: 4 samples of the 640x360 Cornell box in reference
// RNG mode 2093 / 1942 / 1799 / 1719 us with 256 entries and a look-back by one
// thread, and 256 / 512 / 1024 entries with a look-back by a wave; a 1600x900
// textured frame 2124 / 2119 / 2046 / 2049, a 300x200 frame 618 / 609 / 617 / 700.
constexpr int kOrderedBlock = 512;
template <bool MULTI, bool ORDERED>
__global__ __launch_bounds__(ORDERED ? kOrderedBlock : kShadeBlock) void k_shade(RenderArgs a, uint32_t bounce) {
    constexpr int NB = ORDERED ? kOrderedBlock : kShadeBlock;
    __shared__ uint32_t s_tile;
    __shared__ uint32_t s_wave[2][NB / 64];
    __shared__ uint32_t s_base[2];
    __shared__ uint32_t s_last[NB / 64];
    uint32_t tile, ntiles_in, i, n_end;
    if constexpr (ORDERED) {
        const uint32_t n_in = bounce == 0 ? npaths_of<MULTI>(a) : (uint32_t)*seg_at(a, bounce - 1, 0);
        if (threadIdx.x == 0) s_tile = atomicAdd(&a.ctrl->tile_counter[bounce], 1u);
        __syncthreads();
        tile = s_tile;
        ntiles_in = (n_in + NB - 1) / NB;
        if (tile >= ntiles_in) return;
        i = tile * NB + threadIdx.x;
        n_end = n_in;
    } else {
        constexpr uint32_t kLog = 8;
        static_assert(kShadeBlock == 1 << kLog, "a turn is a block");
        SegWalk w;
        if (bounce == 0) seg_counts<kPrimary, MULTI>(a, 0, w);
        else seg_counts<kScatter, MULTI>(a, bounce - 1, w);
        w.init(a.seg_cap, kLog);
        tile = blockIdx.x;
        if (tile >= w.turns) return;
        w.range(tile, i, n_end);
        i += threadIdx.x;
    }
    const QueueView& qi = a.q[bounce & 1];
    const QueueView& qs = a.q[(bounce + 1) & 1];
    const QueueView& qsh = a.q[2];
    bool valid = i < n_end;
    uint32_t job = 0, rr_start = a.rr_start, sample = 0, lpix = 0;
    SceneView sv;
    if constexpr (MULTI) {
        if (valid) {
            job = qi.job[i];  // scene << kJobBits | pass job, copied to the appended entries
            const PassJob pj = ldg(a.pass->jobs + (job & ((1u << kJobBits) - 1)));
            sv = ldg(a.scenes + (job >> kJobBits));
            // a job's paths stop at its own depth
            valid = bounce < pj.j.max_depth;
            if (!valid) {
                const float4 o = qi.o_tmin[i];
                if (o.w == kMisTerm) add_term(a, qi.pix[i] & 0x7fffffffu, C(o.x, o.y, o.z));
            }
            rr_start = pj.j.rr_start;
            const uint32_t word = qi.pix[i] & 0x7fffffffu;
            lpix = word - pj.j.fb_off;
            sample = pj.j.sample;
            if (a.terms) {
                lpix = (word - pj.path_off) >> pj.j.log_s;
                sample += (word - pj.path_off) & ((1u << pj.j.log_s) - 1u);
            }
        }
    } else {
        sv = a.sv;
    }
    bool has_sh = false, has_sc = false;
    Out osh, osc;
    uint32_t pix = 0;
    unsigned long long rng_out = 0;
    if (valid) {
        const float4 dt = qi.d_tmax[i], hh = qi.hit[i], wp = qi.w_pdf[i];
        const uint32_t pw = qi.pix[i];
        pix = pw & 0x7fffffffu;
        if constexpr (!MULTI) {
            lpix = pix >> a.log_s;
            sample = a.base->sample + (pix & ((1u << a.log_s) - 1u));
        }
        const bool spec = (pw >> 31) != 0;
        const v3 rd = V(dt.x, dt.y, dt.z);
        const c3 w = C(wp.x, wp.y, wp.z);
        const int32_t hid = __float_as_int(hh.y);
        float smp[8];
        if constexpr (ORDERED) {
            uint32_t s = qi.seed[i];
#pragma unroll
            for (int k = 0; k < 8; ++k) smp[k] = lcg_next(s);
            qi.seed[i] = s;
        } else {
            const uint64_t inc = pcg_inc(sample, lpix);
            uint64_t s = qi.rng[i];
#pragma unroll
            for (int k = 0; k < 8; ++k) smp[k] = pcg_unit(s, inc);
            rng_out = s;
        }
        if constexpr (ORDERED) {
            if (bounce != 0) {
                const float4 o = qi.o_tmin[i];
                if (o.w == kMisTerm) add_term(a, pix, mis_term(o, hh));
            }
        }
        if (hid != -1) {
            const uint32_t t = (uint32_t)hid;
            const Shade ts = load_shade(sv, t);
            const Geom g = setup_geom(ts, hh.z, hh.w);
            const v3 wo = -norm3(rd);
            gpr_material m = ldg(sv.mats + ts.mat);
            if (sv.ntex != 0 && has_textures(m)) resolve_textures(sv, m, t, ts.flags, hh.z, hh.w);
            const Frame fr = make_frame(g.ns);
            if (bounce == 0 || spec) {
                const c3 le = loadc(m.emission);
                if (!black(le)) {
                    const c3 fl = dot3(wo, g.ns) > 0 ? le : C(0.f);
                    add_term(a, pix, w * fl);
                }
            } else if (!ORDERED && !black(loadc(m.emission))) {
                // a light met by a non-specular scattered ray: k_trace left its MIS term
                const float4 o = qi.o_tmin[i];
                add_term(a, pix, C(o.x, o.y, o.z));
            }
            if (!bsdf_is_delta(m) && sv.nlights > 0) {
                // sample_lights (pathtracer_kernel.h:323-336): uniform by count, uniform on the triangle
                const uint32_t ln = sv.nlights;
                uint32_t lid = (uint32_t)(smp[0] * ln);
                if (lid > ln - 1) lid = ln - 1;
                const uint32_t lt = ldg(sv.lights + lid);
                const float sa = sqrtf(smp[1]);
                const Shade ls = load_shade(sv, lt);
                const Geom lg = setup_geom(ls, 1 - sa, smp[2] * sa);
                float lpdf = 1.f / tri_area(ls);
                lpdf /= ln;
                v3 wi = lg.p - g.p;
                const float d2 = dot3(wi, wi);
                const float dd = sqrtf(d2);
                wi = wi / dd;
                lpdf *= d2 / fabsf(dot3(wi, lg.ns));
                if (isinf(lpdf)) lpdf = 0.f;
                const c3 fl = dot3(-wi, lg.ns) > 0 ? emission_of(sv, ls) : C(0.f);
                c3 fb;
                float bpdf;
                bsdf_eval_local(m, to_local(fr, wo), to_local(fr, wi), fb, bpdf);
                const float wgt = power_heur(lpdf, bpdf);
                if (lpdf > 0.f) {
                    const c3 ow = w * fl * fb * wgt / lpdf;
                    if (!black(ow)) {
                        osh.o = g.p - rd * 1.0e-4f;
                        osh.d = lg.p - osh.o;
                        osh.tmin = 0.f;
                        osh.tmax = 0.9999f;
                        osh.w = ow;
                        osh.pdf = 0.f;
                        osh.spec = true;
                        has_sh = true;
                    }
                }
            }
            {
                const BSample bs = bsdf_sample(m, fr, wo, smp[5], smp[6], smp[4]);
                c3 ow = bs.pdf == 0.f ? C(0.f) : w * bs.f / bs.pdf;
                if (!ORDERED && bounce >= rr_start && !black(ow)) {
                    const float qq = fmax_h(0.05f, 1 - cmax(ow));
                    if (smp[7] < qq) ow = C(0.f);
                    else ow = ow / (1 - qq);
                }
                if (!black(ow)) {
                    osc.o = g.p;
                    osc.d = bs.wi;
                    osc.tmin = 1e-4f;
                    osc.tmax = 1e38f;
                    osc.w = ow;
                    osc.pdf = bs.pdf;
                    osc.spec = bs.specular;
                    has_sc = true;
                }
            }
        } else if (sv.has_env) {
            c3 le = C(sv.env[0], sv.env[1], sv.env[2]);
            if (sv.env_tex) {
                const float4 ot = qi.o_tmin[i];
                le = env_le(sv, V(ot.x, ot.y, ot.z), rd);
            }
            add_term(a, pix, w * le);
        }
    }
    // ---- order-preserving compaction of both appends
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long bsh = __ballot(has_sh), bsc = __ballot(has_sc);
    const uint32_t lsh = __builtin_amdgcn_mbcnt_hi((uint32_t)(bsh >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bsh, 0u));
    const uint32_t lsc = __builtin_amdgcn_mbcnt_hi((uint32_t)(bsc >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bsc, 0u));
    if (lane == 0) {
        s_wave[0][wave] = (uint32_t)__popcll(bsh);
        s_wave[1][wave] = (uint32_t)__popcll(bsc);
    }
    if constexpr (!MULTI && !ORDERED) {
        if (a.log_s) {  // what gpr_renderer_queue_sizes reports of the last sample
            const uint32_t smask = (1u << a.log_s) - 1u;
            const unsigned long long mine = __ballot(valid && (pix & smask) == smask);
            if (lane == 0) s_last[wave] = (uint32_t)__popcll(bsh & mine) << 16 | (uint32_t)__popcll(bsc & mine);
        }
    }
    __syncthreads();
    if constexpr (!MULTI && !ORDERED) {
        if (a.log_s && threadIdx.x == 0) {
            uint32_t l = 0;
#pragma unroll
            for (int k = 0; k < kShadeBlock / 64; ++k) l += s_last[k];
            if (l) atomicAdd(&a.last[bounce * kLastSpread + tile % kLastSpread], (unsigned long long)(l >> 16) << 32 | (l & 0xffffu));
        }
    }
    uint32_t wsh = 0, wsc = 0, tsh = 0, tsc = 0;
#pragma unroll
    for (int k = 0; k < NB / 64; ++k) {
        if (k < wave) {
            wsh += s_wave[0][k];
            wsc += s_wave[1][k];
        }
        tsh += s_wave[0][k];
        tsc += s_wave[1][k];
    }
    if constexpr (!ORDERED) {
        if (threadIdx.x == 0) {
            const uint32_t g = blockIdx.x / kSegGroup % a.nseg;
            unsigned long long at = 0;
            if (tsh + tsc) at = atomicAdd(seg_at(a, bounce, g), (unsigned long long)tsh << 32 | tsc);
            s_base[0] = g * a.seg_cap + (uint32_t)(at >> 32);
            s_base[1] = g * a.seg_cap + (uint32_t)at;
        }
    } else if (wave == 0) {
        unsigned long long* st = a.status + (uint64_t)bounce * a.ntiles;
        const unsigned long long before = look_back(st, tile, pack_status(1, tsh, tsc), &a.base->error);
        if (lane == 0) {
            const uint32_t psh = (uint32_t)(before >> 31), psc = (uint32_t)(before & 0x7fffffffu);
            s_base[0] = psh;
            s_base[1] = psc;
            if (tile == ntiles_in - 1)
                *seg_at(a, bounce, 0) = (unsigned long long)(psh + tsh) << 32 | (psc + tsc);
        }
    }
    __syncthreads();
    if (has_sh) {
        const uint32_t s = s_base[0] + wsh + lsh;
        qsh.o_tmin[s] = make_float4(osh.o.x, osh.o.y, osh.o.z, osh.tmin);
        qsh.d_tmax[s] = make_float4(osh.d.x, osh.d.y, osh.d.z, osh.tmax);
        qsh.w_pdf[s] = make_float4(osh.w.r, osh.w.g, osh.w.b, osh.pdf);
        qsh.pix[s] = pix | 0x80000000u;
        if constexpr (MULTI) qsh.job[s] = job;
    }
    if (has_sc) {
        const uint32_t s = s_base[1] + wsc + lsc;
        qs.o_tmin[s] = make_float4(osc.o.x, osc.o.y, osc.o.z, osc.tmin);
        qs.d_tmax[s] = make_float4(osc.d.x, osc.d.y, osc.d.z, osc.tmax);
        qs.w_pdf[s] = make_float4(osc.w.r, osc.w.g, osc.w.b, osc.pdf);
        qs.pix[s] = pix | (osc.spec ? 0x80000000u : 0u);
        if constexpr (!ORDERED) qs.rng[s] = rng_out;
        if constexpr (MULTI) qs.job[s] = job;
    }
}

__global__ void k_finish(Ctrl* c, uint32_t samples) {
    if (threadIdx.x == 0) c->sample = c->sample + samples;
}

// Adds the terms of a multi-sample pass to their pixels, in sample order and
// within a sample in the order the path met them.
template <bool MULTI>
__global__ __launch_bounds__(256) void k_accum(RenderArgs a) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    uint32_t log_s = a.log_s, path = p << a.log_s, fbi = p;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (MULTI) {
        const PassBuf* pb = a.pass;
        if (p >= pb->npixels) return;
        uint32_t lo = 0, hi = pb->njobs;  // the job holding pixel p: last job whose pix_off <= p
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (pb->jobs[mid].pix_off <= p) lo = mid;
            else hi = mid;
        }
        const EngineJob& jb = pb->jobs[lo].j;
        const uint32_t lp = p - pb->jobs[lo].pix_off;
        log_s = jb.log_s;
        path = pb->jobs[lo].path_off + (lp << log_s);
        fbi = jb.fb_off + lp;
        if (jb.sample != 0) x = a.fb[fbi];
    } else {
        if (p >= (a.paths >> log_s)) return;
        x = a.fb[fbi];
    }
    for (uint32_t j = path; j < path + (1u << log_s); ++j) {
        const uint32_t n = a.nterm[j];
        for (uint32_t k = 0; k < n; ++k) {
            const float4 v = a.terms[(uint64_t)k * a.tstride + j];
            x.x = x.x + v.x;
            x.y = x.y + v.y;
            x.z = x.z + v.z;
        }
    }
    a.fb[fbi] = x;
}

__global__ void k_clear_fb(float4* fb, uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) fb[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

__global__ void k_set_sample(Ctrl* c, uint32_t s) {
    if (threadIdx.x == 0) {
        c->sample = s;
        c->error = 0;
    }
}

constexpr uint64_t kReadPixels = 1ull << 20;  // pixels packed for the host at once

// The three channels of n frame-buffer pixels.
__global__ __launch_bounds__(256) void k_pack_rgb(const float4* __restrict__ fb, uint32_t n, float* __restrict__ out) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float4 x = fb[i];
    out[3ull * i] = x.x;
    out[3ull * i + 1] = x.y;
    out[3ull * i + 2] = x.z;
}

inline uint32_t div_up(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

}  // namespace

// The pixels are packed on the device and land in the caller's buffer.  Bound by
// the host's first touch of that buffer: copied as 16-byte pixels to a buffer of
// their own and repacked by the host, a 1920x1080 image took 10.2 ms, now 3.5
// (of a render of 4 samples 20.7 -> 14.0 ms in all, 803x451 and 8 samples 3.50
// -> 3.20).
int PixelReader::read(int device, const float4* fb, uint64_t n, float* rgb, hipStream_t st) {
    std::lock_guard<std::mutex> lk(mu);
    const uint64_t most = std::min<uint64_t>(n, kReadPixels);
    int now = -1;
    GPR_HIP(hipGetDevice(&now));
    if (now != device || scratch.alloc(12 * most) != GPR_OK) {
        // a thread of another device may not launch on these pixels; or no room for the scratch
        (void)hipGetLastError();
        std::vector<float4> tmp(n);
        GPR_HIP(hipMemcpyAsync(tmp.data(), fb, 16 * n, hipMemcpyDeviceToHost, st));
        GPR_HIP(hipStreamSynchronize(st));
        for (uint64_t i = 0; i < n; ++i) {
            rgb[3 * i] = tmp[i].x;
            rgb[3 * i + 1] = tmp[i].y;
            rgb[3 * i + 2] = tmp[i].z;
        }
        return GPR_OK;
    }
    float* d = scratch.as<float>();
    for (uint64_t at = 0; at < n; at += most) {
        const uint32_t m = (uint32_t)std::min<uint64_t>(most, n - at);
        hipLaunchKernelGGL(k_pack_rgb, dim3(div_up(m, 256)), dim3(256), 0, st, fb + at, m, d);
        GPR_HIP(hipGetLastError());
        GPR_HIP(hipMemcpyAsync(rgb + 3 * at, d, 12ull * m, hipMemcpyDeviceToHost, st));
    }
    GPR_HIP(hipStreamSynchronize(st));
    return GPR_OK;
}

// Multi-sample passes.  A small image (or the
// late bounces of any image) leaves the chip idle and every launch pays the
// latency of its longest ray, so a pass renders up to 2^kMaxLogS samples at
// once.  Paths are pixel-major: the samples of a pixel sit in neighbouring
// lanes, which keeps waves coherent.  16 samples of the 256x256 Cornell box
// take 2.4 ms in one pass against 6.4 ms in 16; 4 samples of the 1920x1080
// sphere grid 17.0 ms against 25.9, and passes of 2^20 / 2^21 / 2^22 / 2^23 /
// 2^24 paths render 8 samples of an 803x451 textured scene in 12.7 / 7.8 / 5.7
// / 5.7 / 5.7 ms and 4 of the sphere grid in 26.5 / 26.5 / 20.1 / 17.6 / 17.3.
// The multi-job engine's passes do the same per job: a batch of 12 scenes at
// 128^2 to 512^2, 16 samples, takes 69 ms instead of 92, a burst of 16 requests
// of 4 to 64 samples to the server 231 instead of 430.
constexpr uint32_t kMaxLogS = 6;
constexpr uint64_t kPassPaths = 1ull << 23;   // paths of a multi-sample pass at most
constexpr uint64_t kPassBytes = 6ull << 30;   // its queues and term lists at most

// ---------------------------------------------------------- engine ----
// Kernel set of one traversal configuration of the multi-job pass.
namespace {
struct PassKernels {
    void (*ext_primary)(RenderArgs, uint32_t);
    void (*trace)(RenderArgs, uint32_t);   // scattered and shadow rays, or the scattered ones where shadow is not null
    void (*shadow)(RenderArgs, uint32_t);
    int nt, sl, layout;
};
template <int NT, int SL, bool R>
PassKernels pass_kernels() {
    if constexpr (R)
        return {k_extend<true, false, true, NT, SL, true>, k_extend<false, false, true, NT, SL, true>,
                k_shadow<NT, SL>, NT, SL, 0};
    else return {k_extend<true, false, true, NT, SL>, k_trace<false, true, NT, SL>, nullptr, NT, SL, 0};
}
const PassKernels& pass_kernel_table(int idx) {
    static const PassKernels t[] = {
        pass_kernels<64, 8, false>(),   pass_kernels<64, 16, false>(),  pass_kernels<64, 32, false>(),
        pass_kernels<128, 8, false>(),  pass_kernels<128, 16, false>(), pass_kernels<128, 32, false>(),
        pass_kernels<256, 8, false>(),  pass_kernels<256, 16, false>(), pass_kernels<256, 32, false>(),
        pass_kernels<512, 8, false>(),  pass_kernels<512, 16, false>(), pass_kernels<512, 32, false>(),
        pass_kernels<64, 8, true>(),    pass_kernels<64, 16, true>(),   pass_kernels<64, 32, true>(),
        pass_kernels<128, 8, true>(),   pass_kernels<128, 16, true>(),  pass_kernels<128, 32, true>(),
        pass_kernels<256, 8, true>(),   pass_kernels<256, 16, true>(),  pass_kernels<256, 32, true>(),
        pass_kernels<512, 8, true>(),   pass_kernels<512, 16, true>(),  pass_kernels<512, 32, true>(),
        {k_extend<true, true, true, 256, 16>, k_trace<true, true, 256, 16>, nullptr, 256, 16, 1},
    };
    return t[idx];
}
constexpr int kPassKernelCount = 25;
int pass_kernel_index(const TraceCfg& c) {
    if (c.layout == 1) return c.refill ? -1 : 24;
    const int a = c.nt == 64 ? 0 : c.nt == 128 ? 1 : c.nt == 256 ? 2 : c.nt == 512 ? 3 : -1;
    const int b = c.sl == 8 ? 0 : c.sl == 16 ? 1 : c.sl == 32 ? 2 : -1;
    return (a < 0 || b < 0) ? -1 : (c.refill ? 12 : 0) + 3 * a + b;
}
}  // namespace

std::vector<TraceCfg> engine_tune_space() {
    std::vector<TraceCfg> v;
    for (int nt : {64, 128, 256, 512})
        for (int sl : {8, 16, 32}) {
            for (int chunk : {64, 128, 256, 512}) v.push_back(TraceCfg{nt, sl, chunk, 0, 0});
            for (int chunk : {64, 128}) v.push_back(TraceCfg{nt, sl, chunk, 0, 1});
        }
    v.push_back(TraceCfg{256, 16, 64, 1, 0});
    return v;
}

namespace {
// Entries of a queue that holds `paths` paths or what a bounce of them appends.
uint32_t queue_entries(uint32_t paths, bool tight) {
    const Segs s = segs_for(paths, tight);
    return std::max(paths, s.nseg * s.cap);
}
// Entries of the queues of passes of up to `paths` paths, in one part or two.
uint32_t pass_entries(uint32_t paths, bool tight) {
    constexpr uint32_t kSlack = 5120;  // segments hold at most that much beyond their paths
    if (parts_for(paths, tight) == 1) return queue_entries(paths, tight);
    return paths + kMaxParts * (kSlack + kShadeBlock);
}
QueueView queue_from(QueueView q, uint32_t at) {
    q.o_tmin += at;
    q.d_tmax += at;
    q.hit += at;
    q.w_pdf += at;
    q.pix += at;
    q.rng += at;
    if (q.job) q.job += at;
    return q;
}
// Sets a pass's arguments up for one of its parts: its share of the queues,
// counters and cursors, and the stack overflow area `side` of the second one.
// `paths` is what the launches cover.  Returns what those of a part cover.
uint32_t set_part(RenderArgs& a, uint32_t paths, uint32_t parts, uint32_t part, bool tight, int2* side) {
    const uint32_t n = parts == 1 ? paths : part_begin(paths, parts, 1);
    const Segs sg = a.rng_mode == GPR_RNG_REFERENCE ? Segs{1, n} : segs_for(n, tight);
    a.parts = parts;
    a.part = part;
    a.nseg = sg.nseg;
    a.seg_cap = sg.cap;
    if (part) {
        for (QueueView& q : a.q) q = queue_from(q, queue_entries(n, tight));
        a.ctrl += 1;
        a.seg += seg_words(kMaxSegs);
        if (a.last) a.last += kMaxBounce * kLastSpread;
        a.spill = side;
    }
    return n;
}
// The second chain of a pass while it is captured: work on st between fork and
// join runs beside what is launched on the stream `fork` returns.
struct SideStream {
    hipStream_t s = nullptr;
    hipEvent_t forked = nullptr, joined = nullptr;
    int make() {
        if (s) return GPR_OK;
        if (!forked) GPR_HIP(hipEventCreateWithFlags(&forked, hipEventDisableTiming));
        if (!joined) GPR_HIP(hipEventCreateWithFlags(&joined, hipEventDisableTiming));
        GPR_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
        return GPR_OK;
    }
    int fork(hipStream_t st) {
        GPR_HIP(hipEventRecord(forked, st));
        GPR_HIP(hipStreamWaitEvent(s, forked, 0));
        return GPR_OK;
    }
    int join(hipStream_t st) {
        GPR_HIP(hipEventRecord(joined, s));
        GPR_HIP(hipStreamWaitEvent(st, joined, 0));
        return GPR_OK;
    }
    ~SideStream() {
        if (s) (void)hipStreamDestroy(s);
        if (forked) (void)hipEventDestroy(forked);
        if (joined) (void)hipEventDestroy(joined);
    }
};
// Device memory that is free.  On a nearly full device the runtime's figure can
// fall below zero and wrap.
int free_bytes(uint64_t* out) {
    size_t free = 0, total = 0;
    GPR_HIP(hipMemGetInfo(&free, &total));
    *out = free <= total ? free : 0;
    return GPR_OK;
}
uint64_t queue_bytes(uint32_t n, bool with_job) { return (uint64_t)n * (16 * 4 + 4 + 8 + (with_job ? 4 : 0)) + 8 * 256; }
int alloc_queue(DevBuf& mem, QueueView& q, uint32_t n, bool with_job) {
    GPR_TRY(mem.alloc(queue_bytes(n, with_job)));
    char* p = mem.as<char>();
    size_t off = 0;
    auto take = [&](size_t bytes) {
        off = (off + 255) & ~(size_t)255;
        char* r = p + off;
        off += bytes;
        return r;
    };
    q.o_tmin = reinterpret_cast<float4*>(take(16ull * n));
    q.d_tmax = reinterpret_cast<float4*>(take(16ull * n));
    q.hit = reinterpret_cast<float4*>(take(16ull * n));
    q.w_pdf = reinterpret_cast<float4*>(take(16ull * n));
    q.pix = reinterpret_cast<uint32_t*>(take(4ull * n));
    q.rng = reinterpret_cast<unsigned long long*>(take(8ull * n));
    q.job = with_job ? reinterpret_cast<uint32_t*>(take(4ull * n)) : nullptr;
    return GPR_OK;
}
}  // namespace

struct Engine {
    int device = 0;
    uint32_t capacity = 0, max_jobs = 0;
    DevBuf qmem[3], ctrl, seg, spill, pass, scenes;
    DevBuf terms, nterm;      // passes of several samples a job
    uint64_t term_limit = 0;  // bytes the term lists may take
    DevBuf side_spill;        // stack overflow area of a pass's second part
    bool side_grows = false;  // it is allocated on use
    SideStream side;
    QueueView q[3];
    int grid[kPassKernelCount] = {};
    hipStream_t cap_stream = nullptr;
    static constexpr int kStage = 4;
    PassBuf* h_pass[kStage] = {};
    hipEvent_t ev[kStage] = {};
    int slot = 0;
    struct GraphKey {
        uint32_t depth;
        int kidx;
        uint32_t chunk;
        uint32_t size;  // launch size class: paths rounded up to a power of two
        float4* fb;
        bool terms;     // several samples a job
        uint32_t parts;
        bool operator==(const GraphKey& o) const {
            return depth == o.depth && kidx == o.kidx && chunk == o.chunk && size == o.size && fb == o.fb &&
                   terms == o.terms && parts == o.parts;
        }
    };
    std::vector<std::pair<GraphKey, hipGraphExec_t>> graphs;
    ~Engine() {
        for (auto& g : graphs) (void)hipGraphExecDestroy(g.second);
        for (int k = 0; k < kStage; ++k) {
            if (ev[k]) (void)hipEventDestroy(ev[k]);
            if (h_pass[k]) (void)hipHostFree(h_pass[k]);
        }
        if (cap_stream) (void)hipStreamDestroy(cap_stream);
    }
};

int engine_create(int device, uint32_t capacity, uint32_t max_jobs, Engine** out) {
    if (capacity == 0 || capacity >= (1u << 30) || max_jobs == 0 || max_jobs > kMaxPassJobs)
        return fail(GPR_ERR_INVALID, "engine: capacity or job count out of range");
    GPR_HIP(hipSetDevice(device));
    Engine* e = new (std::nothrow) Engine();
    if (!e) return fail(GPR_ERR_OOM, "engine: host allocation failed");
    std::unique_ptr<Engine> guard(e);
    e->device = device;
    e->capacity = capacity;
    e->max_jobs = max_jobs;
    for (int k = 0; k < 3; ++k) GPR_TRY(alloc_queue(e->qmem[k], e->q[k], pass_entries(capacity, true), true));
    GPR_TRY(e->ctrl.alloc(kMaxParts * sizeof(Ctrl)));
    GPR_TRY(e->seg.alloc(parts_for(capacity, true) > 1 ? 8ull * kMaxParts * seg_words(kMaxSegs)
                                                       : 8ull * seg_words(segs_for(capacity, true).nseg)));
    GPR_HIP(hipMemsetAsync(e->ctrl.p, 0, kMaxParts * sizeof(Ctrl), stream()));
    GPR_TRY(e->pass.alloc(sizeof(PassBuf)));
    int cus = 0;
    GPR_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    size_t threads = 0;
    for (int k = 0; k < kPassKernelCount; ++k) {
        const PassKernels& pk = pass_kernel_table(k);
        int per_cu = 0;
        GPR_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pk.trace, pk.nt, 0));
        // Blocks of 256 threads and more: four waves a SIMD though five fit.  Batch of
        // 12 scenes / burst of 16 requests, four waves and five: 256x16 40.4 / 144 ms
        // and 42.4 / 148, but 64x8 41.5 / 151 and 40.3 / 146, 128x16 40.8 / 149 and 41.1 / 146.
        if (pk.nt >= 256) per_cu = std::min(per_cu, 1024 / pk.nt);
        // more persistent threads than queue entries would only idle
        e->grid[k] = std::max(1, std::min<int>(cus * std::max(1, per_cu), (int)div_up(capacity, pk.nt)));
        threads = std::max(threads, (size_t)e->grid[k] * pk.nt);
    }
    GPR_TRY(e->spill.alloc(threads * kStackGlobal * sizeof(int2)));
    for (int k = 0; k < Engine::kStage; ++k) {
        GPR_HIP(hipHostMalloc((void**)&e->h_pass[k], sizeof(PassBuf), hipHostMallocDefault));
        GPR_HIP(hipEventCreateWithFlags(&e->ev[k], hipEventDisableTiming));
    }
    GPR_HIP(hipStreamCreateWithFlags(&e->cap_stream, hipStreamNonBlocking));
    GPR_HIP(hipStreamSynchronize(stream()));
    *out = guard.release();
    return GPR_OK;
}

void engine_destroy(Engine* e) { delete e; }

// What counts against a caller's budget.  Counters and cursors (200 KB at most)
// do not: with them small budgets that used to be accepted would be refused.
size_t engine_device_bytes(const Engine* e) {
    return e->qmem[0].bytes + e->qmem[1].bytes + e->qmem[2].bytes + e->spill.bytes + e->pass.bytes + e->scenes.bytes;
}

int engine_set_scenes(Engine* e, const std::vector<SceneView>& views, hipStream_t st) {
    if (views.empty()) return GPR_OK;
    const size_t bytes = views.size() * sizeof(SceneView);
    if (bytes > e->scenes.bytes) {
        GPR_HIP(hipStreamSynchronize(st));
        GPR_TRY(e->scenes.alloc(bytes));
        for (auto& g : e->graphs) (void)hipGraphExecDestroy(g.second);
        e->graphs.clear();
    }
    GPR_HIP(hipMemcpyAsync(e->scenes.p, views.data(), bytes, hipMemcpyHostToDevice, st));
    GPR_HIP(hipStreamSynchronize(st));
    return GPR_OK;
}

namespace {
// Blocks of a configuration's traversal kernels whose walks may overflow to `bytes`.
uint32_t blocks_of_spill(int kidx, uint64_t bytes) {
    return (uint32_t)(bytes / (pass_kernel_table(kidx).nt * kStackGlobal * sizeof(int2)));
}
// Launch grids cover `size` paths (the pass's size class), not the capacity:
// a small pass launches small grids.
int record_pass(Engine* e, uint32_t depth, int kidx, uint32_t chunk, uint32_t size, float4* fb, bool terms,
                uint32_t parts, hipStream_t st) {
    RenderArgs pass{};
    pass.scenes = e->scenes.as<SceneView>();
    pass.pass = e->pass.as<PassBuf>();
    for (int k = 0; k < 3; ++k) pass.q[k] = e->q[k];
    pass.fb = fb;
    pass.ctrl = pass.base = e->ctrl.as<Ctrl>();
    pass.spill = e->spill.as<int2>();
    pass.seg = e->seg.as<unsigned long long>();
    pass.depth = depth;
    pass.chunk_log = 31u - (uint32_t)__builtin_clz(chunk);
    pass.rng_mode = GPR_RNG_PCG;
    if (terms) {
        pass.terms = e->terms.as<float4>();
        pass.nterm = e->nterm.as<uint8_t>();
        pass.tstride = size;
    }
    const PassKernels& pk = pass_kernel_table(kidx);
    if (parts > 1) GPR_TRY(e->side.fork(st));
    for (uint32_t part = 0; part < parts; ++part) {
        RenderArgs a = pass;
        const uint32_t n = set_part(a, size, parts, part, true, e->side_spill.as<int2>());
        const hipStream_t ps = part ? e->side.s : st;
        const uint32_t most = blocks_of_spill(kidx, part ? e->side_spill.bytes : e->spill.bytes);
        const dim3 tg(std::min({(uint32_t)e->grid[kidx], most, div_up(n, pk.nt)})), tb(pk.nt);
        hipLaunchKernelGGL(k_gen<true>, dim3(div_up(n, 256)), dim3(256), 0, ps, a);
        hipLaunchKernelGGL(pk.ext_primary, tg, tb, 0, ps, a, 0u);
        for (uint32_t b = 0; b < depth; ++b) {
            hipLaunchKernelGGL((k_shade<true, false>), dim3(shade_blocks(n, a.nseg)), dim3(kShadeBlock), 0, ps, a, b);
            if (pk.shadow) hipLaunchKernelGGL(pk.shadow, tg, tb, 0, ps, a, b);
            hipLaunchKernelGGL(pk.trace, tg, tb, 0, ps, a, b);
        }
        hipLaunchKernelGGL(k_flush<true>, dim3(std::min(1024u, div_up(n, 256))), dim3(256), 0, ps, a);
    }
    if (parts > 1) GPR_TRY(e->side.join(st));
    if (terms) hipLaunchKernelGGL(k_accum<true>, dim3(div_up(size, 256)), dim3(256), 0, st, pass);
    GPR_HIP(hipGetLastError());
    return GPR_OK;
}
}  // namespace

namespace {
// Whether a pass can run as two parts: the second one's area is there, or can
// be allocated (once, at its largest, as captured passes hold its address).
// The grid of the second part is what the area holds (record_pass): a server
// reserves it for one configuration, and others have up to 1.75 times its threads.
// 16 requests with 64-thread blocks and 8 entries 154 ms in one part, 147-151 so,
// 149-150 with an area for all of them.
bool side_ready(Engine* e, int kidx) {
    if (e->side_grows && !e->side_spill.p) {
        e->side_grows = false;
        if (e->side_spill.alloc(e->spill.bytes) != GPR_OK) (void)hipGetLastError();  // the failed allocation
    }
    return blocks_of_spill(kidx, e->side_spill.bytes) > 0 && e->side.make() == GPR_OK;
}
// Launch size class of a pass: its paths rounded up to a power of two.
uint32_t size_class(const Engine* e, uint64_t paths) {
    uint64_t size = 1u << 16;
    while (size < paths) size <<= 1;
    return (uint32_t)std::min<uint64_t>(size, e->capacity);
}
}  // namespace

int engine_run_pass(Engine* e, const EngineJob* jobs, uint32_t njobs, float4* fb, const TraceCfg& cfg,
                    hipStream_t st) {
    if (njobs == 0) return GPR_OK;
    if (njobs > e->max_jobs) return fail(GPR_ERR_INVALID, "engine: too many jobs in one pass");
    const int kidx = pass_kernel_index(cfg);
    if (kidx < 0 || cfg.chunk < 64 || cfg.chunk % 64 != 0 || cfg.chunk > 4096)
        return fail(GPR_ERR_INVALID, "engine: traversal configuration outside the tuned set");
    const int s = e->slot;
    e->slot = (s + 1) % Engine::kStage;
    GPR_HIP(hipEventSynchronize(e->ev[s]));  // the staging slot's previous upload is done
    PassBuf* h = e->h_pass[s];
    uint64_t off = 0, pixels = 0;
    uint32_t depth = 0;
    bool terms = false;
    for (uint32_t k = 0; k < njobs; ++k) {
        const EngineJob& j = jobs[k];
        if (j.npix == 0 || j.width == 0 || j.max_depth > kMaxBounce || j.log_s > kMaxLogS)
            return fail(GPR_ERR_INVALID, "engine: malformed job");
        h->jobs[k].j = j;
        h->jobs[k].path_off = (uint32_t)off;
        h->jobs[k].pix_off = (uint32_t)pixels;
        off += (uint64_t)j.npix << j.log_s;
        pixels += j.npix;
        terms = terms || j.log_s > 0;
        depth = std::max(depth, j.max_depth);
    }
    if (off > e->capacity) return fail(GPR_ERR_INVALID, "engine: pass exceeds the queue capacity");
    h->npaths = (uint32_t)off;
    h->npixels = (uint32_t)pixels;
    h->njobs = njobs;
    const uint32_t size = size_class(e, off);
    if (depth == 0) depth = 1;
    if (terms && (16ull * size * max_terms(depth) > e->terms.bytes || size > e->nterm.bytes))
        return fail(GPR_ERR_INVALID, "engine: pass exceeds its term lists");
    const size_t bytes = offsetof(PassBuf, jobs) + sizeof(PassJob) * njobs;
    GPR_HIP(hipMemcpyAsync(e->pass.p, h, bytes, hipMemcpyHostToDevice, st));
    GPR_HIP(hipEventRecord(e->ev[s], st));
    uint32_t parts = parts_for(size, true);
    if (parts > 1 && !side_ready(e, kidx)) parts = 1;
    const Engine::GraphKey key{depth, kidx, (uint32_t)cfg.chunk, size, fb, terms, parts};
    hipGraphExec_t exec = nullptr;
    for (auto& g : e->graphs)
        if (g.first == key) exec = g.second;
    if (!exec) {
        hipGraph_t graph;
        GPR_HIP(hipStreamBeginCapture(e->cap_stream, hipStreamCaptureModeThreadLocal));
        const int rc = record_pass(e, depth, kidx, (uint32_t)cfg.chunk, size, fb, terms, parts, e->cap_stream);
        const hipError_t ec = hipStreamEndCapture(e->cap_stream, &graph);
        GPR_TRY(rc);
        if (ec != hipSuccess) return fail(GPR_ERR_HIP, std::string("pass capture: ") + hipGetErrorString(ec));
        const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (ei != hipSuccess) return fail(GPR_ERR_HIP, std::string("pass instantiate: ") + hipGetErrorString(ei));
        e->graphs.push_back({key, exec});
    }
    GPR_HIP(hipGraphLaunch(exec, st));
    return GPR_OK;
}

void engine_limit_terms(Engine* e, uint64_t bytes) {
    e->term_limit = bytes;
    e->side_grows = true;
}

uint64_t engine_side_bytes(const Engine* e) {
    if (parts_for(e->capacity, true) == 1) return 0;
    const int kidx = pass_kernel_index(TraceCfg{256, 16, 64, 0, 0});
    return (uint64_t)e->grid[kidx] * pass_kernel_table(kidx).nt * kStackGlobal * sizeof(int2);
}
int engine_reserve_side(Engine* e) {
    if (e->side_spill.alloc(engine_side_bytes(e)) == GPR_OK) return GPR_OK;
    (void)hipGetLastError();  // the failed allocation
    return GPR_ERR_OOM;
}

uint64_t engine_reserve_terms(Engine* e, uint64_t bytes) {
    const uint64_t paths = std::min<uint64_t>(e->capacity, kPassPaths);  // one term count (a byte) each
    if (bytes <= 64 * paths) return 0;
    if (e->nterm.alloc(paths) != GPR_OK || e->terms.alloc(bytes - paths) != GPR_OK) {
        (void)hipGetLastError();  // the failed allocation
        e->nterm.release();
        return 0;
    }
    e->term_limit = bytes - paths;
    return bytes;
}

namespace {
// Term lists for a pass of `size` paths; false (and none as large from then on)
// where the device has no room for them.  Lists that cannot fit leave the
// present ones as they are.
int grow_terms(Engine* e, uint32_t size, uint32_t depth, hipStream_t st, bool* ok) {
    const uint64_t need = 16ull * size * max_terms(depth);
    *ok = true;
    if (need <= e->terms.bytes && size <= e->nterm.bytes) return GPR_OK;
    uint64_t free = 0;
    GPR_TRY(free_bytes(&free));
    if (need + size > free + e->terms.bytes + e->nterm.bytes) {
        e->term_limit = need - 1;
        *ok = false;
        return GPR_OK;
    }
    GPR_HIP(hipStreamSynchronize(st));  // passes in flight use the old lists
    for (size_t g = e->graphs.size(); g-- > 0;)
        if (e->graphs[g].first.terms) {
            (void)hipGraphExecDestroy(e->graphs[g].second);
            e->graphs.erase(e->graphs.begin() + g);
        }
    if (e->terms.alloc(need) != GPR_OK || e->nterm.alloc(size) != GPR_OK) {
        (void)hipGetLastError();
        e->terms.release();
        e->nterm.release();
        e->term_limit = need - 1;
        *ok = false;
    }
    return GPR_OK;
}
}  // namespace

int engine_fill_pass(Engine* e, std::vector<EngineJob>& jobs, const std::vector<uint32_t>& left, hipStream_t st) {
    uint32_t depth = 1;
    for (const EngineJob& j : jobs) depth = std::max(depth, j.max_depth);
    const uint64_t most = std::min<uint64_t>(e->capacity, kPassPaths);
    // the same power of two for every job that has as many samples left
    const auto samples = [&](size_t i, uint32_t k) {
        uint32_t s = 0;
        while (s < k && (2u << s) <= left[i]) ++s;
        return s;
    };
    for (bool ok = false; !ok;) {
        uint32_t best = 0, size = 0;
        for (uint32_t k = 1; k <= kMaxLogS; ++k) {
            uint64_t paths = 0;
            bool any = false;
            for (size_t i = 0; i < jobs.size(); ++i) {
                const uint32_t s = samples(i, k);
                any = any || s == k;
                paths += (uint64_t)jobs[i].npix << s;
            }
            if (!any || paths > most || 16ull * size_class(e, paths) * max_terms(depth) > e->term_limit) break;
            best = k;
            size = size_class(e, paths);
        }
        if (best == 0) return GPR_OK;
        GPR_TRY(grow_terms(e, size, depth, st, &ok));  // where it fails, the limit is below this pass
        for (size_t i = 0; ok && i < jobs.size(); ++i) jobs[i].log_s = samples(i, best);
    }
    return GPR_OK;
}

int engine_errors(Engine* e, hipStream_t st, uint32_t* flags) {
    uint32_t err = 0;
    GPR_HIP(hipMemcpyAsync(&err, reinterpret_cast<char*>(e->ctrl.p) + offsetof(Ctrl, error), 4,
                           hipMemcpyDeviceToHost, st));
    GPR_HIP(hipStreamSynchronize(st));
    *flags = err;
    return GPR_OK;
}

namespace {
__global__ __launch_bounds__(256) void k_pack_shade(const float* __restrict__ pos, const float* __restrict__ nrm,
                                                    const uint8_t* __restrict__ flags,
                                                    const uint32_t* __restrict__ mat,
                                                    const float* __restrict__ uv, uint32_t n,
                                                    TriShade* __restrict__ out) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const float* p = pos + 9ull * t;
    const float* q = nrm + 9ull * t;
    const uint32_t f = flags[t];
    float w[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (uv) {
#pragma unroll
        for (int k = 0; k < 6; ++k) w[k] = uv[6ull * t + k];
    }
    TriShade r;
    r.a = make_float4(p[0], p[1], p[2], p[3]);
    r.b = make_float4(p[4], p[5], p[6], p[7]);
    r.c = make_float4(p[8], q[0], q[1], q[2]);
    r.d = make_float4(q[3], q[4], q[5], q[6]);
    r.e = make_float4(q[7], q[8], __uint_as_float(f), __uint_as_float(mat[t]));
    r.f = make_float4(w[0], w[1], w[2], w[3]);
    r.g = make_float4(w[4], w[5], 0.f, 0.f);
    r.h = make_float4(0.f, 0.f, 0.f, 0.f);
    out[t] = r;
}
}  // namespace

int pack_shade(gpr_scene* s) {
    const uint32_t n = (uint32_t)s->mat.size();
    GPR_TRY(s->d_shade.alloc(std::max<size_t>(sizeof(TriShade) * n, 256)));
    if (n == 0) return GPR_OK;
    const float* uv = s->uv.empty() || s->textures.empty() ? nullptr : s->d_uv.as<float>();
    hipLaunchKernelGGL(k_pack_shade, dim3((n + 255) / 256), dim3(256), 0, stream(), s->d_pos.as<float>(),
                       s->d_nrm.as<float>(), s->d_flags.as<uint8_t>(), s->d_mat.as<uint32_t>(), uv, n,
                       s->d_shade.as<TriShade>());
    GPR_HIP(hipGetLastError());
    return GPR_OK;
}

}  // namespace gpr

using namespace gpr;

// Stack overflow area of the traversals and buffers of multi-sample passes,
// shared by the renderers of one (device, stream): gpr_render holds the lock
// until its passes have completed, so one call at a time uses them.  Freed with
// the last renderer that used them.
struct PassWork {
    std::mutex mu;
    DevBuf spill;       // kStackGlobal entries per resident lane, allocated once
    DevBuf side_spill;  // those of a pass's second part
    bool side_failed = false;
    DevBuf qmem[3], terms, nterm;
    QueueView q[3];
    uint32_t paths = 0, depth = 0;
    uint64_t gen = 0;  // of the buffers; graphs captured with older ones are dropped
    // the smallest buffers whose allocation failed, and the memory free then (these
    // buffers given back): as large ones are not tried again before more is free
    uint64_t refused = 0, refused_free = 0;
    uint64_t held() const {
        return qmem[0].bytes + qmem[1].bytes + qmem[2].bytes + terms.bytes + nterm.bytes;
    }
    void release_pass() {
        for (DevBuf* b : {&qmem[0], &qmem[1], &qmem[2], &terms, &nterm}) b->release();
        paths = depth = 0;
    }
};
namespace {
std::mutex g_work_mu;
uint64_t g_work_gen = 0;
std::map<std::pair<int, hipStream_t>, std::weak_ptr<PassWork>> g_work;

std::shared_ptr<PassWork> pass_work(int device, hipStream_t st) {
    std::lock_guard<std::mutex> lk(g_work_mu);
    for (auto it = g_work.begin(); it != g_work.end();) it = it->second.expired() ? g_work.erase(it) : std::next(it);
    std::weak_ptr<PassWork>& w = g_work[{device, st}];
    std::shared_ptr<PassWork> p = w.lock();
    if (!p) w = p = std::make_shared<PassWork>();
    return p;
}
uint64_t path_bytes(uint32_t depth) { return 3 * (16 * 4 + 4 + 8) + 16ull * max_terms(depth) + 1; }
}  // namespace

struct gpr_renderer {
    gpr_scene* scene = nullptr;
    gpr_render_opts opts{};
    uint32_t npix = 0, ntiles = 0;
    uint32_t spp_done = 0;
    DevBuf fb, ctrl, status;
    PixelReader reader;
    DevBuf seg;              // queue segment counters, then those of the last sample
    uint32_t last_nseg = 1, last_parts = 1;  // segments and parts of the last pass
    SideStream side;
    DevBuf qmem[3];
    DevBuf seeds[2];
    QueueView q[3];
    int grid_trace = 0;      // resident blocks of the traversal kernels
    uint32_t last_log_s = 0; // samples of the last pass (log2)
    std::shared_ptr<PassWork> work;  // multi-sample passes
    uint64_t work_gen = 0;           // buffers the graphs were captured with
    hipStream_t cap_stream = nullptr;
    hipGraphExec_t graph[kMaxLogS + 1] = {};  // by log2 of the samples of the pass
    SceneView baked{};  // scene view (camera included) the graphs were captured with
    SceneView accum{};  // scene view the accumulated samples were taken with
    bool reset_pending = false;  // PathTracer::m_reset: the next render starts a new accumulation
    void drop_graphs() {
        for (hipGraphExec_t& g : graph) {
            if (g) (void)hipGraphExecDestroy(g);
            g = nullptr;
        }
    }
    bool has_graph() const {
        for (hipGraphExec_t g : graph)
            if (g) return true;
        return false;
    }
    ~gpr_renderer() {
        drop_graphs();
        if (cap_stream) (void)hipStreamDestroy(cap_stream);
    }
};

namespace {
RenderArgs make_args(gpr_renderer* r, uint32_t log_s) {
    RenderArgs a{};
    a.sv = r->scene->view();
    a.fb = r->fb.as<float4>();
    a.ctrl = a.base = r->ctrl.as<Ctrl>();
    a.paths = r->npix << log_s;
    a.depth = r->opts.max_depth;
    a.log_s = log_s;
    if (log_s) {
        const PassWork& w = *r->work;
        for (int k = 0; k < 3; ++k) a.q[k] = w.q[k];
        a.terms = w.terms.as<float4>();
        a.nterm = w.nterm.as<uint8_t>();
        a.tstride = a.paths;
    } else {
        for (int k = 0; k < 3; ++k) a.q[k] = r->q[k];
        a.status = r->status.as<unsigned long long>();
        a.ntiles = r->ntiles;
    }
    a.spill = r->work->spill.as<int2>();
    a.seg = r->seg.as<unsigned long long>();
    a.last = a.seg + kMaxParts * seg_words(kMaxSegs);
    a.rng_mode = r->opts.rng_mode;
    a.chunk_log = 6;
    a.rr_start = r->opts.rr_start;
    a.seed = r->opts.seed;
    return a;
}

// Block size and LDS stack entries per lane of the single-scene renderer's
// traversal.  12 entries take 24 KB of LDS a block, room for six to a CU; the
// registers of both kernels allow five.  8 / 12 / 16 entries: 8 samples of the
// textured scene 5.03 / 4.85 / 4.88 ms, 4 of the sphere grid 16.7 / 16.7 / 17.1.
constexpr int kRenderNT = 256, kRenderSL = 12;

// Parts of a pass of 2^log_s samples.  Reference RNG mode orders its queues by
// pixel: one part.
uint32_t pass_parts(gpr_renderer* r, uint32_t log_s) {
    if (r->opts.rng_mode != GPR_RNG_PCG || parts_for(r->npix << log_s, false) == 1) return 1;
    PassWork& w = *r->work;
    if (!w.side_spill.p && !w.side_failed && w.side_spill.alloc(w.spill.bytes) != GPR_OK) {
        (void)hipGetLastError();  // the failed allocation
        w.side_failed = true;
    }
    return w.side_spill.p && r->side.make() == GPR_OK ? kMaxParts : 1;
}

// One pass of 2^log_s samples: gen -> extend(primary) -> max_depth x {shade, trace} -> flush -> accum -> finish.
int launch_pass(gpr_renderer* r, uint32_t log_s, uint32_t parts, hipStream_t st) {
    const RenderArgs pass = make_args(r, log_s);
    const bool ref = r->opts.traversal == GPR_TRAVERSAL_REF;
    constexpr int NT = kRenderNT, SL = kRenderSL;
    if (parts > 1) GPR_TRY(r->side.fork(st));
    for (uint32_t part = 0; part < parts; ++part) {
        RenderArgs a = pass;
        const uint32_t n = set_part(a, a.paths, parts, part, false, r->work->side_spill.as<int2>());
        const hipStream_t ps = part ? r->side.s : st;
        // the whole grid where the paths are few, too: they are spread thin over it
        const dim3 tg(std::min<uint32_t>(r->grid_trace, n)), tb(kRenderNT);
        hipLaunchKernelGGL(k_gen<false>, dim3(div_up(n, 256)), dim3(256), 0, ps, a);
        if (ref) hipLaunchKernelGGL((k_extend<true, true, false, NT, SL>), tg, tb, 0, ps, a, 0u);
        else hipLaunchKernelGGL((k_extend<true, false, false, NT, SL>), tg, tb, 0, ps, a, 0u);
        for (uint32_t b = 0; b < r->opts.max_depth; ++b) {
            if (a.rng_mode == GPR_RNG_REFERENCE)
                hipLaunchKernelGGL((k_shade<false, true>), dim3(div_up(n, kOrderedBlock)), dim3(kOrderedBlock), 0, ps, a, b);
            else
                hipLaunchKernelGGL((k_shade<false, false>), dim3(shade_blocks(n, a.nseg)), dim3(kShadeBlock), 0, ps, a, b);
            if (ref) hipLaunchKernelGGL((k_trace<true, false, NT, SL>), tg, tb, 0, ps, a, b);
            else hipLaunchKernelGGL((k_trace<false, false, NT, SL>), tg, tb, 0, ps, a, b);
        }
        if (a.depth) hipLaunchKernelGGL(k_flush<false>, dim3(std::min(1024u, div_up(n, 256))), dim3(256), 0, ps, a);
    }
    if (parts > 1) GPR_TRY(r->side.join(st));
    if (log_s) hipLaunchKernelGGL(k_accum<false>, dim3(div_up(r->npix, 256)), dim3(256), 0, st, pass);
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(64), 0, st, pass.base, 1u << log_s);
    GPR_HIP(hipGetLastError());
    return GPR_OK;
}

// The sample sequence captured once into a hipGraph and replayed per sample;
// captured again when the scene view (camera included) has changed.
// Every field of the view is baked into the captured graph's kernel
// arguments; gpr_scene::view() value-initialises the struct, so padding is
// zero and a byte comparison covers all of them.
bool same_view(const SceneView& a, const SceneView& b) { return std::memcmp(&a, &b, sizeof(SceneView)) == 0; }

int pass_graph(gpr_renderer* r, uint32_t log_s, uint32_t parts, hipGraphExec_t* out) {
    const SceneView now = r->scene->view();
    if (r->has_graph() && !same_view(now, r->baked)) {
        GPR_HIP(hipStreamSynchronize(stream()));
        r->drop_graphs();
    }
    hipGraphExec_t& graph = r->graph[log_s];
    if (!graph) {
        r->baked = now;
        if (!r->cap_stream) GPR_HIP(hipStreamCreateWithFlags(&r->cap_stream, hipStreamNonBlocking));
        hipGraph_t g;
        GPR_HIP(hipStreamBeginCapture(r->cap_stream, hipStreamCaptureModeThreadLocal));
        const int rc = launch_pass(r, log_s, parts, r->cap_stream);
        const hipError_t ec = hipStreamEndCapture(r->cap_stream, &g);
        GPR_TRY(rc);
        if (ec != hipSuccess) return fail(GPR_ERR_HIP, std::string("sample capture: ") + hipGetErrorString(ec));
        const hipError_t ei = hipGraphInstantiate(&graph, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (ei != hipSuccess) {
            graph = nullptr;
            return fail(GPR_ERR_HIP, std::string("sample instantiate: ") + hipGetErrorString(ei));
        }
    }
    *out = graph;
    return GPR_OK;
}
}  // namespace

namespace {
// Makes the stream's pass buffers hold `paths` paths of r's depth (w.mu held,
// no pass in flight).  Buffers that cannot fit leave the present ones as they
// are; if memory runs out all the same, nothing is kept of either.
int grow_work(gpr_renderer* r, PassWork& w, uint32_t paths) {
    if (w.paths >= paths && w.terms.bytes >= 16ull * paths * max_terms(r->opts.max_depth)) return GPR_OK;
    uint64_t free = 0;
    GPR_TRY(free_bytes(&free));
    free += w.held();
    const auto bytes = [](uint32_t n, uint32_t depth) {
        return 3 * queue_bytes(pass_entries(n, false), false) + 16ull * n * max_terms(depth) + n;
    };
    const uint32_t depth = std::max(w.depth, r->opts.max_depth);
    const uint32_t n = std::max(w.paths, paths);
    // a deeper render after a larger one: not both at once if that breaks the bound
    const bool both = n * path_bytes(depth) <= kPassBytes && bytes(n, depth) <= free;
    const uint32_t np = both ? n : paths, nd = both ? depth : r->opts.max_depth;
    const uint64_t need = bytes(np, nd);
    const bool tried = w.refused && need >= w.refused && free < w.refused_free + (64ull << 20);
    if (tried || need > free) return fail(GPR_ERR_OOM, "no device memory for a pass of several samples");
    {
        std::lock_guard<std::mutex> lk(g_work_mu);
        w.gen = ++g_work_gen;
    }
    // given back first, so that the old and the new buffers never exist together
    w.release_pass();
    int rc = GPR_OK;
    for (int k = 0; k < 3 && rc == GPR_OK; ++k) rc = alloc_queue(w.qmem[k], w.q[k], pass_entries(np, false), false);
    if (rc == GPR_OK) rc = w.terms.alloc(16ull * np * max_terms(nd));
    if (rc == GPR_OK) rc = w.nterm.alloc(np);
    if (rc != GPR_OK) {
        (void)hipGetLastError();  // the failed allocation
        w.release_pass();
        w.refused = need;
        w.refused_free = free;
        return rc;
    }
    if (need >= w.refused) w.refused = 0;
    w.paths = np;
    w.depth = nd;
    return GPR_OK;
}

// Samples (log2) of the passes that render `spp` more, and their buffers.
// Reference RNG mode keeps slot-indexed seeds from sample to sample: one
// sample a pass.  Where the buffers do not fit the device, smaller passes do.
uint32_t plan_passes(gpr_renderer* r, PassWork& w, uint32_t spp) {
    if (r->opts.rng_mode != GPR_RNG_PCG) return 0;
    uint32_t k = 0;
    while (k < kMaxLogS && (2u << k) <= spp && ((uint64_t)r->npix << (k + 1)) <= kPassPaths &&
           ((uint64_t)r->npix << (k + 1)) * path_bytes(r->opts.max_depth) <= kPassBytes)
        ++k;
    while (k > 0 && grow_work(r, w, r->npix << k) != GPR_OK) --k;
    if (k > 0 && r->work_gen != w.gen) {
        r->drop_graphs();
        r->work_gen = w.gen;
    }
    return k;
}

// Frame buffer, queues and traversal resources for the scene's current image size.
int renderer_alloc(gpr_renderer* r) {
    gpr_scene* s = r->scene;
    const uint64_t npix = (uint64_t)s->width * s->height;
    if (npix == 0 || npix >= (1ull << 31)) return fail(GPR_ERR_INVALID, "image size out of range");
    r->npix = (uint32_t)npix;
    GPR_HIP(hipSetDevice(s->device));
    GPR_TRY(r->fb.alloc(16ull * npix));
    GPR_TRY(r->ctrl.alloc(kMaxParts * sizeof(Ctrl)));
    GPR_TRY(r->seg.alloc(8ull * kMaxParts * (seg_words(kMaxSegs) + kMaxBounce * kLastSpread)));
    r->ntiles = div_up(npix, kShadeBlock);
    GPR_TRY(r->status.alloc(8ull * kMaxBounce * r->ntiles));
    for (int k = 0; k < 3; ++k) GPR_TRY(alloc_queue(r->qmem[k], r->q[k], pass_entries(r->npix, false), false));
    for (int k = 0; k < 2; ++k) {
        GPR_TRY(r->seeds[k].alloc(4ull * npix));
        GPR_HIP(hipMemsetAsync(r->seeds[k].p, 0, 4ull * npix, stream()));  // DEVICE_BUFFER allocations start zeroed (buffer.h:62)
        r->q[k].seed = r->seeds[k].as<uint32_t>();
    }
    int cus = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, s->device) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_trace<false, false, kRenderNT, kRenderSL>,
                                                     kRenderNT, 0) != hipSuccess)
        return fail(GPR_ERR_HIP, "occupancy query failed");
    r->grid_trace = std::max(1, cus * std::max(1, per_cu));
    return GPR_OK;
}
}  // namespace

extern "C" {

int gpr_renderer_create(gpr_scene* s, const gpr_render_opts* o, gpr_renderer** out) {
    if (!s || !o || !out) return fail(GPR_ERR_INVALID, "gpr_renderer_create: null argument");
    if (!s->committed) return fail(GPR_ERR_INVALID, "gpr_renderer_create: scene not committed");
    if (o->max_depth > kMaxBounce) return fail(GPR_ERR_INVALID, "max_depth above 64");
    if (o->rng_mode > GPR_RNG_PCG || o->traversal > GPR_TRAVERSAL_REF)
        return fail(GPR_ERR_INVALID, "gpr_renderer_create: unknown mode");
    gpr_renderer* r = new (std::nothrow) gpr_renderer();
    if (!r) return fail(GPR_ERR_OOM, "gpr_renderer_create: host allocation failed");
    r->scene = s;
    r->opts = *o;
    int rc = renderer_alloc(r);
    if (rc == GPR_OK) rc = gpr_renderer_reset(r);
    if (rc != GPR_OK) {
        delete r;
        return rc;
    }
    ++s->renderers;
    *out = r;
    return GPR_OK;
}

int gpr_renderer_zoom(gpr_renderer* r, float d) {
    if (!r) return fail(GPR_ERR_INVALID, "gpr_renderer_zoom: null renderer");
    float* e = r->scene->eye;
    const float* v = r->scene->dir;
    for (int k = 0; k < 3; ++k) e[k] = e[k] + v[k] * d;  // m_eye += m_dir * d
    r->reset_pending = true;
    return GPR_OK;
}

int gpr_renderer_translate(gpr_renderer* r, float x, float y) {
    if (!r) return fail(GPR_ERR_INVALID, "gpr_renderer_translate: null renderer");
    gpr_scene* s = r->scene;
    const v3 d = norm3(V(s->dir[0], s->dir[1], s->dir[2]));
    const v3 h = norm3(cross3(d, V(s->up[0], s->up[1], s->up[2])));
    const v3 vv = norm3(cross3(h, d));
    const v3 m = h * x + vv * y;
    s->eye[0] = s->eye[0] + m.x;
    s->eye[1] = s->eye[1] + m.y;
    s->eye[2] = s->eye[2] + m.z;
    r->reset_pending = true;
    return GPR_OK;
}

int gpr_renderer_rotate(gpr_renderer* r, float yaw, float pitch) {
    if (!r) return fail(GPR_ERR_INVALID, "gpr_renderer_rotate: null renderer");
    gpr_scene* s = r->scene;
    s->yaw += yaw;
    s->pitch += pitch;
    s->dir[0] = std::sin(s->yaw) * std::cos(s->pitch);
    s->dir[1] = std::sin(s->pitch);
    s->dir[2] = std::cos(s->yaw) * std::cos(s->pitch);
    r->reset_pending = true;
    return GPR_OK;
}

int gpr_renderer_resize(gpr_renderer* r, uint32_t w, uint32_t h) {
    if (!r || w == 0 || h == 0) return fail(GPR_ERR_INVALID, "gpr_renderer_resize: bad argument");
    gpr_scene* s = r->scene;
    GPR_HIP(hipStreamSynchronize(stream()));
    s->width = w;
    s->height = h;
    if (!s->cam_free) camera_raster_to_camera(w, h, s->fov, s->r2c);
    // Camera::updateAspectRation: fov.y = atan(tan(fov.x * 0.5) / aspect) * 2 (in double)
    const float aspect = (float)w / (float)h;
    s->fovy = (float)(std::atan(std::tan(s->fovx * 0.5) / aspect) * 2.0);
    r->drop_graphs();
    GPR_TRY(renderer_alloc(r));
    return gpr_renderer_reset(r);
}

int gpr_renderer_get_resolution(const gpr_renderer* r, uint32_t* w, uint32_t* h) {
    if (!r || !w || !h) return fail(GPR_ERR_INVALID, "gpr_renderer_get_resolution: null argument");
    *w = r->scene->width;
    *h = r->scene->height;
    return GPR_OK;
}

int gpr_renderer_reset(gpr_renderer* r) {
    if (!r) return fail(GPR_ERR_INVALID, "gpr_renderer_reset: null renderer");
    hipLaunchKernelGGL(k_clear_fb, dim3(div_up(r->npix, 256)), dim3(256), 0, stream(), r->fb.as<float4>(), r->npix);
    hipLaunchKernelGGL(k_set_sample, dim3(1), dim3(64), 0, stream(), r->ctrl.as<Ctrl>(), 0u);
    GPR_HIP(hipGetLastError());
    r->spp_done = 0;
    r->reset_pending = false;
    r->accum = r->scene->view();
    return GPR_OK;
}

int gpr_renderer_set_opts(gpr_renderer* r, const gpr_render_opts* o) {
    if (!r || !o) return fail(GPR_ERR_INVALID, "gpr_renderer_set_opts: null argument");
    if (o->max_depth > kMaxBounce) return fail(GPR_ERR_INVALID, "max_depth above 64");
    if (o->rng_mode > GPR_RNG_PCG || o->traversal > GPR_TRAVERSAL_REF)
        return fail(GPR_ERR_INVALID, "gpr_renderer_set_opts: unknown mode");
    if (r->has_graph()) GPR_HIP(hipStreamSynchronize(stream()));
    r->drop_graphs();  // the options are baked into them
    r->opts = *o;
    return gpr_renderer_reset(r);
}

int gpr_renderer_restore(gpr_renderer* r, const float* rgb, uint32_t spp) {
    if (!r || !rgb) return fail(GPR_ERR_INVALID, "gpr_renderer_restore: null argument");
    if (r->opts.rng_mode != GPR_RNG_PCG)
        return fail(GPR_ERR_UNSUPPORTED,
                    "gpr_renderer_restore: reference RNG mode keeps slot-indexed seeds across samples; "
                    "only PCG renders can be continued");
    std::vector<float4> tmp(r->npix);
    for (uint64_t i = 0; i < r->npix; ++i) tmp[i] = make_float4(rgb[3 * i], rgb[3 * i + 1], rgb[3 * i + 2], 0.f);
    GPR_HIP(hipMemcpyAsync(r->fb.p, tmp.data(), 16ull * r->npix, hipMemcpyHostToDevice, stream()));
    hipLaunchKernelGGL(k_set_sample, dim3(1), dim3(64), 0, stream(), r->ctrl.as<Ctrl>(), spp);
    GPR_HIP(hipGetLastError());
    GPR_HIP(hipStreamSynchronize(stream()));  // tmp is released on return
    r->spp_done = spp;
    r->reset_pending = false;
    r->accum = r->scene->view();
    return GPR_OK;
}

int gpr_render(gpr_renderer* r, uint32_t spp) {
    if (!r) return fail(GPR_ERR_INVALID, "gpr_render: null renderer");
    if (r->scene->bvh.n == 0) return fail(GPR_ERR_UNSUPPORTED, "gpr_render: scene has no triangles");
    if ((uint64_t)r->scene->width * r->scene->height != r->npix)
        return fail(GPR_ERR_INVALID, "gpr_render: the scene's image size changed; use gpr_renderer_resize");
    if (r->reset_pending) GPR_TRY(gpr_renderer_reset(r));
    // The camera lives on the scene: another renderer's zoom / translate /
    // rotate on the same scene, or a new camera set on it, changes the view
    // under this renderer.  Samples of two views must not share one sum, so
    // the accumulation starts again, as PathTracer::m_reset makes it
    // (pathtracer.cu:177-200).
    if (r->spp_done > 0 && !same_view(r->scene->view(), r->accum)) GPR_TRY(gpr_renderer_reset(r));
    hipStream_t st = stream();
    std::shared_ptr<PassWork> w = pass_work(r->scene->device, st);
    if (w != r->work) {
        r->drop_graphs();
        r->work = std::move(w);
    }
    std::lock_guard<std::mutex> lk(r->work->mu);
    GPR_TRY(r->work->spill.alloc((size_t)r->grid_trace * kRenderNT * kStackGlobal * sizeof(int2)));
    uint32_t log_s = spp > 1 ? plan_passes(r, *r->work, spp) : 0;
    for (uint32_t left = spp; left;) {
        while ((1u << log_s) > left) --log_s;
        hipGraphExec_t g = nullptr;
        const uint32_t parts = pass_parts(r, log_s);
        GPR_TRY(pass_graph(r, log_s, parts, &g));
        GPR_HIP(hipGraphLaunch(g, st));
        left -= 1u << log_s;
        RenderArgs a = make_args(r, log_s);
        set_part(a, a.paths, parts, 0, false, nullptr);
        r->last_log_s = log_s;
        r->last_parts = parts;
        r->last_nseg = a.nseg;
    }
    r->spp_done += spp;
    uint32_t err = 0;
    GPR_HIP(hipMemcpyAsync(&err, reinterpret_cast<char*>(r->ctrl.p) + offsetof(Ctrl, error), 4,
                           hipMemcpyDeviceToHost, st));
    GPR_HIP(hipStreamSynchronize(st));
    if (err) return fail(GPR_ERR_INVALID, "render error flags " + std::to_string(err));
    return GPR_OK;
}

int gpr_renderer_read(gpr_renderer* r, float* rgb, uint32_t* cnt) {
    if (!r) return fail(GPR_ERR_INVALID, "gpr_renderer_read: null renderer");
    if (cnt) std::fill_n(cnt, r->npix, r->spp_done);
    if (!rgb) {
        GPR_HIP(hipStreamSynchronize(stream()));
        return GPR_OK;
    }
    return r->reader.read(r->scene->device, r->fb.as<float4>(), r->npix, rgb, stream());
}

int gpr_renderer_queue_sizes(gpr_renderer* r, uint32_t* shadow, uint32_t* scatter, uint32_t cap) {
    if (!r) return fail(GPR_ERR_INVALID, "gpr_renderer_queue_sizes: null renderer");
    std::vector<unsigned long long> c(r->seg.bytes / 8);
    GPR_HIP(hipMemcpyAsync(c.data(), r->seg.p, r->seg.bytes, hipMemcpyDeviceToHost, stream()));
    GPR_HIP(hipStreamSynchronize(stream()));
    for (uint32_t b = 0; b < cap && b < kMaxBounce; ++b) {
        uint32_t sh = 0, sc = 0;
        // of several samples the last one alone
        const uint32_t words = r->last_log_s ? kLastSpread : r->last_nseg;
        for (uint32_t p = 0; p < r->last_parts; ++p)
            for (uint32_t k = 0; k < words; ++k) {
                const unsigned long long n =
                    r->last_log_s ? c[kMaxParts * seg_words(kMaxSegs) + (p * kMaxBounce + b) * kLastSpread + k]
                                  : c[p * seg_words(kMaxSegs) + (b * r->last_nseg + k) * seg_stride(r->last_nseg)];
                sh += (uint32_t)(n >> 32);
                sc += (uint32_t)n;
            }
        if (shadow) shadow[b] = sh;
        if (scatter) scatter[b] = sc;
    }
    return GPR_OK;
}

int gpr_renderer_free(gpr_renderer* r) {
    if (r) {
        (void)hipStreamSynchronize(stream());
        --r->scene->renderers;
        delete r;
    }
    return GPR_OK;
}

}  // extern "C"

// ---------------------------------------------------------------- PNG ----
namespace {
uint32_t crc_table[256];
bool crc_ready = false;
uint32_t crc32(const unsigned char* p, size_t n, uint32_t c = 0xffffffffu) {
    if (!crc_ready) {
        for (uint32_t i = 0; i < 256; ++i) {
            uint32_t v = i;
            for (int k = 0; k < 8; ++k) v = (v & 1) ? 0xedb88320u ^ (v >> 1) : v >> 1;
            crc_table[i] = v;
        }
        crc_ready = true;
    }
    for (size_t i = 0; i < n; ++i) c = crc_table[(c ^ p[i]) & 0xff] ^ (c >> 8);
    return c;
}
void put32(std::vector<unsigned char>& o, uint32_t v) {
    o.push_back((unsigned char)(v >> 24));
    o.push_back((unsigned char)(v >> 16));
    o.push_back((unsigned char)(v >> 8));
    o.push_back((unsigned char)v);
}
void chunk(std::vector<unsigned char>& o, const char* type, const std::vector<unsigned char>& data) {
    put32(o, (uint32_t)data.size());
    std::vector<unsigned char> td(type, type + 4);
    td.insert(td.end(), data.begin(), data.end());
    o.insert(o.end(), td.begin(), td.end());
    put32(o, crc32(td.data(), td.size()) ^ 0xffffffffu);
}
// 8-bit RGB PNG with stored (uncompressed) deflate blocks.
int write_png(const std::string& path, uint32_t w, uint32_t h, const std::vector<unsigned char>& rgb) {
    std::vector<unsigned char> raw;
    raw.reserve((3ull * w + 1) * h);
    for (uint32_t y = 0; y < h; ++y) {
        raw.push_back(0);
        raw.insert(raw.end(), rgb.begin() + 3ull * w * y, rgb.begin() + 3ull * w * (y + 1));
    }
    std::vector<unsigned char> z = {0x78, 0x01};
    size_t pos = 0;
    do {
        const size_t len = std::min<size_t>(65535, raw.size() - pos);
        z.push_back(pos + len == raw.size() ? 1 : 0);
        z.push_back((unsigned char)(len & 0xff));
        z.push_back((unsigned char)(len >> 8));
        z.push_back((unsigned char)(~len & 0xff));
        z.push_back((unsigned char)((~len >> 8) & 0xff));
        z.insert(z.end(), raw.begin() + pos, raw.begin() + pos + len);
        pos += len;
    } while (pos < raw.size());
    uint32_t s1 = 1, s2 = 0;
    for (unsigned char c : raw) {
        s1 = (s1 + c) % 65521u;
        s2 = (s2 + s1) % 65521u;
    }
    put32(z, (s2 << 16) | s1);
    std::vector<unsigned char> out = {0x89, 'P', 'N', 'G', 0x0d, 0x0a, 0x1a, 0x0a};
    std::vector<unsigned char> ihdr;
    put32(ihdr, w);
    put32(ihdr, h);
    ihdr.insert(ihdr.end(), {8, 2, 0, 0, 0});
    chunk(out, "IHDR", ihdr);
    chunk(out, "IDAT", z);
    chunk(out, "IEND", {});
    FILE* f = std::fopen(path.c_str(), "wb");
    if (!f) return fail(GPR_ERR_IO, "cannot open " + path);
    const size_t wr = std::fwrite(out.data(), 1, out.size(), f);
    std::fclose(f);
    if (wr != out.size()) return fail(GPR_ERR_IO, "short write to " + path);
    return GPR_OK;
}
// Radiance RGBE of one pixel (Ward's float2rgbe): e from the largest channel,
// mantissas scaled so that channel / 2^(e-8) fits a byte.  Non-finite or
// negative channels are written as 0.
void rgbe_of(const float* c, unsigned char* o) {
    float v[3];
    for (int k = 0; k < 3; ++k) v[k] = std::isfinite(c[k]) && c[k] > 0.f ? c[k] : 0.f;
    const float m = std::max(v[0], std::max(v[1], v[2]));
    if (m < 1e-32f) {
        o[0] = o[1] = o[2] = o[3] = 0;
        return;
    }
    int e;
    const float scale = std::frexp(m, &e) * 256.f / m;
    for (int k = 0; k < 3; ++k) o[k] = (unsigned char)std::min(255.f, v[k] * scale);
    o[3] = (unsigned char)(e + 128);
}
// Radiance .hdr, 32-bit_rle_rgbe: new-style scanlines (each component as
// literal dumps of up to 128 bytes) where the format allows them (8 <= w <
// 32768), flat pixels otherwise; `rgb` rows top first.
int write_hdr(const std::string& path, uint32_t w, uint32_t h, const std::vector<float>& rgb) {
    std::string out = "#?RADIANCE\nFORMAT=32-bit_rle_rgbe\n\n-Y " + std::to_string(h) + " +X " + std::to_string(w) + "\n";
    std::vector<unsigned char> px(4ull * w);
    for (uint32_t y = 0; y < h; ++y) {
        for (uint32_t x = 0; x < w; ++x) rgbe_of(&rgb[3 * ((uint64_t)y * w + x)], &px[4 * x]);
        if (w < 8 || w >= 32768) {
            out.append(reinterpret_cast<const char*>(px.data()), px.size());
            continue;
        }
        out += (char)2;
        out += (char)2;
        out += (char)(w >> 8);
        out += (char)(w & 0xff);
        for (int c = 0; c < 4; ++c)
            for (uint32_t x0 = 0; x0 < w; x0 += 128) {
                const uint32_t cnt = std::min<uint32_t>(128, w - x0);
                out += (char)cnt;
                for (uint32_t x = x0; x < x0 + cnt; ++x) out += (char)px[4 * x + c];
            }
    }
    FILE* f = std::fopen(path.c_str(), "wb");
    if (!f) return fail(GPR_ERR_IO, "cannot open " + path);
    const size_t wr = std::fwrite(out.data(), 1, out.size(), f);
    std::fclose(f);
    if (wr != out.size()) return fail(GPR_ERR_IO, "short write to " + path);
    return GPR_OK;
}
}  // namespace

// filter_kernel (pathtracer_kernel.h:792-810): mean, sRGB bytes, alpha from
// GammaCorrect(1); pixel i of the frame buffer to out[i] (R in the low byte).
__global__ __launch_bounds__(256) void k_resolve_rgba8(const float4* __restrict__ fb, uint32_t npix, float n,
                                                       uint32_t* __restrict__ out) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= npix) return;
    const float4 s = fb[i];
    out[i] = srgb_byte(s.x / n) | (srgb_byte(s.y / n) << 8) | (srgb_byte(s.z / n) << 16) | (srgb_byte(1.f) << 24);
}

extern "C" int gpr_renderer_resolve_rgba8(gpr_renderer* r, uint32_t* out, uint32_t flags) {
    if (!r || !out) return fail(GPR_ERR_INVALID, "gpr_renderer_resolve_rgba8: null argument");
    if (flags & ~GPR_RESOLVE_DEVICE_PTRS) return fail(GPR_ERR_INVALID, "gpr_renderer_resolve_rgba8: unknown flags");
    const float n = (float)std::max(1u, r->spp_done);
    const uint32_t grid = (uint32_t)((r->npix + 255) / 256);
    if (flags & GPR_RESOLVE_DEVICE_PTRS) {
        hipLaunchKernelGGL(k_resolve_rgba8, dim3(grid), dim3(256), 0, stream(), r->fb.as<float4>(), r->npix, n, out);
        GPR_HIP(hipGetLastError());
        return GPR_OK;
    }
    DevBuf d;
    GPR_TRY(d.alloc(4ull * r->npix));
    hipLaunchKernelGGL(k_resolve_rgba8, dim3(grid), dim3(256), 0, stream(), r->fb.as<float4>(), r->npix, n,
                       d.as<uint32_t>());
    GPR_HIP(hipGetLastError());
    GPR_HIP(hipMemcpyAsync(out, d.p, 4ull * r->npix, hipMemcpyDeviceToHost, stream()));
    GPR_HIP(hipStreamSynchronize(stream()));
    return GPR_OK;
}

extern "C" int gpr_renderer_write_png(gpr_renderer* r, const char* path) {
    if (!r || !path) return fail(GPR_ERR_INVALID, "gpr_renderer_write_png: null argument");
    const uint32_t w = r->scene->width, h = r->scene->height;
    std::vector<float> rgb(3ull * r->npix);
    GPR_TRY(gpr_renderer_read(r, rgb.data(), nullptr));
    std::vector<unsigned char> px(3ull * r->npix);
    const float n = (float)std::max(1u, r->spp_done);
    // FrameBuffer::output (framebuffer.cpp:11-26): mean, gamma, x255 + 0.5,
    // clamp, truncate; rows flipped on write (imageio.cpp:65).
    for (uint32_t y = 0; y < h; ++y)
        for (uint32_t x = 0; x < w; ++x) {
            const uint64_t src = (uint64_t)y * w + x, dst = (uint64_t)(h - 1 - y) * w + x;
            for (int c = 0; c < 3; ++c) px[3 * dst + c] = (unsigned char)srgb_byte(rgb[3 * src + c] / n);
        }
    return write_png(path, w, h, px);
}

// WriteImage (imageio.cpp:59-82) chosen by the file extension.
extern "C" int gpr_renderer_write_image(gpr_renderer* r, const char* path) {
    if (!r || !path) return fail(GPR_ERR_INVALID, "gpr_renderer_write_image: null argument");
    std::string p(path), ext;
    const size_t dot = p.find_last_of('.');
    if (dot != std::string::npos) ext = p.substr(dot);
    for (char& ch : ext) ch = (char)std::tolower((unsigned char)ch);
    if (ext == ".png") return gpr_renderer_write_png(r, path);
    if (ext != ".hdr") return fail(GPR_ERR_UNSUPPORTED, "gpr_renderer_write_image: extension must be .png or .hdr");
    const uint32_t w = r->scene->width, h = r->scene->height;
    std::vector<float> rgb(3ull * r->npix), mean(3ull * r->npix);
    GPR_TRY(gpr_renderer_read(r, rgb.data(), nullptr));
    const float n = (float)std::max(1u, r->spp_done);
    for (uint32_t y = 0; y < h; ++y)  // rows flipped on write, as for the PNG
        for (uint32_t x = 0; x < w; ++x)
            for (int c = 0; c < 3; ++c)
                mean[3 * ((uint64_t)(h - 1 - y) * w + x) + c] = rgb[3 * ((uint64_t)y * w + x) + c] / n;
    return write_hdr(path, w, h, mean);
}
