// Software BVH traversal for gfx950 (CDNA4 has no ray-tracing instructions).
//
// Persistent "while-while" traversal (Aila and Laine, "Understanding the
// Efficiency of Ray Traversal on GPUs", HPG 2009) laid out for 64-wide
// wavefronts:
//  * one wavefront per workgroup, one lane per ray; once REFILL_MIN lanes
//    have ended their rays they take new ones from the wavefront's granule
//    (one atomic per wavefront for a new granule, below), so no lane waits
//    for the slowest ray of its batch;
//  * a lane that meets a leaf waits until a share of the lanes hold one (the
//    default, LEAF_SHARE), or, with leaf postponing, until no lane can step
//    through an inner node; then each of them tests one triangle of its leaf;
//  * the traversal stack keeps its first SHORT_STACK entries in LDS, laid out
//    [entry][lane] (a wavefront's 8-byte pushes hit consecutive words, no bank
//    conflicts), and deeper entries in a per-lane global overflow area sized
//    from the tree's exact worst case; while no lane of the wavefront is that
//    deep, pushes and pops run without any overflow handling;
//  * closest-hit rays visit children nearest first; each stack entry keeps its
//    entry distance so popped subtrees beyond the current hit are skipped.
// Boxes use Ize's conservative slab test and a 1 + 2^-20 culling margin, so
// rounding never culls a triangle: the closest hit is the BVH-independent
// minimum of (t, flattened triangle index).
#pragma once

#include <hip/hip_runtime.h>

#include "../core/traverse.h"

namespace btrc {

constexpr int TRACE_BLOCK = 64;   // one wavefront per workgroup
// LDS stack entries per lane. One level's closest-hit rays: 6 KB a wavefront
// and 80 registers let 24 wavefronts share a CU (31.0 ms of traversal per
// field frame against 33.4 with 16 entries and 20 wavefronts: every step is a
// trip to memory). Visibility rays push unsorted, hence deeper stacks: 16
// entries and 20 wavefronts (12.7 against 13.9 ms). The two levels' registers
// stop at 20.
constexpr int SHORT_STACK_CLOSEST = 12, SHORT_STACK_ANY = 16, SHORT_STACK_TWO = 16;
constexpr int SHORT_STACK_MIN = 12; // what the overflow area is sized by
constexpr int short_stack(bool any, bool two)
{
    return two ? SHORT_STACK_TWO : any ? SHORT_STACK_ANY : SHORT_STACK_CLOSEST;
}
// Idle lanes that trigger a refill: 24 for one level (35.8 / 34.7 / 33.8 ms of
// closest-hit traversal per 1080p, 32 spp field frame at 12 / 16 / 24), 16 for
// two (12.35 against 12.5 ms at 24 per four-view frame)
constexpr int REFILL_MIN_ONE = 24, REFILL_MIN_TWO = 16;
// Triangle tests wait until one in LEAF_SHARE of the lanes that still trace
// holds a leaf (closest-hit rays, one level). A 1080p, 32 spp field frame takes
// 78.9 / 78.8 / 79.7 / 80.6 ms at 1 in 4 / 6 / 10 / 64, and a million incoherent
// rays 442 / 456 / 469 / 471 us; a fixed count of 16 lanes made small frames
// wait for lanes that had no ray (5.9 against 5.4 ms per 720p frame at 1 spp).
// Visibility rays lose what a test's early end saves (13.5 / 13.8 / 13.9 / 14.2
// / 15.0 ms per field frame waiting for 1 / 6 / 12 / 20 / 32 lanes), and so do
// the two levels, whose lanes inside an instance wait for those between
// instances (12.1 / 12.5 / 13.0 / 14.2 / 16.7 ms per four-view frame).
constexpr int LEAF_SHARE = 4;
// persistent grid: wavefronts per compute unit (default), and the most that
// fit of the visibility, two-level and media shadow kernels (more would hold
// back the rays handed out by workgroup index)
constexpr int TRACE_WAVES_PER_CU = 24;
constexpr int TRACE_WAVES_ANY = 20;
constexpr int TRACE_WAVES_TWO_LEVEL = 20;
constexpr int TRACE_WAVES_MEDIA = 16;
constexpr int TRACE_WAVES_PER_CU_MAX = 32;

// Device-scope atomics on one address serialise at about 11 ns each on
// MI355X (a wavefront-per-atomic microbenchmark: 65,536 atomics on one word
// take 746 us, spread over 64 words 22 us). Work counters are therefore
// striped: COUNTER_STRIPES counters, each on its own 128-byte line
// (COUNTER_STRIDE 32-bit words apart).
constexpr int COUNTER_STRIPES = 16;
constexpr int COUNTER_STRIDE = 32;
constexpr int FETCH_WORDS = COUNTER_STRIPES * COUNTER_STRIDE; // a traversal's fetch counters
constexpr int GRANULE = 64; // rays a traversal wavefront takes from a chunk counter at a time

// traversal schedules: leaves tested when reached, leaves postponed until
// every lane holds one, or the two-level (instance) structure
enum : int
{
    SCHED_EAGER = 0,
    SCHED_POSTPONE = 1,
    SCHED_TWO_LEVEL = 2,          // | SCHED_POSTPONE for postponed leaves
    SCHED_TWO_LEVEL_POSTPONE = 3,
};

// stack entry / node codes
constexpr uint32_t CODE_LEAF = 0x80000000u;   // | (count - 1) << 28 | first triangle
constexpr uint32_t CODE_INST = 0x40000000u;   // with CODE_LEAF: | instance (top-level leaf)
constexpr uint32_t CODE_DONE = 0xffffffffu;
constexpr uint32_t CODE_EXIT = 0xfffffffeu;   // stack marker: back to the top level
constexpr uint32_t MAX_LEAF_FIRST = 0x0ffffffeu;

// triangle leaves: CODE_LEAF set, CODE_INST (set in every other code with
// CODE_LEAF) not
__device__ __forceinline__ bool is_triangle_leaf(uint32_t code) { return (code >> 30) == 2u; }

// an instance of the two-level structure: the top level's leaves point here
struct TraceInstance
{
    float w2l[12];       // world_to_local rows
    uint32_t blas_root;  // node index of its geometry's tree
    uint32_t prim_base;  // flattened index of its first triangle
    uint32_t pad[2];
};

// A triangle in leaf order, one row of three vertices per axis: the
// watertight test reads the rows in its ray's axis order, so the permutation
// costs addresses instead of two selects per coordinate. 64 bytes, half a
// cache line: no record straddles two (48-byte records did, three in eight).
struct alignas(64) TraceTri
{
    float v[3][3 + 1]; // v[axis][vertex]; v[axis][3]: flattened index (two levels: primitive in geometry), as bits
    uint32_t inst;     // one level: instance
    uint32_t prim;     // primitive in its geometry
    uint32_t pad[2];
};

__host__ __device__ inline TraceTri make_trace_tri(const float *p, uint32_t index, uint32_t inst, uint32_t prim)
{
    TraceTri t;
    for(int a = 0; a < 3; ++a)
    {
        for(int k = 0; k < 3; ++k)
            t.v[a][k] = p[3 * k + a];
        t.v[a][3] = u2f(index);
    }
    t.inst = inst;
    t.prim = prim;
    t.pad[0] = t.pad[1] = 0;
    return t;
}

struct TraceScene
{
    const BvhNode4 *nodes;
    const TraceTri *tris;      // leaf order; one level: world space, two levels: local space
    const TraceInstance *inst; // two levels only
    float extent;              // largest world coordinate magnitude of the triangles
};

// per-lane global stack entries (code, entry distance) beyond the LDS part:
// [entry - SHORT_STACK][lane]
struct TraceOverflow
{
    uint2 *entry;
    int32_t lanes;   // stride between entries = lanes of the launch grid
};

struct HitRecord
{
    float t, b1, b2;
    bool hit;
    uint32_t inst;  // closest hits
    uint32_t prim;
};

// The two-level variant (TWO): node 0 roots the instance tree, whose leaves
// are instance codes; entering one pushes CODE_EXIT, moves the ray into the
// instance's local space (same parametric t) and continues at its
// geometry's tree; popping CODE_EXIT restores the world ray.
//
// Traces rays [0, n): each wavefront's first TRACE_BLOCK rays by its
// workgroup index, the rest [grid * TRACE_BLOCK, n) in granules of
// GRANULE rays dealt round robin to C = min(COUNTER_STRIPES, grid)
// chunks, chunk k's granules handed out by counter fetch[k * COUNTER_STRIDE]
// (all FETCH_WORDS words start at 0) to the wavefronts of workgroups
// b = k (mod C). Sink provides
//   uint32_t load(uint32_t base, uint32_t i, V3 &o, V3 &d, float &tmin, float &tmax)
//       (ray i of a refill that hands out rays base .. base + 63; returns
//       the key its result is stored under)
//   void store(uint32_t key, const HitRecord &h)
// ANY ends a ray at its first hit in [tmin, tmax]. POSTPONE: triangle tests
// wait until no lane can step through an inner node.
//
// Bound by the trips to memory of a node's seven 16-byte loads (VALU busy 69 %
// of the field frame's launches, 47 % of the lanes active; 80 % and 29 % when
// each lane tested its whole leaf when it met it: a tenth of the lanes reach
// a leaf at a time, and a leaf's test takes as long as the wavefront's longest).
// Per 1080p, 32 spp field frame closest-hit traversal went from 50.4 to 31.0 ms
// and visibility rays from 18.0 to 12.7: one triangle per lane and pass,
// distances by one fused multiply-add a plane, triangle rows in the ray's axis
// order, pushes and pops without overflow handling while no lane is deep, and
// every load of a step issued together.
//
// block, grid: this workgroup's index among the workgroups that trace these
// rays, and their number (a launch may hold two sets). s_stack: LDS of
// short_stack(ANY, TWO) * TRACE_BLOCK entries.
template<int TRI, bool ANY, bool POSTPONE, bool TWO, class Sink>
__device__ __forceinline__ void trace_persistent(
    const TraceScene &sc, Sink &sink, int32_t n, uint32_t *fetch, const TraceOverflow &ovf, uint32_t block, uint32_t grid,
    uint2 *s_stack)
{
    constexpr int REFILL_MIN = TWO ? REFILL_MIN_TWO : REFILL_MIN_ONE;
    constexpr int SHORT_STACK = short_stack(ANY, TWO);
    const int lane = (int)threadIdx.x;
    const int gl = (int)(block * TRACE_BLOCK + threadIdx.x);
    const uint64_t lanes_below = (1ull << lane) - 1ull;

    bool active = false;
    uint32_t ray = 0; // the sink's key of the lane's ray
    V3 o = v3s(0.0f), d = v3s(0.0f); // the world ray (two levels, Moeller-Trumbore)
    float tmin = 0.0f;
    float margin = 0.0f; // culling margin of the ray (cull_margin)
    RayBoxPre rb;
    uint32_t rows = 0; // byte offsets: of the near planes in a node, of the triangle rows (ray_rows)
    WatertightPre wt;
    MTPre mt;
    float best_t = 0.0f, best_b1 = 0.0f, best_b2 = 0.0f;
    float cull = 0.0f; // cull_distance(best_t, margin)
    uint32_t best_tri = 0xffffffffu;  // the closest hit's triangle record
    uint32_t best_inst = 0xffffffffu; // two levels: its instance
    uint32_t node = CODE_DONE;
    int32_t sp = 0;
    // Rays [0, static_span) go out as one batch of TRACE_BLOCK per wavefront
    // (workgroup b's first refill takes rays TRACE_BLOCK b + 0..63), so a
    // small launch takes no atomics. The rest go out in granules of
    // GRANULE rays: granule g belongs to chunk g % C, and chunk k's
    // counter hands its granules out in order to the wavefronts of
    // workgroups b = k (mod C). Every chunk spans the whole queue (balanced
    // work) and the granules in flight stay close together (coherent rays;
    // contiguous chunks per XCD, the dry ones helped out, left the field
    // frame's traversal as it was and slowed smaller frames by up to a
    // fifth). A wavefront keeps the rest of its granule for its next refill.
    const uint32_t static_span = grid * (uint32_t)TRACE_BLOCK;
    const uint32_t chunks = min((uint32_t)COUNTER_STRIPES, grid); // every chunk has wavefronts
    const uint32_t home = block % chunks;
    uint32_t *counter = fetch + home * COUNTER_STRIDE;
    // wavefront-uniform: reserved rays not yet handed out, whether the home
    // chunk has run dry, and whether no ray is left for this wavefront
    uint32_t res_lo = min((uint32_t)n, block * (uint32_t)TRACE_BLOCK);
    uint32_t res_hi = min((uint32_t)n, res_lo + (uint32_t)TRACE_BLOCK);
    bool dry = static_span >= (uint32_t)n;
    bool exhausted = dry && res_lo == res_hi;
    uint32_t cur_inst = 0xffffffffu, cur_base = 0; // two levels: the instance being traversed

    auto set_ray = [&](V3 ro, V3 rd) {
        rb = raybox_pre(ro, rd);
        // hi_x sits 16 bytes after lo_x, and so on: bits 4, 12, 20 pick the
        // far one; bits 5-6, 13-14, 21-22 hold the watertight test's axes
        rows = (rb.neg_x ? 1u << 4 : 0u) | (rb.neg_y ? 1u << 12 : 0u) | (rb.neg_z ? 1u << 20 : 0u);
        if(TRI == TRI_WATERTIGHT)
        {
            wt = watertight_pre(ro, rd);
            rows |= (uint32_t)wt.kx << 5 | (uint32_t)wt.ky << 13 | (uint32_t)wt.kz << 21;
        }
        else
            mt = mt_pre(ro, rd);
    };

    // a push or pop of any depth
    auto push_deep = [&](uint32_t code, float t) {
        const uint2 e = make_uint2(code, __float_as_uint(t));
        if(sp < SHORT_STACK)
            s_stack[sp * TRACE_BLOCK + lane] = e;
        else
            ovf.entry[(size_t)(sp - SHORT_STACK) * ovf.lanes + gl] = e;
        ++sp;
    };
    // next entry whose subtree may still hold a closer hit, or CODE_DONE
    auto pop = [&]() -> uint32_t {
        if(!__any(sp > SHORT_STACK))
        {
            while(sp > 0)
            {
                --sp;
                const uint2 e = s_stack[sp * TRACE_BLOCK + lane];
                if(__uint_as_float(e.y) <= cull)
                    return e.x;
            }
            return CODE_DONE;
        }
        while(sp > 0)
        {
            --sp;
            uint2 e;
            if(sp < SHORT_STACK)
            {
                e = s_stack[sp * TRACE_BLOCK + lane];
                asm volatile("" : "+v"(e.x), "+v"(e.y)); // keeps the two loads apart: no flat load of either address
            }
            else
                e = ovf.entry[(size_t)(sp - SHORT_STACK) * ovf.lanes + gl];
            if(__uint_as_float(e.y) <= cull)
                return e.x;
        }
        return CODE_DONE;
    };

    for(;;)
    {
        // ---- hand new rays to idle lanes
        const uint64_t idle = __ballot(!active);
        const int nidle = (int)__popcll(idle);
        if(nidle >= REFILL_MIN && !exhausted)
        {
            // first the rest of the reserved granule, then, for lanes still
            // idle, the home chunk's next granule (every lane runs this
            // loop, so lane 0 takes it for the wavefront)
            const uint32_t base_a = res_lo;
            const uint32_t take_a = min((uint32_t)nidle, res_hi - res_lo);
            res_lo += take_a;
            uint32_t base_b = 0, take_b = 0;
            if(take_a < (uint32_t)nidle && !dry)
            {
                uint32_t g = 0;
                if(lane == 0)
                    g = atomicAdd(counter, 1u);
                g = __builtin_amdgcn_readfirstlane(g);
                const uint64_t lo = (uint64_t)static_span + ((uint64_t)g * chunks + home) * GRANULE;
                if(lo < (uint64_t)n)
                {
                    res_lo = (uint32_t)lo;
                    res_hi = min((uint32_t)n, res_lo + (uint32_t)GRANULE);
                    base_b = res_lo;
                    take_b = min((uint32_t)nidle - take_a, res_hi - res_lo);
                    res_lo += take_b;
                }
                else
                    dry = true;
            }
            exhausted = dry && res_lo == res_hi;
            if(!active)
            {
                // idle lane number `rank` takes ray base_a + rank, or ray
                // base_b + rank - take_a of the new granule
                const uint32_t rank = (uint32_t)__popcll(idle & lanes_below);
                bool got = false;
                float tmax = 0.0f;
                if(take_a > 0 && rank < take_a)
                {
                    ray = sink.load(base_a, base_a + rank, o, d, tmin, tmax);
                    got = true;
                }
                if(take_b > 0 && rank >= take_a && rank < take_a + take_b)
                {
                    ray = sink.load(base_b, base_b + (rank - take_a), o, d, tmin, tmax);
                    got = true;
                }
                if(got)
                {
                    set_ray(o, d);
                    margin = cull_margin(sc.extent, o);
                    cur_inst = 0xffffffffu;
                    best_t = tmax;
                    cull = cull_distance(tmax, margin);
                    best_b1 = best_b2 = 0.0f;
                    best_tri = 0xffffffffu;
                    node = 0;
                    sp = 0;
                    active = true;
                }
            }
        }
        if(!__any(active))
            break;

        // ---- step until enough lanes have finished, or all of them have
        for(;;)
        {
            const uint64_t leaves = __builtin_amdgcn_ballot_w64(active && is_triangle_leaf(node));
            const uint64_t inner = __builtin_amdgcn_ballot_w64(active && node != CODE_DONE && !is_triangle_leaf(node));
            if((leaves | inner) == 0)
                break;
            if(!exhausted && (int)__popcll(~(leaves | inner)) >= REFILL_MIN)
                break; // enough lanes to refill

            // ---- one triangle of every leaf
            const bool enough = ANY || TWO ? leaves != 0
                                           : LEAF_SHARE * (int)__popcll(leaves) >= (int)__popcll(leaves | inner);
            if(inner == 0 || (!POSTPONE && enough))
            {
                if(active && is_triangle_leaf(node))
                {
                    const uint32_t k = node & 0x0fffffffu;
                    // records are 64-byte aligned: a row's offset is or-ed in
                    const uintptr_t tb = reinterpret_cast<uintptr_t>(sc.tris + k);
                    float t, u, v;
                    uint32_t id;
                    bool ok;
                    if(TRI == TRI_WATERTIGHT)
                    {
                        const float4 rx = *reinterpret_cast<const float4 *>(tb | ((rows >> 1) & 0x30u));
                        const float4 ry = *reinterpret_cast<const float4 *>(tb | ((rows >> 9) & 0x30u));
                        const float4 rz = *reinterpret_cast<const float4 *>(tb | ((rows >> 17) & 0x30u));
                        id = __float_as_uint(rx.w);
                        ok = watertight_hit(wt, v3(rx.x, rx.y, rx.z), v3(ry.x, ry.y, ry.z), v3(rz.x, rz.y, rz.z), tmin,
                                            best_t, &t, &u, &v);
                    }
                    else
                    {
                        const float4 rx = *reinterpret_cast<const float4 *>(tb);
                        const float4 ry = *reinterpret_cast<const float4 *>(tb | 16);
                        const float4 rz = *reinterpret_cast<const float4 *>(tb | 32);
                        id = __float_as_uint(rx.w);
                        ok = mt_hit(mt, v3(rx.x, ry.x, rz.x), v3(rx.y, ry.y, rz.y), v3(rx.z, ry.z, rz.z), tmin, best_t,
                                    &t, &u, &v);
                    }
                    // t <= best_t here; equal distances go to the lower
                    // flattened index, looked up only then
                    if(!ANY && ok && t == best_t && best_tri != 0xffffffffu)
                    {
                        const uint32_t gid = TWO ? cur_base + id : id;
                        const uint32_t other = __float_as_uint(sc.tris[best_tri].v[0][3]);
                        ok = gid < (TWO ? sc.inst[best_inst].prim_base + other : other);
                    }
                    if(ok)
                    {
                        best_t = t;
                        cull = cull_distance(t, margin);
                        best_b1 = u;
                        best_b2 = v;
                        best_tri = k;
                        best_inst = cur_inst;
                    }
                    if(ANY && ok)
                        node = CODE_DONE;
                    else if(((node >> 28) & 3u) != 0)
                        node = node - (1u << 28) + 1u; // the leaf's next triangle
                    else
                        node = pop();
                }
            }

            // ---- inner nodes
            if(active && node != CODE_DONE && !is_triangle_leaf(node))
            {
                if(TWO && node == CODE_EXIT)
                {
                    set_ray(o, d); // back to the world ray
                    cur_inst = 0xffffffffu;
                    node = pop();
                }
                else if(TWO && (node & CODE_LEAF))
                {
                    // enter an instance: world -> local, continue in its tree
                    const TraceInstance &ti = sc.inst[node & 0x0fffffffu];
                    push_deep(CODE_EXIT, -INFINITY);
                    const float *r = ti.w2l;
                    const V3 lo = v3(r[0] * o.x + r[1] * o.y + r[2] * o.z + r[3],
                                     r[4] * o.x + r[5] * o.y + r[6] * o.z + r[7],
                                     r[8] * o.x + r[9] * o.y + r[10] * o.z + r[11]);
                    const V3 ld = v3(r[0] * d.x + r[1] * d.y + r[2] * d.z,
                                     r[4] * d.x + r[5] * d.y + r[6] * d.z,
                                     r[8] * d.x + r[9] * d.y + r[10] * d.z);
                    set_ray(lo, ld);
                    cur_inst = node & 0x0fffffffu;
                    cur_base = ti.prim_base;
                    node = ti.blas_root;
                }
                else
                {
                    // the node stores lo then hi (16 bytes each) per axis: the
                    // near and far planes are picked by address from the
                    // ray's direction signs, not by selects after the load
                    const char *nb = reinterpret_cast<const char *>(sc.nodes);
                    const uint32_t off = node * (uint32_t)sizeof(BvhNode4);
                    uint4 code = *reinterpret_cast<const uint4 *>(nb + (off + 96u));
                    const uint32_t at_x = off | (rows & 16u), at_y = off | ((rows >> 8) & 16u), at_z = off | ((rows >> 16) & 16u);
                    const float4 nxv = *reinterpret_cast<const float4 *>(nb + at_x);
                    const float4 fxv = *reinterpret_cast<const float4 *>(nb + (at_x ^ 16u));
                    const float4 nyv = *reinterpret_cast<const float4 *>(nb + at_y + 32u);
                    const float4 fyv = *reinterpret_cast<const float4 *>(nb + (at_y ^ 16u) + 32u);
                    const float4 nzv = *reinterpret_cast<const float4 *>(nb + at_z + 64u);
                    const float4 fzv = *reinterpret_cast<const float4 *>(nb + (at_z ^ 16u) + 64u);
                    // the codes arrive with the boxes: without this the first
                    // one's load moves behind its box test, a second trip to
                    // memory in every step
                    asm volatile("" : "+v"(code.x), "+v"(code.y), "+v"(code.z), "+v"(code.w));
                    const float bnx[4] = { nxv.x, nxv.y, nxv.z, nxv.w };
                    const float bfx[4] = { fxv.x, fxv.y, fxv.z, fxv.w };
                    const float bny[4] = { nyv.x, nyv.y, nyv.z, nyv.w };
                    const float bfy[4] = { fyv.x, fyv.y, fyv.z, fyv.w };
                    const float bnz[4] = { nzv.x, nzv.y, nzv.z, nzv.w };
                    const float bfz[4] = { fzv.x, fzv.y, fzv.z, fzv.w };
                    const uint32_t cc[4] = { code.x, code.y, code.z, code.w };
                    float k[4];
                    uint32_t c[4];
#pragma unroll
                    for(int j = 0; j < 4; ++j)
                    {
                        float te;
                        const bool hit = raybox_nf(rb, bnx[j], bfx[j], bny[j], bfy[j], bnz[j], bfz[j],
                                                   tmin, cull, &te);
                        k[j] = hit ? te : INFINITY;
                        c[j] = hit ? cc[j] : CODE_DONE;
                    }
#define BTRC_CSWAP(a, b)                                                  \
                    if(k[b] < k[a])                                       \
                    {                                                     \
                        const float tk = k[a]; k[a] = k[b]; k[b] = tk;    \
                        const uint32_t tc = c[a]; c[a] = c[b]; c[b] = tc; \
                    }
                    if(ANY)
                    {
                        // any order will do: the first child that is hit
                        // goes next (13.0 against 13.5 ms of visibility rays
                        // per field frame with the nearest first)
                        if(c[0] == CODE_DONE) { c[0] = c[1]; c[1] = CODE_DONE; }
                        if(c[0] == CODE_DONE) { c[0] = c[2]; c[2] = CODE_DONE; }
                        if(c[0] == CODE_DONE) { c[0] = c[3]; c[3] = CODE_DONE; }
                    }
                    else
                    {
                        BTRC_CSWAP(0, 1)
                        BTRC_CSWAP(2, 3)
                        BTRC_CSWAP(0, 2)
                        BTRC_CSWAP(1, 3)
                        BTRC_CSWAP(1, 2)
                    }
#undef BTRC_CSWAP
                    if(!__any(sp > SHORT_STACK - 3))
                    {
                        // farthest first; an entry that is no child is
                        // overwritten by the next one or stays above the top
                        uint2 *top = s_stack + sp * TRACE_BLOCK + lane;
                        *top = make_uint2(c[3], __float_as_uint(k[3]));
                        top += c[3] != CODE_DONE ? TRACE_BLOCK : 0;
                        *top = make_uint2(c[2], __float_as_uint(k[2]));
                        top += c[2] != CODE_DONE ? TRACE_BLOCK : 0;
                        *top = make_uint2(c[1], __float_as_uint(k[1]));
                        sp += (c[3] != CODE_DONE ? 1 : 0) + (c[2] != CODE_DONE ? 1 : 0) + (c[1] != CODE_DONE ? 1 : 0);
                    }
                    else
                    {
                        if(c[3] != CODE_DONE) push_deep(c[3], k[3]);
                        if(c[2] != CODE_DONE) push_deep(c[2], k[2]);
                        if(c[1] != CODE_DONE) push_deep(c[1], k[1]);
                    }
                    node = c[0];
                    if(node == CODE_DONE)
                        node = pop();
                }
            }
        }

        // ---- finished rays leave their result
        if(active && node == CODE_DONE)
        {
            HitRecord h;
            h.t = best_t;
            h.b1 = best_b1;
            h.b2 = best_b2;
            h.hit = best_tri != 0xffffffffu;
            h.inst = h.prim = 0xffffffffu;
            if(!ANY && h.hit)
            {
                h.inst = TWO ? best_inst : sc.tris[best_tri].inst;
                h.prim = sc.tris[best_tri].prim;
            }
            sink.store(ray, h);
            active = false;
        }
    }
}

} // namespace btrc
