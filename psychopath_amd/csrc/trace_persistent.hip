// Persistent BVH4 traversal for gfx950 with per-lane ray refill.
//
// Same traversal as trace.hip (each ray walks the reference's depth-first
// order, src/accel/bvh4.rs:101-184, with the same box and triangle tests),
// reorganised for throughput on incoherent rays:
//   * one wave64 per workgroup, launched only as many waves as the chip holds
//     at once; each wave starts on its share of the rays and then keeps
//     taking chunks from a counter (one per range of rays);
//   * lanes whose ray finished are refilled in bulk once at least
//     `refill_min` lanes of the wave are idle, from the wave's chunk (an
//     atomic only when the chunk is used up), the new rays spread over the
//     idle lanes by a ballot prefix count;
//   * the traversal is "while-while": lanes descend internal nodes (popping
//     past dead ends) until the whole wave stands on leaves, then run the
//     leaf tests together;
//   * kernels are specialised on whether the scene has instance transforms
//     (XF), time-sampled bounds or vertices (MOTION) and nested assemblies
//     (NESTED: each assembly's own instance BVH walked in its space, as
//     trace_assembly recurses, tracer.rs:87-150), so the common static case
//     keeps no transform, lerp or nesting state in registers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "layout.h"
#include "psymath.h"
#include "trace.h"
#include "trace_device.h"

namespace psy {

namespace {

constexpr int WAVE = 64;
// Most rays a wave takes from a counter at once.  Larger chunks
// spread the rays in flight over a wider stretch of the queue: on queues in
// pixel order (a renderer's camera and bounce rays) that costs coherence, 4%
// on the large instanced scene at 512, while 64 leaves the counters contended
// on small scenes.
constexpr uint32_t CHUNK_MAX = 256;

// The rays are dealt to TRACE_RANGES ranges in blocks of RANGE_BLOCK rays,
// round robin, and wave w starts on range w % TRACE_RANGES, on a share that
// needs no counter.  One counter for all rays cost its waves their turn on
// one address, about 12 ns each: 49 us for a launch without rays, while a
// launch with few ran them 64 to a wave on a corner of the chip.  4,096 rays
// on the 65,536-triangle sphere: 174 -> 122 us; the Cornell box at 64x64, 4
// spp: 1.27 -> 0.75 ms; the large scene at full HD, whose later bounces are
// small launches: 15.1 -> 12.5 ms.  Blocks of 512 rays time the same or 1-2%
// more and of 4,096 up to 9% more (coherent rays: less balance, no more
// locality).  Ray k of range x:
constexpr uint32_t RANGE_BITS = 6;
constexpr uint32_t RANGE_BLOCK = 1u << RANGE_BITS;
__device__ __forceinline__ uint32_t range_ray(uint32_t x, uint32_t k) {
    return (((k >> RANGE_BITS) * TRACE_RANGES + x) << RANGE_BITS) + (k & (RANGE_BLOCK - 1u));
}
// Rays of range x; range 0 is never the shorter.
__host__ __device__ __forceinline__ uint32_t range_count(uint32_t n, uint32_t x) {
    const uint32_t round = RANGE_BLOCK * TRACE_RANGES, rest = n % round, before = x * RANGE_BLOCK;
    const uint32_t part = rest < before ? 0u : rest - before;
    return (n / round) * RANGE_BLOCK + (part < RANGE_BLOCK ? part : RANGE_BLOCK);
}
// Rays of its range each wave starts on without asking a counter: all of
// them where that is at most one ray per lane, spread evenly over the waves;
// else half of an even share, and the rest comes from the counters.
__host__ __device__ __forceinline__ uint32_t first_rays(uint32_t n, uint32_t waves) {
    const uint32_t per_range = waves / TRACE_RANGES;
    const uint32_t share = (range_count(n, 0) + per_range - 1u) / per_range;
    if (share <= (uint32_t)WAVE) return share;
    const uint32_t half = share / 2u;
    return half < (uint32_t)WAVE ? (uint32_t)WAVE : half < CHUNK_MAX ? half : CHUNK_MAX;
}

// Short stack: the newest entries of each lane live in an LDS ring of RING
// entries (one column per lane, stride WAVE); a node step first moves the
// oldest entries to a private overflow array until three fit, and they come
// back only when the stack unwinds to them, so the pushes and pops of the
// hot path touch LDS only and need no bounds test of their own.  `sp` and
// `bot` count entries in units of ENTRY, the bytes between two entries of a
// column; entries [0, bot) are in the overflow array.  Macros keep them in
// registers (a struct holding the array would live in private memory as a
// whole).
constexpr uint32_t ENTRY = WAVE * sizeof(uint32_t);
#define SSTACK_AT(at) (*reinterpret_cast<uint32_t*>(lds_bytes + (((at) & (RING * ENTRY - ENTRY)) | lane4)))
#define SSTACK_MAKE_ROOM(k)                             \
    while (sp - bot > (RING - (k)) * ENTRY) {           \
        spill[bot / ENTRY] = SSTACK_AT(bot);            \
        bot += ENTRY;                                   \
    }
#define SSTACK_POP(out)                                 \
    do {                                                \
        sp -= ENTRY;                                    \
        if (sp < bot) {                                 \
            bot = sp;                                   \
            (out) = spill[sp / ENTRY];                  \
        } else {                                        \
            (out) = SSTACK_AT(sp);                      \
        }                                               \
    } while (0)

// Node parts a static descent step reads: the six box rows and the child
// references (the last 16 bytes are not needed, layout.h).
constexpr uint32_t NODE_PARTS = 7;

// The local ray of an assembly level: the lerped composed transforms into
// the assembly applied to the world ray, or the identity at the root
// (update_local, tracer.rs:65-70, 101-109, 131-148).
__device__ __forceinline__ void level_local_ray(const TraceArgs& a, const GpuGroup& g, float time, V3 o, V3 d, V3& lo,
                                                V3& di) {
    Xf x = xf_identity();
    if (g.xf_count > 0) {
        uint32_t i1;
        float a2;
        if (!lerp_slice_pos(g.xf_count, time, i1, a2)) x = load_xf(a.xforms + g.xf_start + i1);
        else x = xf_lerp(load_xf(a.xforms + g.xf_start + i1), load_xf(a.xforms + g.xf_start + i1 + 1), a2);
    }
    lo = xf_point(x, o);
    const V3 ld = xf_vector(x, d);
    di = v3(1.0f / ld.x, 1.0f / ld.y, 1.0f / ld.z);
}

// RING: LDS stack entries per lane, a power of two.  BIG: the node array is
// longer than 4 GB, so node addresses take 64-bit offsets.  DIRECT: the scene
// is one mesh instance without a transform (its instance BVH is that leaf).
template <bool COUNT, bool XF, bool MOTION, uint32_t RING, int MIN_WAVES, bool COOP, bool NESTED, bool BIG, bool DIRECT>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(MIN_WAVES)))
void trace_persistent_kernel(TraceArgs a, unsigned int* work, uint32_t refill_min, uint32_t leaf_min) {
    __shared__ uint32_t lds_stack[RING * WAVE];
    // COOP: the nodes the wave's lanes stand on are fetched by the wave
    // together, consecutive lanes loading consecutive 16-byte parts of one
    // node (one cache line per node instead of one tag lookup per lane and
    // part), staged here and read back by their lanes.
    __shared__ uint4 lds_nodes[COOP ? WAVE * NODE_PARTS : 1];
    __shared__ uint32_t lds_slot[COOP ? WAVE : 1];
    const int lane = threadIdx.x;
    const uint32_t lane4 = 4u * (uint32_t)lane;
    char* const lds_bytes = reinterpret_cast<char*>(lds_stack);
    uint32_t spill[TRACE_STACK_CAPACITY];
    uint32_t sp = 0, bot = 0;

    // Rays [0, n1) stand at their own index, [n1, n) are the second set's.
    const uint32_t n1 = a.n_dev ? *a.n_dev : (uint32_t)a.n;
    const uint32_t n = n1 + (a.n2_dev ? *a.n2_dev : 0u);
    if (blockIdx.x == 0) {
        if (a.work_next && lane < (int)TRACE_RANGES) a.work_next[lane * TRACE_RANGE_WORDS] = 0u;
        if (a.clear_run && lane < (int)a.clear_run_n) a.clear_run[lane] = 0u;
        if (lane == 0) {
            if (a.clear0) *a.clear0 = 0u;
            if (a.clear1) *a.clear1 = 0u;
            if (a.tally) atomicAdd(a.tally, (unsigned long long)n);
        }
    }
    // A scene that is one untransformed instance needs no walk to it: its rays
    // start on the mesh's root.  That saves every ray a leaf round with two
    // dependent loads and is worth the two registers (98 instead of 96, so
    // 16 waves per CU instead of 20): 16.7M incoherent rays on the
    // 1M-triangle sphere 3.39 -> 3.24 ms, 4.0M shadow rays 0.943 -> 0.895.  A
    // build of its own, so that other static scenes keep their waves: 4.2M
    // rays on the sphere cut into 16 meshes take 1.51 ms, and took 1.64 where
    // one build chose at run time.
    GpuInstance only{};
    GpuMesh only_mesh{};
    if (DIRECT) {
        only = a.instances[(a.top_root & ~REF_LEAF) >> 2];
        only_mesh = a.meshes[only.mesh];
    }
    const Xf ident = xf_identity();

    // Per-lane ray state.
    bool has = false;
    uint32_t ray = 0;
    V3 o{}, d{};
    float time = 0.0f, tmax = 0.0f;
    bool occl = false;
    TriPre pre{};
    V3 lo{}, di{};
    // From the local ray: where on each axis the plane it meets first stands
    // in a node (0 or 16 bytes on), the split axes it runs down as bits of
    // REF_AXIS_MASK, and whether slab_finite serves it.
    uint32_t near_x = 0, near_y = 0, near_z = 0, down = 0;
    bool finite = false;
    auto local_ray_set = [&]() {
        near_x = di.x < 0.0f ? 16u : 0u;
        near_y = di.y < 0.0f ? 16u : 0u;
        near_z = di.z < 0.0f ? 16u : 0u;
        down = octant_of(di) << REF_AXIS_SHIFT;
        finite = !a.odd_boxes && !(tmax != tmax) && finite_ray(lo, di);
    };
    uint32_t cur = REF_EMPTY;
    bool in_inst = false;
    uint32_t inst_base = 0;
    bool has_space = false;
    Xf space;
    uint32_t inst_id = PSY_NONE;
    uint32_t grp = 0, gbase = 0;  // NESTED: the current assembly path and its first instance record
    uint64_t tri_base = 0;
    uint32_t tri_stride = sizeof(GpuTriStatic), tri_samples = 1;
    uint8_t kind = PSY_HIT_MISS;
    float ht = 0.0f, hb0 = 0.0f, hb1 = 0.0f, hb2 = 0.0f;
    uint32_t hprim = PSY_NONE, hinst = PSY_NONE;
    uint64_t c_nodes = 0, c_mnodes = 0, c_tris = 0, c_mtris = 0, c_inst = 0;
    // The wave's chunk: rays [next, end) of range rx taken and not yet handed
    // to a lane.  Rays below `dealt` of every range are the waves' first
    // chunks; the counter of a range counts on from there.  `seen`: where
    // rx's counter stood when last looked at; `drained`: every range's rays
    // are taken.
    const uint32_t per_range = gridDim.x / TRACE_RANGES;
    const uint32_t first = first_rays(n, gridDim.x);
    const uint32_t dealt = first * per_range;
    uint32_t rx = blockIdx.x % TRACE_RANGES, seen = 0;
    uint32_t next = min((blockIdx.x / TRACE_RANGES) * first, range_count(n, rx));
    uint32_t end = min(next + first, range_count(n, rx));
    bool drained = dealt >= range_count(n, 0);
    bool exhausted = drained && next == end;

    for (;;) {
        // ---- refill idle lanes ------------------------------------------
        // Idle lanes take the rest of the wave's chunk first; when it is
        // used up one atomic fetches another, sized by guided
        // self-scheduling (the range's remaining rays over 2x its waves, at
        // most CHUNK_MAX), so the counters see few atomics while the last
        // rays still spread over all waves.  A wave whose range is used up
        // goes on with the next one that is not.
        const uint64_t idle = __ballot(!has);
        if (!exhausted && (uint32_t)__popcll(idle) >= refill_min) {
            const uint32_t want = (uint32_t)__popcll(idle);
            while (next == end && !drained) {
                const uint32_t count = range_count(n, rx);
                const uint32_t left = count > dealt + seen ? count - dealt - seen : 0u;
                if (left != 0u) {
                    const uint32_t take = max(want, min(left / (2u * per_range), (uint32_t)CHUNK_MAX));
                    uint32_t at = 0;
                    if (lane == 0) at = atomicAdd(work + rx * TRACE_RANGE_WORDS, take);
                    at = __builtin_amdgcn_readfirstlane(at);
                    seen = at + take;
                    next = min(dealt + at, count);
                    end = min(dealt + at + take, count);
                } else {
                    uint32_t at = 0;
                    bool open = false;
                    if (lane < (int)TRACE_RANGES) {
                        at = __hip_atomic_load(work + lane * TRACE_RANGE_WORDS, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
                        open = dealt + at < range_count(n, (uint32_t)lane);
                    }
                    const uint32_t m = (uint32_t)__ballot(open);
                    drained = m == 0u;
                    // the first open range after rx, round robin
                    const uint32_t turned = (m | (m << TRACE_RANGES)) >> (rx + 1u);
                    if (!drained) rx = (rx + (uint32_t)__ffs(turned)) % TRACE_RANGES;
                    seen = (uint32_t)__shfl((int)at, (int)rx);
                }
            }
            const uint32_t avail = end - next;
            if (!has) {
                const uint32_t rank = (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
                if (rank < avail) {
                    has = true;
                    ray = range_ray(rx, next + rank);
                    const bool second = ray >= n1;
                    if (second) ray = ray - n1 + a.n2_at;
                    o = v3(a.ox[ray], a.oy[ray], a.oz[ray]);
                    d = v3(a.dx[ray], a.dy[ray], a.dz[ray]);
                    time = MOTION || XF ? a.time[ray] : 0.0f;
                    tmax = a.max_t[ray];
                    occl = second || a.all_occlusion != 0 || (a.flags != nullptr && (a.flags[ray] & 1u) != 0);
                    if (second) ray = a.n2_out[ray];  // (from here on only the result's place)
                    // Top-level local ray: update_local with the identity
                    // (tracer.rs:65-70).
                    lo = xf_point(ident, o);
                    V3 ld = xf_vector(ident, d);
                    di = v3(1.0f / ld.x, 1.0f / ld.y, 1.0f / ld.z);
                    local_ray_set();
                    pre = tri_precompute(d);
                    cur = a.top_root;
                    sp = 0;
                    bot = 0;
                    in_inst = false;
                    if (DIRECT) {
                        if (COUNT) c_inst++;
                        cur = only_mesh.root;
                        in_inst = true;
                        inst_base = 0;
                        inst_id = only.id;
                        tri_base = only_mesh.tri_offset;
                        if (MOTION) {
                            tri_stride = only_mesh.tri_stride;
                            tri_samples = only_mesh.time_samples;
                        }
                    }
                    grp = 0;
                    gbase = 0;
                    kind = PSY_HIT_MISS;
                }
            }
            next += min(want, avail);
            exhausted = drained && next == end;
        }
        if (__ballot(has) == 0) {
            if (exhausted) break;
            continue;
        }
        if (!has) continue;

        // ---- descend internal nodes ---------------------------------------
        // leaf_min 0: each lane descends until it stands on a leaf or on a
        // dead end (a node whose children all miss), which pops after the
        // leaf round.  leaf_min 1..64: dead ends pop inside the loop, so the
        // lane keeps working while others descend, and the loop runs while
        // some lane stands on an internal node and fewer than `leaf_min`
        // lanes wait (at a leaf, or at the end of their level: the
        // instance's subtree or the whole stack); lanes still on internal
        // nodes then carry on after the leaf round.  Every lane takes its own
        // depth-first steps in the same order either way; only their timing
        // changes, so results do not depend on leaf_min.
        //
        // The wave's lanes standing on internal nodes (`inner`, ballot `m`)
        // have their nodes' parts loaded by all active lanes together:
        // parts item = slot * 7 + part, item k of a batch by the k-th active
        // lane, four loads in flight per lane; returns this lane's slot.
        auto coop_fetch = [&](bool inner, uint64_t m) -> uint32_t {
            const uint64_t below = (1ull << lane) - 1ull;
            const uint32_t slot = (uint32_t)__popcll(m & below);
            const uint32_t items = NODE_PARTS * (uint32_t)__popcll(m);
            const uint64_t act = __ballot(1);
            const uint32_t na = (uint32_t)__popcll(act), ar = (uint32_t)__popcll(act & below);
            if (inner) lds_slot[slot] = cur & ~REF_AXIS_MASK;
            __syncthreads();
            for (uint32_t base = 0; base < items; base += 4 * na) {
                uint4 v[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t item = base + (uint32_t)k * na + ar;
                    if (item < items)
                        v[k] = reinterpret_cast<const uint4*>(a.nodes + lds_slot[item / NODE_PARTS])[item % NODE_PARTS];
                }
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t item = base + (uint32_t)k * na + ar;
                    if (item < items) lds_nodes[item] = v[k];
                }
            }
            __syncthreads();
            return slot;
        };
        // One descent step of a lane standing on an internal node: its four
        // child boxes, then the hit children pushed in visit order.  The step
        // is most of the kernel's instructions, and issuing them bounds it
        // (with the L1's one tag lookup per lane and part): so the planes are
        // loaded in the order the ray meets them, the box test of finite rays
        // is min3/max3, and order and pushes take no branches, about 115
        // vector instructions where a compare-and-select test, a table order
        // and a branch per child took 230.  16.7M incoherent rays on the
        // 1M-triangle sphere: 3.98 -> 3.41 ms at 24 waves per CU and leaf_min
        // 32, 6.77 -> 5.17 ms at 16 and 0.
        auto node_step = [&](uint32_t slot) {
            // The node's parts; `toward` gives a plane's distance from the
            // node's start.
            const char* const base = reinterpret_cast<const char*>(a.nodes);
            const uint32_t off = cur << 7;  // drops the axis bits, and the index bits of a BIG scene
            const char* const big = base + ((uint64_t)(cur & ~REF_AXIS_MASK) << 7);
            const char* const staged = reinterpret_cast<const char*>(lds_nodes + (COOP ? slot * NODE_PARTS : 0u));
            auto part = [&](uint32_t plane) {
                return COOP ? reinterpret_cast<const float4*>(staged + plane)
                            : reinterpret_cast<const float4*>(BIG ? big + plane : base + (uint64_t)(off + plane));
            };
            const uint4 refs = *reinterpret_cast<const uint4*>(part(0) + 6);
            // Time-sampled scenes also read the last 16 bytes, for the
            // bounds' sample count and location.
            uint4 tail = make_uint4(0u, 0u, 0u, 0u);
            if (MOTION) tail = *reinterpret_cast<const uint4*>(part(0) + 7);
            const uint32_t blen = MOTION ? ((tail.z >> 8) & 0xffu) : 1u;
            // The four boxes' planes as the ray meets them: low and high
            // planes are 16 bytes apart, swapped where the ray runs down.
            float4 nx, fx, ny, fy, nz, fz;
            if (!MOTION || blen <= 1) {
                nx = *part(near_x);               fx = *part(near_x ^ 16u);
                ny = *(part(near_y) + 2);         fy = *(part(near_y ^ 16u) + 2);
                nz = *(part(near_z) + 4);         fz = *(part(near_z ^ 16u) + 4);
                if (COUNT) c_nodes++;
            } else {
                uint32_t i1;
                float a2;
                const bool between = lerp_slice_pos(blen, time, i1, a2);
                const float4* m = reinterpret_cast<const float4*>(a.motion + tail.w + i1);
                float4 lx = m[0], hx = m[1], ly = m[2], hy = m[3], lz = m[4], hz = m[5];
                if (between) {
                    m += 6;
                    lx = lerp4(lx, m[0], a2); hx = lerp4(hx, m[1], a2);
                    ly = lerp4(ly, m[2], a2); hy = lerp4(hy, m[3], a2);
                    lz = lerp4(lz, m[4], a2); hz = lerp4(hz, m[5], a2);
                }
                nx = near_x ? hx : lx; fx = near_x ? lx : hx;
                ny = near_y ? hy : ly; fy = near_y ? ly : hy;
                nz = near_z ? hz : lz; fz = near_z ? lz : hz;
                if (COUNT) c_mnodes++;
            }
            bool h0, h1, h2, h3;
            if (__ballot(!finite) == 0) {
                h0 = slab_finite(nx.x, fx.x, ny.x, fy.x, nz.x, fz.x, lo, di, tmax);
                h1 = slab_finite(nx.y, fx.y, ny.y, fy.y, nz.y, fz.y, lo, di, tmax);
                h2 = slab_finite(nx.z, fx.z, ny.z, fy.z, nz.z, fz.z, lo, di, tmax);
                h3 = slab_finite(nx.w, fx.w, ny.w, fy.w, nz.w, fz.w, lo, di, tmax);
                if (MOTION) {
                    // lerped planes of an absent slot may be NaN
                    h1 = h1 && (refs.y | REF_AXIS_MASK) != REF_EMPTY;
                    h3 = h3 && (refs.w | REF_AXIS_MASK) != REF_EMPTY;
                }
            } else {
                // Some lane's ray has a zero direction component or the like:
                // the test in its own operand order, low plane first.
                // (child by child, so the rare path holds few registers)
                auto ordered = [&](float na, float fa, float nb, float fb, float nc, float fc) {
                    const bool h = slab(near_x ? fa : na, near_x ? na : fa, near_y ? fb : nb, near_y ? nb : fb,
                                        near_z ? fc : nc, near_z ? nc : fc, lo, di, tmax);
                    __builtin_amdgcn_sched_barrier(0);
                    return h;
                };
                h0 = ordered(nx.x, fx.x, ny.x, fy.x, nz.x, fz.x);
                h1 = ordered(nx.y, fx.y, ny.y, fy.y, nz.y, fz.y) && (refs.y | REF_AXIS_MASK) != REF_EMPTY;
                h2 = ordered(nx.z, fx.z, ny.z, fy.z, nz.z, fz.z);
                h3 = ordered(nx.w, fx.w, ny.w, fy.w, nz.w, fz.w) && (refs.w | REF_AXIS_MASK) != REF_EMPTY;
            }
            // The hit children in visit order (layout.h): REF_EMPTY where a
            // slot was missed, then the swaps within and of the two sides.
            const uint32_t r0 = h0 ? refs.x : REF_EMPTY, r1 = h1 ? refs.y : REF_EMPTY;
            const uint32_t r2 = h2 ? refs.z : REF_EMPTY, r3 = h3 ? refs.w : REF_EMPTY;
            const bool swap_l = (refs.y & down) != 0u, swap_r = (refs.w & down) != 0u, swap_t = (refs.x & down) != 0u;
            const uint32_t l0 = swap_l ? r1 : r0, l1 = swap_l ? r0 : r1;
            const uint32_t g0 = swap_r ? r3 : r2, g1 = swap_r ? r2 : r3;
            const uint32_t v0 = swap_t ? g0 : l0, v1 = swap_t ? g1 : l1, v2 = swap_t ? l0 : g0, v3 = swap_t ? l1 : g1;
            // The first becomes the current node; the others go on the stack,
            // last first.  Every step stores three entries above the top and
            // counts those that are real.
            const bool e0 = v0 != REF_EMPTY, e1 = v1 != REF_EMPTY, e2 = v2 != REF_EMPTY, e3 = v3 != REF_EMPTY;
            SSTACK_MAKE_ROOM(4);
            SSTACK_AT(sp) = v3;
            sp += e3 && (e0 || e1 || e2) ? ENTRY : 0u;
            SSTACK_AT(sp) = v2;
            sp += e2 && (e0 || e1) ? ENTRY : 0u;
            SSTACK_AT(sp) = v1;
            sp += e1 && e0 ? ENTRY : 0u;
            cur = e0 ? v0 : e1 ? v1 : e2 ? v2 : v3;
        };
        // leaf_min 0: dead ends leave the loop, and it runs until no lane
        // stands on an internal node.
        const uint32_t n_active = (uint32_t)__popcll(__ballot(1));
        for (;;) {
            if (leaf_min != 0 && cur == REF_EMPTY && sp > (in_inst ? inst_base : 0u)) SSTACK_POP(cur);
            const bool inner = !(cur & REF_LEAF);
            const uint64_t m = __ballot(inner);
            const uint32_t n_inner = (uint32_t)__popcll(m);
            if (n_inner == 0 || (leaf_min != 0 && n_active - n_inner >= leaf_min)) break;
            const uint32_t slot = COOP ? coop_fetch(inner, m) : 0u;
            if (inner) node_step(slot);
        }

        // ---- leaf --------------------------------------------------------
        bool finished = false;
        if (cur != REF_EMPTY && (cur & REF_LEAF)) {
            const uint32_t first = (cur & ~(REF_LEAF | REF_AXIS_MASK)) >> 2;
            const uint32_t count = cur & 3u;
            const uint32_t ii = NESTED ? gbase + first : first;
            if (NESTED && !in_inst && count == 0u) {
                // Level marker: the sub-assembly is done; back to the
                // enclosing assembly's path and local ray (tracer.rs:131-148).
                grp = first;
                const GpuGroup g = a.groups[grp];
                gbase = g.base;
                level_local_ray(a, g, time, o, d, lo, di);
                local_ray_set();
                cur = REF_EMPTY;
            } else if (NESTED && !in_inst && a.instances[ii].kind == PSY_OBJECT_ASSEMBLY) {
                // Sub-assembly instance (tracer.rs:95-128): remember the
                // enclosing path on the stack, move the ray into the
                // sub-assembly's space and walk its instance BVH.
                if (COUNT) c_inst++;
                SSTACK_MAKE_ROOM(1);
                SSTACK_AT(sp) = make_level_marker(grp);
                sp += ENTRY;
                grp = a.instances[ii].mesh;
                const GpuGroup g = a.groups[grp];
                gbase = g.base;
                level_local_ray(a, g, time, o, d, lo, di);
                local_ray_set();
                cur = g.root;
            } else if (!in_inst && XF && a.instances[ii].kind != PSY_OBJECT_MESH) {
                // Light instance (tracer.rs:95-128 with a light object; light
                // instances always carry transforms).
                const GpuInstance inst = a.instances[ii];
                if (COUNT) c_inst++;
                const Xf x = instance_xf(a.xforms, inst, time);
                const V3 llo = xf_point(x, o);
                const V3 lld = xf_vector(x, d);
                float lt, l0, l1, l2;
                uint32_t lp;
                if (light_leaf_test(a.rect_lights, a.sphere_lights, a.light_samples, time, inst, x, o, pre, llo, lld,
                                    tmax, lt, l0, l1, l2, lp)) {
                    if (occl) {
                        kind = PSY_HIT_OCCLUDE;
                        finished = true;
                    } else {
                        tmax = lt;
                        finite = finite && lt == lt;
                        kind = PSY_HIT_SURFACE;
                        ht = lt; hb0 = l0; hb1 = l1; hb2 = l2;
                        hprim = lp;
                        hinst = inst.id;
                    }
                }
                cur = REF_EMPTY;
            } else if (!DIRECT && !in_inst) {
                // Instance leaf (tracer.rs:95-128).
                const GpuInstance inst = a.instances[ii];
                const GpuMesh mesh = a.meshes[inst.mesh];
                if (COUNT) c_inst++;
                if (XF) {
                    if (inst.xf_count > 0) {
                        uint32_t i1;
                        float a2;
                        Xf x;
                        if (!lerp_slice_pos(inst.xf_count, time, i1, a2))
                            x = load_xf(a.xforms + inst.xf_start + i1);
                        else
                            x = xf_lerp(load_xf(a.xforms + inst.xf_start + i1),
                                        load_xf(a.xforms + inst.xf_start + i1 + 1), a2);
                        lo = xf_point(x, o);
                        V3 ld = xf_vector(x, d);
                        di = v3(1.0f / ld.x, 1.0f / ld.y, 1.0f / ld.z);
                        local_ray_set();
                        space = inst.xf_count == 1 ? load_xf(a.inv_static + inst.inv_static) : xf_inverse(x);
                        has_space = true;
                    } else {
                        has_space = false;
                    }
                }
                in_inst = true;
                inst_base = sp;
                inst_id = inst.id;
                tri_base = mesh.tri_offset;
                if (MOTION) {
                    tri_stride = mesh.tri_stride;
                    tri_samples = mesh.time_samples;
                }
                cur = mesh.root;
            } else {
                // Triangle leaf (triangle_mesh.rs:174-260).
                for (uint32_t j = 0; j < count; j++) {
                    const uint8_t* rec = a.tris + tri_base + (uint64_t)(first + j) * tri_stride;
                    V3 v0, v1, v2;
                    uint32_t prim;
                    if (!MOTION || tri_samples == 1) {
                        const float4* f = reinterpret_cast<const float4*>(rec);
                        const float4 q0 = f[0], q1 = f[1], q2 = f[2];
                        v0 = v3(q0.x, q0.y, q0.z);
                        v1 = v3(q0.w, q1.x, q1.y);
                        v2 = v3(q1.z, q1.w, q2.x);
                        prim = __float_as_uint(q2.y);
                        if (COUNT) c_tris++;
                    } else {
                        const float* f = reinterpret_cast<const float*>(rec);
                        uint32_t i1;
                        float a2;
                        if (!lerp_slice_pos(tri_samples, time, i1, a2)) {
                            const float* s0 = f + i1 * 9;
                            v0 = v3(s0[0], s0[1], s0[2]);
                            v1 = v3(s0[3], s0[4], s0[5]);
                            v2 = v3(s0[6], s0[7], s0[8]);
                        } else {
                            const float* s0 = f + i1 * 9;
                            const float* s1 = s0 + 9;
                            v0 = lerp3(v3(s0[0], s0[1], s0[2]), v3(s1[0], s1[1], s1[2]), a2);
                            v1 = lerp3(v3(s0[3], s0[4], s0[5]), v3(s1[3], s1[4], s1[5]), a2);
                            v2 = lerp3(v3(s0[6], s0[7], s0[8]), v3(s1[6], s1[7], s1[8]), a2);
                        }
                        prim = *reinterpret_cast<const uint32_t*>(f + 9 * tri_samples);
                        if (COUNT) c_mtris++;
                    }
                    if (XF && has_space) {
                        v0 = xf_point(space, v0);
                        v1 = xf_point(space, v1);
                        v2 = xf_point(space, v2);
                    }
                    float t, b0, b1, b2;
                    if (tri_test(o, pre, tmax, v0, v1, v2, t, b0, b1, b2)) {
                        if (occl) {
                            kind = PSY_HIT_OCCLUDE;
                            finished = true;
                            break;
                        }
                        tmax = t;
                        finite = finite && t == t;
                        kind = PSY_HIT_SURFACE;
                        ht = t; hb0 = b0; hb1 = b1; hb2 = b2;
                        hprim = prim;
                        hinst = inst_id;
                    }
                }
                cur = REF_EMPTY;
            }
        }

        // ---- pop, leaving the instance when its subtree is done -----------
        if (!finished && cur == REF_EMPTY) {
            if (in_inst && sp == inst_base) {
                in_inst = false;
                if (NESTED) {
                    level_local_ray(a, a.groups[grp], time, o, d, lo, di);
                    local_ray_set();
                } else if (XF) {
                    lo = xf_point(ident, o);
                    V3 ld = xf_vector(ident, d);
                    di = v3(1.0f / ld.x, 1.0f / ld.y, 1.0f / ld.z);
                    local_ray_set();
                }
            }
            if (sp == 0) finished = true;
            else SSTACK_POP(cur);
        }

        if (finished) {
            if (a.n2_kind != nullptr && occl) {
                a.n2_kind[ray] = kind;
            } else if (a.rec != nullptr) {
                // One 32-byte record per ray, two 16-byte stores: rays finish
                // out of order, and a whole record fills a memory sector
                // where the seven arrays of the SoA form leave seven partial
                // lines.
                const bool s = kind == PSY_HIT_SURFACE;
                uint4* r = a.rec + 2ull * ray;
                r[0] = make_uint4(s ? __float_as_uint(ht) : 0u, s ? __float_as_uint(hb0) : 0u,
                                  s ? __float_as_uint(hb1) : 0u, s ? __float_as_uint(hb2) : 0u);
                r[1] = make_uint4(s ? hprim : PSY_NONE, s ? hinst : PSY_NONE, (uint32_t)kind, 0u);
            } else {
                a.kind[ray] = kind;
                if (kind == PSY_HIT_SURFACE) {
                    a.t[ray] = ht;
                    a.b0[ray] = hb0;
                    a.b1[ray] = hb1;
                    a.b2[ray] = hb2;
                    a.prim_id[ray] = hprim;
                    a.inst_id[ray] = hinst;
                }
            }
            has = false;
        }
    }
    if (COUNT) {
        atomicAdd(a.counters + 0, (unsigned long long)c_nodes);
        atomicAdd(a.counters + 1, (unsigned long long)c_mnodes);
        atomicAdd(a.counters + 2, (unsigned long long)c_tris);
        atomicAdd(a.counters + 3, (unsigned long long)c_mtris);
        atomicAdd(a.counters + 4, (unsigned long long)c_inst);
    }
}

// Zeroes the ranges' counters with a kernel, so the launch sequence can be
// captured in a graph (no memset node).
__global__ void reset_work_kernel(unsigned int* work) { work[threadIdx.x * TRACE_RANGE_WORDS] = 0u; }

// Launches one build of the kernel with at most as many waves as the chip
// holds at once (its registers and LDS decide; the same on every gfx950, so
// asked once per build): the waves start on equal shares of the rays, and a
// wave that has to wait for another to end starts its share that late.
// Launched at 24 per CU where 20 fit, 16.7M incoherent rays took 3.42 ms and
// at 20 3.33; the motion scene's 1M rays 1.70 ms at 20 where 16 fit and 1.35
// at 16.  A CU hands out its LDS in LDS_GRANULE pieces, which the runtime's
// answer leaves out: 18 waves with 8 KB fit, not 20 (4.2M rays on the
// 1M-triangle sphere cut into 16 meshes, stack_lds 24: 1.50 ms at 18 waves,
// 1.70 at 19 and 20).
constexpr uint32_t LDS_PER_CU = 160u << 10, LDS_GRANULE = 1280;
template <auto KERNEL>
hipError_t launch_resident(const TraceArgs& a, unsigned int* work, const TraceTuning& tune, hipStream_t s) {
    static std::atomic<uint32_t> resident{0};
    uint32_t per_cu = resident.load(std::memory_order_relaxed);
    if (per_cu == 0) {
        int blocks = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, KERNEL, WAVE, 0);
        hipFuncAttributes fa{};
        if (e == hipSuccess) e = hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(KERNEL));
        if (e != hipSuccess) return e;
        const uint32_t pieces = ((uint32_t)fa.sharedSizeBytes + LDS_GRANULE - 1u) / LDS_GRANULE;
        per_cu = std::max(1u, std::min((uint32_t)std::max(1, blocks), LDS_PER_CU / LDS_GRANULE / std::max(1u, pieces)));
        resident.store(per_cu, std::memory_order_relaxed);
    }
    const uint32_t waves =
        (tune.cus * std::min(tune.waves_per_cu, per_cu) + TRACE_RANGES - 1u) / TRACE_RANGES * TRACE_RANGES;
    // Waves that start on all of the rays read no counter.
    if (!a.work_next && (a.n_dev || a.n2_dev ||
        (uint64_t)first_rays((uint32_t)a.n, waves) * (waves / TRACE_RANGES) < range_count((uint32_t)a.n, 0))) {
        hipLaunchKernelGGL(reset_work_kernel, dim3(1), dim3(TRACE_RANGES), 0, s, work);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(KERNEL, dim3(waves), dim3(WAVE), 0, s, a, work, tune.refill_min, tune.leaf_min);
    return hipGetLastError();
}

template <bool COUNT, bool XF, bool MOTION, uint32_t RING, bool NESTED, bool BIG, bool DIRECT>
hipError_t launch_one(const TraceArgs& a, unsigned int* work, const TraceTuning& tune, hipStream_t s) {
    // Register budget: at most 128 VGPRs (four waves per SIMD), or what the
    // compiler takes of its own (96 and 98 in static builds, 126 with
    // transforms, up to 152 with time samples as well, which leaves three
    // waves).  A budget of eight waves, 64 VGPRs, would spill in the node
    // step: at 24 waves per CU and leaf_min 32, 4.2M rays on the 1M-triangle
    // sphere took 1.98 ms so and 1.13 with 98 registers, 1M rays on the
    // motion scene 2.62 and 0.88.
    // The cooperative node fetch serves static single-level scenes.
    if constexpr (!COUNT && !MOTION && !NESTED && !BIG) {
        if (tune.coop) {
            if (tune.occupancy >= 8) return launch_resident<&trace_persistent_kernel<false, XF, false, RING, 1, true, false, false, DIRECT>>(a, work, tune, s);
            return launch_resident<&trace_persistent_kernel<false, XF, false, RING, 4, true, false, false, DIRECT>>(a, work, tune, s);
        }
    }
    if constexpr (!COUNT && !BIG) {
        if (tune.occupancy >= 8) return launch_resident<&trace_persistent_kernel<false, XF, MOTION, RING, 1, false, NESTED, false, DIRECT>>(a, work, tune, s);
    }
    return launch_resident<&trace_persistent_kernel<COUNT, XF, MOTION, RING, 4, false, NESTED, BIG, DIRECT>>(a, work, tune, s);
}

template <bool COUNT, bool XF, bool MOTION, bool NESTED, bool DIRECT>
hipError_t launch_depth(const TraceArgs& a, unsigned int* work, const TraceTuning& tune, hipStream_t s) {
    if constexpr (COUNT || NESTED) {
        return launch_one<COUNT, XF, MOTION, 16, NESTED, false, DIRECT>(a, work, tune, s);
    } else {
        switch (tune.lds_depth) {
            case 8: return launch_one<COUNT, XF, MOTION, 8, false, false, DIRECT>(a, work, tune, s);
            case 24: return launch_one<COUNT, XF, MOTION, 32, false, false, DIRECT>(a, work, tune, s);
            default: return launch_one<COUNT, XF, MOTION, 16, false, false, DIRECT>(a, work, tune, s);
        }
    }
}

template <bool COUNT>
hipError_t launch_feat(const TraceArgs& a, unsigned int* work, const TraceTuning& tune, bool xf, bool motion,
                       hipStream_t s) {
    const bool direct = !a.groups && !xf && a.top_root != REF_EMPTY && (a.top_root & REF_LEAF);
    // More than 4 GB of nodes: builds with 64-bit node offsets, by the same
    // features (in one build for all of them, 4.2M rays on the 1M-triangle
    // sphere addressed so took 1.63 ms and 1.08 in the static one, 1M rays on
    // the large instanced scene 0.59 and 0.50).
    if (a.wide) {
        if (a.groups) return launch_one<COUNT, true, true, 16, true, true, false>(a, work, tune, s);
        if (motion) return launch_one<COUNT, true, true, 16, false, true, false>(a, work, tune, s);
        if (xf) return launch_one<COUNT, true, false, 16, false, true, false>(a, work, tune, s);
        if (direct) return launch_one<COUNT, false, false, 16, false, true, true>(a, work, tune, s);
        return launch_one<COUNT, false, false, 16, false, true, false>(a, work, tune, s);
    }
    // Nested scenes take the transform path, with or without time samples.
    if (a.groups) {
        if (motion) return launch_depth<COUNT, true, true, true, false>(a, work, tune, s);
        return launch_depth<COUNT, true, false, true, false>(a, work, tune, s);
    }
    if (xf && motion) return launch_depth<COUNT, true, true, false, false>(a, work, tune, s);
    if (xf) return launch_depth<COUNT, true, false, false, false>(a, work, tune, s);
    if (motion && direct) return launch_depth<COUNT, false, true, false, true>(a, work, tune, s);
    if (motion) return launch_depth<COUNT, false, true, false, false>(a, work, tune, s);
    if (direct) return launch_depth<COUNT, false, false, false, true>(a, work, tune, s);
    return launch_depth<COUNT, false, false, false, false>(a, work, tune, s);
}

}  // namespace

hipError_t launch_trace_persistent(const TraceArgs& args, bool counted, bool has_xf, bool has_motion,
                                   unsigned int* work, const TraceTuning& tune, hipStream_t stream) {
    if (args.n == 0 && !args.n2_dev) return hipSuccess;
    if (args.n >= 0x80000000ull || tune.cus == 0 || tune.waves_per_cu == 0 || tune.refill_min == 0 ||
        tune.refill_min > 64 || tune.leaf_min > 64)
        return hipErrorInvalidValue;
    return counted ? launch_feat<true>(args, work, tune, has_xf, has_motion, stream)
                   : launch_feat<false>(args, work, tune, has_xf, has_motion, stream);
}

}  // namespace psy
