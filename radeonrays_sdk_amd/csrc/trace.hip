// trace.hip — BVH2 ray traversal for gfx950.
//
// Behavioural spec: vlk/kernels/isect.comp:88-246 (single level) and
// isect_2l.comp:136-323 (two level): one lane per ray, depth-first stack
// traversal that descends into the nearer of two hit children first
// (child0 on ties) and defers the other; a TLAS leaf transforms the ray by
// the instance's inverse transform, pushes a sentinel and restarts at the
// BLAS root; popping the sentinel restores the world ray.
// Differences from the reference, all deliberate:
//   * triangles use the watertight test (rr_device.h) and closest hits are
//     ordered by (t, instance, primitive), so the result does not depend on
//     the BVH's shape;
//   * slab tests are conservative (widened by a few ulp);
//   * the stack keeps 8, 16 or 32 entries per lane in LDS as a ring (16 by
//     default) and spills the oldest entry to scratch one at a time; a ray
//     that needs more than kStackCapacity entries ends and sets the
//     stack-overflow error word instead of dropping entries silently;
//   * a miss writes a complete record (inst_id = prim_id = ~0);
//   * every kernel checks the buffer's header first: a buffer this library
//     did not write sets the bad-buffer error word, and a kernel for the
//     other level returns at once (rrCmdIntersect on a buffer the host has
//     not seen built launches both levels and lets the header decide).
#include <hip/hip_runtime.h>

#include "device_errors.h"
#include "rr_device.h"
#include "trace.h"
#include "trace_grid.h"

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>

namespace rr {

namespace {

constexpr int kBlock = kTraceBlock;

// Trace scratch: kQueues ray-queue counters, each on its own 128-byte line,
// then kSpillEntries stack slots per lane.
constexpr uint32_t kQueues = 8;
constexpr uint32_t kQueueStride = 32;
constexpr uint32_t kQueueHeadWords = kQueues * kQueueStride;

struct RayIn {
    float4 a;  // origin.xyz, min_t
    float4 b;  // direction.xyz, max_t
};

__device__ __forceinline__ RayIn LoadRay(const float4* __restrict__ rays, uint32_t i) {
    RayIn r;
    r.a = LdG4(rays + 2 * (size_t)i);
    r.b = LdG4(rays + 2 * (size_t)i + 1);
    return r;
}

// True if the buffer's header names kind `want`.  A buffer this library did
// not write (wrong magic or kind) sets the bad-buffer error word and gives
// false, as does a valid buffer of the other kind (silently).
__device__ __forceinline__ bool HeaderIs(const AccelHeader* h, uint32_t want, uint32_t* err) {
    const uint32_t magic = h->magic, kind = h->kind;
    if (magic == kAccelMagic && (kind == kAccelBlas || kind == kAccelTlas)) return kind == want;
    if (err && blockIdx.x == 0 && threadIdx.x == 0) StG(err + kErrBadAccel, 1u);
    return false;
}

// LDS ring of DEPTH entries + scratch spill stack for one lane.
template <int DEPTH = kLdsStackEntries>
struct LaneStack {
    static_assert((DEPTH & (DEPTH - 1)) == 0, "ring depth must be a power of two");
    static_assert(DEPTH >= kMinLdsStackEntries && kStackCapacity - DEPTH <= kSpillEntries, "spill slots per lane");
    uint32_t (*lds)[64];  // this wave's rows
    uint32_t* spill;  // this wave's spill slots (uniform): lane l's are [l * kSpillEntries, (l + 1) * kSpillEntries)
    uint32_t* err;    // device error words (may be null)
    int sp;     // entries pushed so far (index of the next push)
    int gbase;  // entries [0, gbase) live in scratch, [gbase, sp) in LDS

    // A 32-bit lane offset from the wave's base: one register, not a 64-bit pointer per lane.
    __device__ __forceinline__ uint32_t* slot(int k) const { return spill + ((threadIdx.x & 63u) * (uint32_t)kSpillEntries + (uint32_t)k); }

    __device__ __forceinline__ bool empty() const { return sp == 0; }
    __device__ __forceinline__ void clear() { sp = gbase = 0; }
    __device__ __forceinline__ void push(uint32_t v) {
        if (sp == kStackCapacity) {
            // Tree deeper than the stack: report it and end the ray (its
            // deferred nodes, and in a scene the instance sentinel, are
            // discarded, so the lane finishes the current descent and stops).
            if (err) StG(err + kErrStackOverflow, 1u);
            clear();
            return;
        }
        if (sp - gbase == DEPTH) {
            StG(slot(gbase), lds[gbase & (DEPTH - 1)][threadIdx.x & 63u]);
            ++gbase;
        }
        lds[sp & (DEPTH - 1)][threadIdx.x & 63u] = v;
        ++sp;
    }
    __device__ __forceinline__ uint32_t pop() {
        --sp;
        // Read the LDS slot unconditionally (a plain ds_read) and replace it
        // from scratch only when the entry was spilled.
        uint32_t v = lds[sp & (DEPTH - 1)][threadIdx.x & 63u];
        if (sp < gbase) {
            gbase = sp;
            v = LdG(slot(sp));
        }
        return v;
    }
};

template <bool ANY, int OUT, bool TWO_LEVEL, bool STATS>
__global__ __launch_bounds__(kBlock) void TraceKernel(const uint8_t* __restrict__ accel, const float4* __restrict__ rays,
                                                      uint32_t ray_count, const uint32_t* __restrict__ indirect,
                                                      void* __restrict__ hits, uint32_t* __restrict__ scratch,
                                                      uint32_t* __restrict__ stats, uint32_t* err) {
    __shared__ uint32_t s_stack[kBlock / 64][kLdsStackEntries][64];
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    uint32_t n = ray_count;
    if (indirect) n = min(n, *indirect);
    if (i >= n) return;

    const AccelHeader* hdr = reinterpret_cast<const AccelHeader*>(accel);
    if (!HeaderIs(hdr, TWO_LEVEL ? kAccelTlas : kAccelBlas, err)) return;
    const uint32_t top_count = hdr->node_count;
    const BvhNode* top_nodes = reinterpret_cast<const BvhNode*>(accel + hdr->nodes_offset);
    bool boxes = !TWO_LEVEL && (hdr->flags & kAccelFlagAabbs) != 0;  // leaf kind of the level traversed
    const Transform* xforms = nullptr;
    const uint64_t* blas_table = nullptr;
    if (TWO_LEVEL) {
        xforms = reinterpret_cast<const Transform*>(accel + hdr->transforms_offset);
        blas_table = reinterpret_cast<const uint64_t*>(accel + hdr->blas_table_offset);
    }

    const RayIn ray = LoadRay(rays, i);
    RayState r;
    SetupRay(r, ray.a.x, ray.a.y, ray.a.z, ray.a.w, ray.b.x, ray.b.y, ray.b.z);
    const float tmax = ray.b.w;

    float best_t = tmax;
    uint32_t best_prim = kInvalid, best_inst = kInvalid;
    float bV = 0.0f, bW = 0.0f, bdet = 1.0f;
    float limit = WidenLimit(tmax);
    uint32_t n_internal_visits = 0, n_leaf_visits = 0, n_box_tests = 0, n_tri_tests = 0;

    LaneStack<> st{s_stack[threadIdx.x / 64], scratch + kQueueHeadWords + (size_t)(blockIdx.x * kBlock + (threadIdx.x & ~63u)) * kSpillEntries, err, 0, 0};
    const BvhNode* nodes = top_nodes;
    uint32_t node_count = top_count;  // of the level being traversed (bounds every node index)
    uint32_t inst = kInvalid;  // kInvalid while in the top level
    uint32_t node = 0;
    bool alive = top_count != 0;
    while (alive) {
        if (node >= node_count) break;  // corrupt buffer: stop this ray rather than read out of bounds
        float4 q0, q1, q2, q3;
        LoadNode(nodes, node, q0, q1, q2, q3);
        const uint32_t c0 = __float_as_uint(q0.w);
        const uint32_t c1 = __float_as_uint(q1.w);
        if (c0 != kInvalid) {
            if (STATS) { ++n_internal_visits; n_box_tests += 2; }
            float ta, tb;
            const bool h0 = SlabTest(r, limit, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, ta);
            const bool h1 = SlabTest(r, limit, q2.x, q2.y, q2.z, q3.x, q3.y, q3.z, tb);
            if (h0 || h1) {
                const bool c1first = h1 && (!h0 || ta > tb);
                if (h0 && h1) st.push(c1first ? c0 : c1);
                node = c1first ? c1 : c0;
                continue;
            }
        } else if (TWO_LEVEL && inst == kInvalid) {
            // Enter instance c1 (isect_2l.comp:222-237).
            if (STATS) ++n_leaf_visits;
            const uint8_t* blas = reinterpret_cast<const uint8_t*>(LdG(blas_table + c1));
            const AccelHeader* bh = reinterpret_cast<const AccelHeader*>(blas);
            const uint32_t bn = LdG(&bh->node_count);
            if (bn != 0) {
                const Transform x = xforms[2 * (size_t)c1];
                const float ox = ((x.m[0][0] * ray.a.x + x.m[0][1] * ray.a.y) + x.m[0][2] * ray.a.z) + x.m[0][3];
                const float oy = ((x.m[1][0] * ray.a.x + x.m[1][1] * ray.a.y) + x.m[1][2] * ray.a.z) + x.m[1][3];
                const float oz = ((x.m[2][0] * ray.a.x + x.m[2][1] * ray.a.y) + x.m[2][2] * ray.a.z) + x.m[2][3];
                const float dx = (x.m[0][0] * ray.b.x + x.m[0][1] * ray.b.y) + x.m[0][2] * ray.b.z;
                const float dy = (x.m[1][0] * ray.b.x + x.m[1][1] * ray.b.y) + x.m[1][2] * ray.b.z;
                const float dz = (x.m[2][0] * ray.b.x + x.m[2][1] * ray.b.y) + x.m[2][2] * ray.b.z;
                SetupRay(r, ox, oy, oz, ray.a.w, dx, dy, dz);
                inst = c1;
                nodes = reinterpret_cast<const BvhNode*>(blas + LdG(&bh->nodes_offset));
                node_count = bn;
                boxes = (LdG(&bh->flags) & kAccelFlagAabbs) != 0;
                st.push(kTopLevelSentinel);
                node = 0;
                continue;
            }
        } else {
            if (STATS) { ++n_leaf_visits; ++n_tri_tests; }
            TriHit h;
            if (LeafTest(boxes, r, best_t, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, q2.x, q2.y, q2.z, h) && h.t >= r.tmin &&
                h.t <= best_t) {
                const uint32_t hit_inst = TWO_LEVEL ? inst : 0u;
                if (ANY) {
                    best_t = h.t; best_prim = c1; best_inst = hit_inst;
                    bV = h.V; bW = h.W; bdet = h.det;
                    break;
                }
                if (CloserHit(h.t, hit_inst, c1, best_t, best_inst, best_prim)) {
                    best_t = h.t; best_prim = c1; best_inst = hit_inst;
                    bV = h.V; bW = h.W; bdet = h.det;
                    limit = WidenLimit(best_t);
                }
            }
        }
        // Pop the next deferred node.
        for (;;) {
            if (st.empty()) { alive = false; break; }
            node = st.pop();
            if (TWO_LEVEL && node == kTopLevelSentinel) {
                // Leave the instance and restore the world ray (isect_2l.comp:278-286).
                inst = kInvalid;
                nodes = top_nodes;
                node_count = top_count;
                boxes = false;
                SetupRay(r, ray.a.x, ray.a.y, ray.a.z, ray.a.w, ray.b.x, ray.b.y, ray.b.z);
                continue;
            }
            break;
        }
    }

    if (STATS) {
        uint4* s = reinterpret_cast<uint4*>(stats) + i;
        *s = make_uint4(n_internal_visits, n_leaf_visits, n_box_tests, n_tri_tests);
    }
    const bool hit = best_prim != kInvalid;
    const float u = hit ? bV / bdet : 0.0f;
    const float v = hit ? bW / bdet : 0.0f;
    if (OUT == kOutFullHit) {
        reinterpret_cast<float4*>(hits)[i] = hit ? make_float4(u, v, __uint_as_float(best_inst), __uint_as_float(best_prim))
                                                 : make_float4(0.0f, 0.0f, __uint_as_float(kInvalid), __uint_as_float(kInvalid));
    } else if (OUT == kOutInstanceId) {
        // Single level writes the primitive id (isect.comp:235), two level the instance (isect_2l.comp:311).
        reinterpret_cast<uint32_t*>(hits)[i] = hit ? (TWO_LEVEL ? best_inst : best_prim) : kInvalid;
    } else {
        float4* o = reinterpret_cast<float4*>(hits) + 2 * (size_t)i;
        o[0] = hit ? make_float4(u, v, __uint_as_float(best_inst), __uint_as_float(best_prim))
                   : make_float4(0.0f, 0.0f, __uint_as_float(kInvalid), __uint_as_float(kInvalid));
        o[1] = make_float4(hit ? best_t : tmax, 0.0f, 0.0f, 0.0f);
    }
}

// Write the query's output record for ray i.
template <int OUT, bool TWO_LEVEL>
__device__ __forceinline__ void WriteHit(void* __restrict__ hits, uint32_t i, bool hit, float u, float v,
                                         uint32_t inst, uint32_t prim, float t, float tmax) {
    if (OUT == kOutFullHit) {
        StG4(reinterpret_cast<float4*>(hits) + i,
             hit ? make_float4(u, v, __uint_as_float(inst), __uint_as_float(prim))
                 : make_float4(0.0f, 0.0f, __uint_as_float(kInvalid), __uint_as_float(kInvalid)));
    } else if (OUT == kOutInstanceId) {
        StG(reinterpret_cast<uint32_t*>(hits) + i, hit ? (TWO_LEVEL ? inst : prim) : kInvalid);
    } else {
        float4* o = reinterpret_cast<float4*>(hits) + 2 * (size_t)i;
        StG4(o, hit ? make_float4(u, v, __uint_as_float(inst), __uint_as_float(prim))
                    : make_float4(0.0f, 0.0f, __uint_as_float(kInvalid), __uint_as_float(kInvalid)));
        StG4(o + 1, make_float4(hit ? t : tmax, 0.0f, 0.0f, 0.0f));
    }
}

// ---------------------------------------------------------------------------
// Persistent single-level traversal.
//
// The grid holds only as many waves as the GPU keeps resident.  Rays are split
// into kQueues contiguous ranges, one per XCD (workgroups are dispatched to
// the XCDs round-robin), so that neighbouring rays share an L2; each wave
// starts with a piece of its range, takes further pieces with one atomic each
// and hands the rays to lanes as theirs finish, moving on to the other ranges
// once its own is empty.  Each lane runs a while-while loop (Aila & Laine, "Understanding
// the Efficiency of Ray Traversal on GPUs", HPG 2009): inner nodes until every
// busy lane holds a postponed leaf, then the leaves.  Leaves are still tested
// in depth-first order, so closest and any hits are those of the plain
// kernel; only the number of boxes tested differs.

__global__ void QueueInitKernel(uint32_t* counters, uint32_t ray_count, const uint32_t* __restrict__ indirect) {
    uint32_t n = ray_count;
    if (indirect) n = min(n, *indirect);
    const uint32_t part = (n + kQueues - 1) / kQueues;
    const uint32_t k = threadIdx.x;
    if (k < kQueues) counters[k * kQueueStride] = min(k * part, n);
}

// The same set-up done by a one-block persistent launch that runs before
// the full one (instead of a QueueInitKernel launch): the fence and barrier
// make it visible to the block's own atomics, stream order to the next launch.
__device__ __forceinline__ void InitQueues(uint32_t* counters, uint32_t n) {
    const uint32_t part = (n + kQueues - 1) / kQueues;
    if (threadIdx.x < kQueues) counters[threadIdx.x * kQueueStride] = min(threadIdx.x * part, n);
    __threadfence();
    __syncthreads();
}

// A wave's view of the ray queues (wave-uniform): rays [next, end) are its
// own, and it takes `piece` more at a time from queue q.
struct RayQueue {
    uint32_t next, end, q, piece;
    uint32_t blocks;  // workgroups whose waves started with a piece
    uint32_t tries;   // queues found empty
    bool drained;     // no more rays to take
};

// The rays at the head of queue q that the waves of `blocks` workgroups
// starting on it have from the beginning, a piece each (none for 0): its
// counter counts those behind them.
__device__ __forceinline__ uint32_t QueueFirst(uint32_t q, uint32_t piece, uint32_t blocks) {
    return (blocks + kQueues - 1 - q) / kQueues * (kBlock / 64) * piece;
}

// A wave's first rays.  When the grid's lanes hold every ray, each wave has
// an equal share of them, at most one per lane, and takes none from the
// queues (true); else its piece at the head of its queue, without an atomic
// (all waves at once would wait for each other's: 4M rays of a camera above
// the 1M-triangle terrain 506 -> 491 us, 4M rays towards a 3,000-triangle
// soup 337 -> 330).
//
// A grid for equal shares relies on the pool.  Waves that cannot pool keep
// equal shares of up to kLoneShare rays; beyond that the query is left to the
// first `lone` workgroups, the grid that it has without equal shares, and its
// waves take every piece from the queues (and so refill their lanes).
// Closest hits in a scene of 524,287 instances, rays from outside / inside,
// equal shares against the queues: 24,500 rays (4 a wave) 1093/1135 against
// 1879/2324 us, 49,000 (8) 1640/1485 against 2216/2507, 98,000 (16) 2156/1933
// against 2051/2416, 393,216 (64) 4543/3675 against 2983/3056.  A first piece
// without an atomic gave them nothing (98,000 rays from inside 2416 -> 2759).
constexpr uint32_t kLoneShare = 8;
__device__ __forceinline__ bool StartQueue(RayQueue& s, uint32_t n, uint32_t part, uint32_t fetch, bool pools, uint32_t lone) {
    const uint32_t waves = gridDim.x * (kBlock / 64);
    const uint32_t share = n / waves + (n % waves != 0);
    const bool fixed = share <= (pools ? 64u : kLoneShare);
    s.q = blockIdx.x % kQueues;
    s.piece = fixed ? share : fetch;
    s.blocks = gridDim.x;
    s.tries = 0;
    const uint32_t block = fixed ? XcdContiguousBlock(blockIdx.x, gridDim.x) : blockIdx.x / kQueues;
    const uint32_t first = fixed ? 0 : s.q * part, end = fixed ? n : min((s.q + 1) * part, n);
    const uint32_t w = block * (kBlock / 64) + threadIdx.x / 64;
    s.next = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)min(first + (uint64_t)w * s.piece, (uint64_t)end));
    s.end = s.next + min(s.piece, end - s.next);
    s.drained = fixed && s.next == s.end;
    if (!pools && !fixed) {
        s.blocks = 0;
        s.end = s.next;
        s.drained = blockIdx.x >= lone;
    }
    return fixed;
}

// Takes the next piece, from the next queue that has any once its own is empty.
__device__ __forceinline__ void TakeRays(RayQueue& s, uint32_t* counters, uint32_t n, uint32_t part) {
    while (!s.drained) {
        uint32_t b = 0;
        if (__lane_id() == 0) b = atomicAdd(&counters[s.q * kQueueStride], s.piece);
        b = (uint32_t)__builtin_amdgcn_readfirstlane((int)b) + QueueFirst(s.q, s.piece, s.blocks);
        const uint32_t end = min((s.q + 1) * part, n);
        if (b < end) {
            s.next = b;
            s.end = min(b + s.piece, end);
            return;
        }
        s.drained = ++s.tries == kQueues;
        s.q = s.q + 1 == kQueues ? 0 : s.q + 1;
    }
}

// First spill word of a wave: its lanes' slots, or with equal shares, where
// the grid may have more lanes than rays, its rays' slots.
__device__ __forceinline__ size_t SpillStart(bool fixed, uint32_t first_ray) {
    return (size_t)(fixed ? first_ray : blockIdx.x * kBlock + (threadIdx.x & ~63u)) * kSpillEntries;
}

// ---------------------------------------------------------------------------
// Pooled traversal of a wave's last rays.
//
// Once a wave finds no more rays to fetch, the subtrees its lanes still have
// to visit go into one list in LDS (the lanes' stacks lie there already),
// and the whole wave works on it: each step takes up to 64 entries from the
// top, one per lane, whichever rays they belong to, and pushes the children
// that are hit back.  A ray's remaining work then takes about as many steps
// as the tree is deep instead of one step per node, and every lane has a
// node in each step while 64 are left.  A ray's state stays in its lane's
// registers and is shuffled to the lanes that work for it.
//
// A ray's entries are in depth-first order from the top: lanes take entries in
// that order and their children replace them in that order (near child
// first).  Any hit needs it: the first hit in depth-first order wins, so a
// hit cancels what its ray has below it (later in that order), and a hit
// found above it afterwards replaces it.  Closest hits do not depend on the
// order.  Entries of different rays mix freely, and PoolPush puts each ray's
// next one above everyone's far children: in one depth-first list the top
// 64 entries were a few rays' far subtrees, visited before the near ones
// could cull them (32 camera rays in a 65,536-triangle soup: 98 nodes a ray
// and 54 steps, now 49 and 29; 131,072 such rays 186 -> 118 us, 1M-triangle
// terrain 190 -> 121, scene of 1,000 instances 1265 -> 1084).
//
// What bounds it: the chain of node fetches, a tree's depth of steps of one
// memory round trip each; with many rays left also VALU issue (a step is
// about 130 instructions, 64 entries at once, where the lanes' own loop
// spends a node's on a quarter of its lanes).  4M incoherent rays over the
// 1M-triangle terrain: closest 574 -> 451 us, any 532 -> 399 us, against
// lanes that traverse (closest hit: and split) their rays alone to the end;
// 1,000 rays 111 -> 33 us.  The list takes the stacks' LDS; 72 VGPRs leave
// seven waves per SIMD instead of eight (held to 64 it spills, and was
// slower: 529 us), which costs long rays less than the end of the launch
// gains (65,536-triangle soup, 4M rays from inside: 2524 -> 2401, any
// 1889 -> 1740 us).
//
// An entry is (node, slot | depth << 6): the lane that holds the ray, and
// how many entries the ray's own stack would hold when the node is popped
// from it, so that a tree deeper than kStackCapacity is reported as by the
// other kernels.
constexpr uint32_t kPoolSlotBits = 6;
// Entries kept free for the children of one entry taken at a time, whose
// ray's depth grows by at most kStackCapacity.
constexpr int kPoolReserve = kStackCapacity + 16;

// LDS rows of a wave's stacks and pool.  The pool keeps 16 rows where a stack
// has eight: eight hold 256 entries, and with 96 of them in reserve most
// steps took a few entries only.  On eight-entry stacks, a pool of eight rows
// against 16, closest hits: 65,536-triangle soup, 260,000 camera rays 846 ->
// 178 us; 1M-triangle terrain, 260,000 camera rays 509 -> 188; scene of 1,000
// instances, 390,000 camera rays 4249 -> 857.  The registers leave seven
// waves per SIMD either way (two levels: six, 16 rows fit them).
template <int DEPTH>
constexpr int kPoolRows = DEPTH < 16 ? 16 : DEPTH;
template <int DEPTH>
constexpr int kPoolCapacity = kPoolRows<DEPTH> * 32;  // two words each

// Orders this wave's LDS accesses across lanes for the compiler (the
// hardware keeps a wave's LDS accesses in order).
__device__ __forceinline__ void WaveLdsFence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

__device__ __forceinline__ float ReadLaneF(float v, int l) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), l));
}

// How many subtrees a lane has left: its stack, current node and postponed leaf.
__device__ __forceinline__ uint32_t PoolOwn(uint32_t sp, uint32_t node, uint32_t leaf, uint32_t rid) {
    return rid != kInvalid ? sp + (node != kInvalid) + (leaf != kInvalid) : 0u;
}

// Inclusive prefix sum over the lanes of a wave.
__device__ __forceinline__ uint32_t WavePrefixSum(uint32_t v) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(v, o, 64);
        if (__lane_id() >= (uint32_t)o) v += y;
    }
    return v;
}

// Whether what the lanes have left fits into a pool, with room to work:
// without SPILLED, only what no lane spilled to scratch.  Every lane of the
// wave calls it.
template <bool SPILLED, int DEPTH>
__device__ __forceinline__ bool PoolFits(const LaneStack<DEPTH>& st, uint32_t node, uint32_t leaf, uint32_t rid) {
    if (!SPILLED && __any(rid != kInvalid && st.gbase != 0)) return false;
    const uint32_t sum = WavePrefixSum(PoolOwn((uint32_t)st.sp, node, leaf, rid));
    return (uint32_t)__builtin_amdgcn_readlane((int)sum, 63) + kPoolReserve <= (uint32_t)kPoolCapacity<DEPTH>;
}

// A pool shorter than this goes on with as many rays as it has (PoolPush); a
// longer one finishes some first, or it would outgrow its room and shrink to
// few entries a step (64 long rays a wave: a batch of 32 requests 1240 us,
// without this limit 1300; a quarter or three quarters of the room instead
// of half: 262,144 camera rays over the terrain 215 and 143 against 154 us,
// the 1,000-instance scene 1073 and 1408 against 1084).
template <int DEPTH>
constexpr uint32_t kPoolWide = (kPoolCapacity<DEPTH> - kPoolReserve) / 2;

// The single-level kernel pools what its eight-entry stacks spilled: with a
// tree deeper than they are, some lane nearly always has spilled (1M-triangle
// terrain, 2M camera rays, closest / any: 585/561 us without, 367/330 with;
// 300,000 rays from anywhere in the unit cube 187/170 and 99/98).
template <int DEPTH>
constexpr bool kPoolSpilled = DEPTH < 16;

// Turns the wave's stacks into the pool, in place: lane 0's entries on top,
// each lane's in the order of its stack (a short pool: every ray's first
// entry above everyone's others).  Returns the number of entries.
template <bool SPILLED, int DEPTH>
__device__ __forceinline__ uint32_t PoolFromStacks(const LaneStack<DEPTH>& st, uint32_t node, uint32_t leaf, uint32_t rid) {
    const uint32_t lane = __lane_id();
    const uint32_t sp = (uint32_t)st.sp, entries = rid != kInvalid ? sp : 0u;
    const uint32_t spilled = SPILLED && rid != kInvalid ? (uint32_t)st.gbase : 0u;
    uint32_t sum = WavePrefixSum(PoolOwn(sp, node, leaf, rid));
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)sum, 63);
    const bool lead = total < kPoolWide<DEPTH> && rid != kInvalid && (node != kInvalid || leaf != kInvalid);
    const uint64_t leads = __ballot(lead);
    sum -= RankIn(leads) + (lead ? 1u : 0u);
    const uint32_t rest = total - (uint32_t)__popcll(leads);
    uint32_t row[DEPTH];
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) row[i] = st.lds[i][lane];
    WaveLdsFence();
    uint2* pool = reinterpret_cast<uint2*>(st.lds);
    uint2* at = pool + (rest - sum);
    for (uint32_t i = 0; i < spilled; ++i) at[i] = make_uint2(LdG(st.slot((int)i)), lane | i << kPoolSlotBits);
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
        __builtin_amdgcn_sched_barrier(0);  // one entry's second word at a time in registers
        const uint32_t e = spilled + (((uint32_t)i - spilled) & (uint32_t)(DEPTH - 1));  // the entry in row i
        if (e < entries) at[e] = make_uint2(row[i], lane | e << kPoolSlotBits);
    }
    at += entries;
    const uint32_t word = lane | entries << kPoolSlotBits;
    if (rid != kInvalid && node != kInvalid && (leaf != kInvalid || !lead)) *at++ = make_uint2(node, word);
    if (rid != kInvalid && leaf != kInvalid && !lead) *at = make_uint2(leaf, word);
    if (lead) pool[total - 1 - RankIn(leads)] = make_uint2(leaf != kInvalid ? leaf : node, word);
    WaveLdsFence();
    return total;
}

// Pushes a step's children: on top the first one of each ray (closest hit:
// every near child), so that the next step goes on with as many rays as
// there are, and their far children are left until the near ones are done
// and may have made them needless; below them the rest, in the order of the
// entries they came from.  A ray's own entries stay in depth-first order
// (closest hit does not need it).  With the list half full, all in order:
// that keeps it short.
template <bool CLOSEST>
__device__ __forceinline__ void PoolPush(uint2* pool, uint32_t& count, uint32_t wide, uint32_t* first, uint32_t step, int slot,
                                         uint32_t near, uint32_t near_word, uint32_t far, uint32_t far_word) {
    const uint32_t lane = __lane_id();
    bool lead = false;
    if (count < wide) {
        lead = near != kInvalid;
        if (!CLOSEST) {
            // The lowest lane with a child of this ray.
            const uint32_t key = step << 6 | (63u - lane);
            if (lead) atomicMax(&first[slot], key);
            WaveLdsFence();
            lead = lead && first[slot] == key;
        }
    }
    const uint64_t m0 = __ballot(lead), m1 = __ballot(near != kInvalid && !lead), m2 = __ballot(far != kInvalid);
    const uint32_t rest = count + (uint32_t)(__popcll(m1) + __popcll(m2));
    const uint32_t below = RankIn(m1) + RankIn(m2);
    if (near != kInvalid) {
        const uint32_t at = lead ? rest + (uint32_t)__popcll(m0) - 1 - RankIn(m0) : rest - 1 - below;
        pool[at] = make_uint2(near, near_word);
    }
    if (far != kInvalid) pool[rest - 1 - below - (near != kInvalid && !lead ? 1u : 0u)] = make_uint2(far, far_word);
    WaveLdsFence();
    count = rest + (uint32_t)__popcll(m0);
}

// A lane's best hit while the pool is worked on (in LDS: read and written
// only when a triangle is hit).
struct PoolHits {
    float t[64];  // any hit: the hit's distance (the ray's best_t stays its t_max)
    float u[64], v[64];
    uint32_t prim[64];
    uint32_t first[64];  // PoolPush
};

// The geometry a pool's entries belong to: one for the launch, or (batched
// queries) the one of the lane that holds the ray.
struct PoolBvh {
    const BvhNode* nodes;
    uint32_t n_int, total;
    bool boxes, any;
};
enum PoolKind : int { kPoolClosest = 0, kPoolAny = 1, kPoolPerLane = 2 };

// Visits the pool's entries until none is left.  best_t: the distance of the
// best hit of this lane's ray (its t_max while it has none, and throughout
// for any hit); best.prim starts as the best hit so far.
template <int KIND, int DEPTH>
__device__ __forceinline__ void PoolTraverse(uint2* pool, uint32_t count, const PoolBvh& bvh, const RayState& own,
                                             float& best_t, PoolHits& best, uint32_t* first, uint32_t* err) {
    const uint32_t lane = __lane_id();
    uint32_t step = 0;
    if (KIND != kPoolClosest) {
        first[lane] = 0;
        WaveLdsFence();
    }
    constexpr uint32_t kRoom = kPoolCapacity<DEPTH> - kPoolReserve;
    constexpr uint32_t kSlotMask = (1u << kPoolSlotBits) - 1;
    while (count) {
        const uint32_t take = min(min(count, 64u), count < kRoom ? kRoom - count : 1u);
        count -= take;
        uint2 e = make_uint2(kInvalid, lane);
        if (lane < take) e = pool[count + take - 1 - lane];
        WaveLdsFence();
        const int slot = (int)(e.y & kSlotMask);
        const BvhNode* nodes = bvh.nodes;
        uint32_t n_int = bvh.n_int, total = bvh.total;
        bool boxes = bvh.boxes, any = KIND == kPoolAny;
        if (KIND == kPoolPerLane) {
            const uint64_t own_nodes = reinterpret_cast<uint64_t>(bvh.nodes);
            const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)own_nodes, slot, 64);
            const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(own_nodes >> 32), slot, 64);
            nodes = reinterpret_cast<const BvhNode*>((uint64_t)hi << 32 | lo);
            n_int = (uint32_t)__shfl((int)bvh.n_int, slot, 64);
            total = (uint32_t)__shfl((int)bvh.total, slot, 64);  // the header's count bounds every node, as in the lanes' loop
            const int kinds = __shfl((bvh.boxes ? 1 : 0) | (bvh.any ? 2 : 0), slot, 64);
            boxes = (kinds & 1) != 0;
            any = (kinds & 2) != 0;
        }
        float4 q0, q1, q2, q3;
        if (e.x < total) LoadNode(nodes, e.x, q0, q1, q2, q3);
        RayState r;
        r.ox = __shfl(own.ox, slot, 64); r.oy = __shfl(own.oy, slot, 64); r.oz = __shfl(own.oz, slot, 64);
        r.tmin = __shfl(own.tmin, slot, 64);
        r.ix = __shfl(own.ix, slot, 64); r.iy = __shfl(own.iy, slot, 64); r.iz = __shfl(own.iz, slot, 64);
        const float tbest = __shfl(best_t, slot, 64);
        uint32_t near = kInvalid, far = kInvalid;
        if (e.x < n_int) {
            const uint32_t c0 = __float_as_uint(q0.w), c1 = __float_as_uint(q1.w);
            float ta, tb;
            const float limit = WidenLimit(tbest);
            const bool h0 = SlabTest(r, limit, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, ta);
            const bool h1 = SlabTest(r, limit, q2.x, q2.y, q2.z, q3.x, q3.y, q3.z, tb);
            const bool c1first = h1 && (!h0 || ta > tb);
            if (h0 || h1) near = c1first ? c1 : c0;
            if (h0 && h1) far = c1first ? c0 : c1;
            if (far != kInvalid && (e.y >> kPoolSlotBits) >= (uint32_t)kStackCapacity) {
                // Deeper than the stack: reported, and this part of the ray ends.
                if (err) StG(err + kErrStackOverflow, 1u);
                near = far = kInvalid;
            }
        }
        const bool is_leaf = e.x >= n_int && e.x < total;
        if (__any(is_leaf)) {
            r.sx = __shfl(own.sx, slot, 64); r.sy = __shfl(own.sy, slot, 64); r.sz = __shfl(own.sz, slot, 64);
            r.k = (uint32_t)__shfl((int)own.k, slot, 64);
            TriHit h;
            bool hit = is_leaf && LeafTest(boxes, r, tbest, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, q2.x, q2.y, q2.z, h) &&
                       h.t >= r.tmin && h.t <= tbest;
            uint64_t cancelled = 0;  // any hit: slots whose later entries end
            for (uint64_t m = __ballot(hit); m;) {
                const int f = __builtin_ctzll(m);
                const int o = __builtin_amdgcn_readlane(slot, f);
                const float ft = ReadLaneF(h.t, f);
                const uint32_t fp = (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(q1.w), f);
                const bool any_f = KIND == kPoolPerLane ? __builtin_amdgcn_readlane(any ? 1 : 0, f) != 0 : any;
                const float ot = ReadLaneF(best_t, o);
                // The same for every lane.
                if (any_f || CloserHit(ft, 0u, fp, ot, 0u, best.prim[o])) {
                    if (!any_f && (int)lane == o) best_t = ft;
                    if ((int)lane == f) {
                        if (any_f) best.t[o] = ft;
                        best.u[o] = h.V / h.det;
                        best.v[o] = h.W / h.det;
                        best.prim[o] = fp;
                    }
                    WaveLdsFence();
                }
                m &= m - 1;
                if (any_f) {
                    // Lanes above f hold later entries.
                    if ((int)lane > f && slot == o) {
                        hit = false;
                        near = far = kInvalid;
                    }
                    cancelled |= 1ull << o;
                    m &= __ballot(hit);
                }
            }
            if (KIND != kPoolClosest && cancelled) {
                for (uint32_t i = lane; i < count; i += 64)
                    if ((cancelled >> (pool[i].y & kSlotMask)) & 1ull) pool[i].x = kInvalid;
                WaveLdsFence();
            }
        }
        PoolPush<KIND == kPoolClosest>(pool, count, kPoolWide<DEPTH>, first, ++step, slot, near,
                                       e.y + (far != kInvalid ? 1u << kPoolSlotBits : 0u), far, e.y);
    }
}

template <bool ANY, int OUT, int DEPTH>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(DEPTH <= 16 ? 7 : 4))) void TracePersistentKernel(const uint8_t* __restrict__ accel,
                                                                const float4* __restrict__ rays, uint32_t ray_count,
                                                                const uint32_t* __restrict__ indirect,
                                                                void* __restrict__ hits, uint32_t* __restrict__ scratch,
                                                                uint32_t min_busy, uint32_t fetch, uint32_t init_queues,
                                                                uint32_t* err) {
    __shared__ uint32_t s_stack[kBlock / 64][kPoolRows<DEPTH>][64];
    __shared__ PoolHits s_best[kBlock / 64];
    uint32_t n = ray_count;
    if (indirect) n = min(n, *indirect);
    if (init_queues) InitQueues(scratch, n);
    const AccelHeader* hdr = reinterpret_cast<const AccelHeader*>(accel);
    if (!HeaderIs(hdr, kAccelBlas, err)) return;
    const uint32_t total = hdr->node_count;
    const uint32_t n_int = hdr->prim_count ? hdr->prim_count - 1 : 0;
    const BvhNode* nodes = reinterpret_cast<const BvhNode*>(accel + hdr->nodes_offset);
    const bool boxes = (hdr->flags & kAccelFlagAabbs) != 0;
    uint32_t* counters = scratch;
    const uint32_t lane = __lane_id();
    const uint32_t part = (n + kQueues - 1) / kQueues;

    // Wave-uniform queue state.
    RayQueue rq;
    const bool fixed = StartQueue(rq, n, part, fetch, true, 0);
    bool pooled = false;  // the wave's last rays go on in a pool

    // Lane state.
    uint32_t rid = kInvalid;
    RayState r;
    // best_t starts at the ray's tmax and changes only with best_prim, so on
    // a miss it still holds tmax.  bU, bV: barycentrics of the best hit so
    // far (divided by the determinant when the hit is taken).
    float best_t = 0.0f, bU = 0.0f, bV = 0.0f;
    float any_limit = 0.0f;  // any hit: the culling limit, fixed per ray (the first hit ends the ray)
    uint32_t best_prim = kInvalid;
    uint32_t node = kInvalid, leaf = kInvalid;
    LaneStack<DEPTH> st{s_stack[threadIdx.x / 64], scratch + kQueueHeadWords + SpillStart(fixed, rq.next), err, 0, 0};
    for (;;) {
        // Refill idle lanes.
        const uint64_t idle = __ballot(rid == kInvalid);
        if (idle && !rq.drained) {
            if (rq.next == rq.end) TakeRays(rq, counters, n, part);
            const uint32_t take = min((uint32_t)__popcll(idle), rq.end - rq.next);
            const uint32_t rank = RankIn(idle);
            if (rid == kInvalid && rank < take) {
                rid = rq.next + rank;
                const RayIn ray = LoadRay(rays, rid);
                SetupRay(r, ray.a.x, ray.a.y, ray.a.z, ray.a.w, ray.b.x, ray.b.y, ray.b.z);
                best_t = ray.b.w;
                if (ANY) any_limit = WidenLimit(best_t);
                best_prim = kInvalid;
                bU = 0.0f; bV = 0.0f;
                st.clear();
                node = total ? 0u : kInvalid;
                leaf = kInvalid;
            }
            rq.next += take;
            if (fixed) rq.drained = true;  // a share is at most one ray per lane
        }
        if (__ballot(rid != kInvalid) == 0) {
            if (rq.drained) break;
            continue;
        }
        if (rq.drained && PoolFits<kPoolSpilled<DEPTH>>(st, node, leaf, rid)) {
            pooled = true;
            break;
        }
        if (rid == kInvalid) continue;
        const uint64_t entered = __ballot(1);

        // Traverse until the ray ends or fewer than min_busy lanes are still
        // traversing, then go back and hand new rays to the idle lanes.
        for (;;) {
            // Phase A: inner nodes until every traversing lane has postponed a leaf.
            while (node < n_int) {
                float4 q0, q1, q2, q3;
                LoadNode(nodes, node, q0, q1, q2, q3);
                const uint32_t c0 = __float_as_uint(q0.w);
                const uint32_t c1 = __float_as_uint(q1.w);
                float ta, tb;
                // Closest hit: recomputed (one register fewer across the loop).
                const float limit = ANY ? any_limit : WidenLimit(best_t);
                const bool h0 = SlabTest(r, limit, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, ta);
                const bool h1 = SlabTest(r, limit, q2.x, q2.y, q2.z, q3.x, q3.y, q3.z, tb);
                if (h0 || h1) {
                    const bool c1first = h1 && (!h0 || ta > tb);
                    if (h0 && h1) st.push(c1first ? c0 : c1);
                    node = c1first ? c1 : c0;
                } else {
                    node = st.empty() ? kInvalid : st.pop();
                }
                if (node >= total && node != kInvalid) node = kInvalid;  // corrupt index: end the ray
                if (node != kInvalid && node >= n_int && leaf == kInvalid) {
                    leaf = node;
                    node = st.empty() ? kInvalid : st.pop();
                }
                // Leave for the leaf phase once every descending lane holds a
                // leaf, or once too few lanes are still descending.
                if (!__any(leaf == kInvalid) || (!rq.drained && (uint32_t)__popcll(__ballot(1)) < min_busy)) break;
            }
            // Phase B: the postponed leaf, then any leaves that come next in order.
            if (leaf == kInvalid && node != kInvalid && node >= n_int) {
                leaf = node < total ? node : kInvalid;  // corrupt index: dropped
                node = st.empty() ? kInvalid : st.pop();
            }
            bool finished = false;
            while (leaf != kInvalid) {
                float4 q0, q1, q2, q3;
                LoadNode(nodes, leaf, q0, q1, q2, q3);
                const uint32_t prim = __float_as_uint(q1.w);
                TriHit h;
                if (LeafTest(boxes, r, best_t, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, q2.x, q2.y, q2.z, h) &&
                    h.t >= r.tmin && h.t <= best_t) {
                    if (ANY) {
                        best_t = h.t; best_prim = prim;
                        bU = h.V / h.det; bV = h.W / h.det;
                        finished = true;
                        break;
                    }
                    if (CloserHit(h.t, 0u, prim, best_t, 0u, best_prim)) {
                        best_t = h.t; best_prim = prim;
                        bU = h.V / h.det; bV = h.W / h.det;
                    }
                }
                leaf = kInvalid;
                if (node != kInvalid && node >= n_int && node < total) {
                    leaf = node;
                    node = st.empty() ? kInvalid : st.pop();
                }
            }
            if (finished || (node == kInvalid && leaf == kInvalid)) {
                node = kInvalid;
                leaf = kInvalid;
                const bool hit = best_prim != kInvalid;
                WriteHit<OUT, false>(hits, rid, hit, hit ? bU : 0.0f, hit ? bV : 0.0f, 0u, best_prim,
                                     best_t, best_t);
                rid = kInvalid;
                break;
            }
            if (!rq.drained && (uint32_t)__popcll(__ballot(1)) < min_busy) break;  // refill (nothing left once rq.drained)
            // Drained, but the pool had no room: try again once a lane is done.
            if (rq.drained && __ballot(1) != entered) break;
        }
    }
    // The wave's last rays.
    if (pooled) {
        const uint32_t count = PoolFromStacks<kPoolSpilled<DEPTH>>(st, node, leaf, rid);
        PoolHits& best = s_best[threadIdx.x / 64];
        best.u[lane] = bU;
        best.v[lane] = bV;
        best.prim[lane] = best_prim;
        WaveLdsFence();
        PoolTraverse<ANY ? kPoolAny : kPoolClosest, DEPTH>(reinterpret_cast<uint2*>(st.lds), count,
                                                           PoolBvh{nodes, n_int, total, boxes, ANY}, r, best_t, best, best.first, err);
        if (rid != kInvalid) {
            best_prim = best.prim[lane];
            const bool hit = best_prim != kInvalid;
            WriteHit<OUT, false>(hits, rid, hit, hit ? best.u[lane] : 0.0f, hit ? best.v[lane] : 0.0f, 0u, best_prim,
                                 ANY && hit ? best.t[lane] : best_t, best_t);
        }
    }
}

// ---------------------------------------------------------------------------
// Persistent two-level traversal: the single-level kernel's ray queues and
// while-while loop over a TLAS whose leaves are instances.  A lane that
// reaches an instance leaf enters it at once (world ray to object space,
// sentinel pushed, BLAS root next; isect_2l.comp:222-237).  Triangle leaves
// are postponed as in the single-level kernel, and a lane never pops the
// sentinel (leaves the instance) while it holds a postponed leaf, so every
// leaf is tested against its own instance's ray and nodes, and leaves are
// still tested in depth-first order: closest and any hits are those of the
// plain kernel.  Inner nodes and leaves are told apart by index (inner nodes
// [0, N-1), leaves [N-1, 2N-1) at both levels).

// Pooled traversal of a scene (see the single-level pool): an entry's second
// word also names the instance it lies in (kPoolWorld: the scene's own
// level).  The world ray is in LDS already; an entry inside an instance
// transforms it again, as entering the instance does, so each step costs
// that and one more dependent load (the instance's BLAS address), against
// one step per node of a ray's whole chain.  A scene of 1,000 instances of 2,000-triangle soups built and
// traced: 262,144 any-hit rays 1.70 -> 1.08 ms, 40,000 closest-hit rays
// 1.44 -> 0.46 ms.
constexpr uint32_t kPoolDepthBits = 7;
constexpr uint32_t kPoolInstShift = kPoolSlotBits + kPoolDepthBits;
constexpr uint32_t kPoolWorld = (1u << (32 - kPoolInstShift)) - 1;  // and the number of instances a pool can name
static_assert(kStackCapacity < (1 << kPoolDepthBits), "an entry's depth fits its field");

// As PoolFromStacks: entries above the sentinel lie in the lane's instance,
// those below in the scene; the sentinel itself, and an index past its
// level's nodes (corrupt buffer), becomes an entry without a node.
template <int DEPTH>
__device__ __forceinline__ uint32_t PoolFromStacks2L(uint32_t (*lds)[64], uint32_t sp, uint32_t node, uint32_t leaf,
                                                     uint32_t rid, uint32_t inst, uint32_t top_total,
                                                     uint32_t cur_total) {
    const uint32_t lane = __lane_id();
    const uint32_t entries = rid != kInvalid ? sp : 0u;
    uint32_t sum = WavePrefixSum(PoolOwn(sp, node, leaf, rid));
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)sum, 63);
    const bool lead = total < kPoolWide<DEPTH> && rid != kInvalid && (node != kInvalid || leaf != kInvalid);
    const uint64_t leads = __ballot(lead);
    sum -= RankIn(leads) + (lead ? 1u : 0u);
    const uint32_t rest = total - (uint32_t)__popcll(leads);
    uint32_t row[DEPTH];
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) row[i] = lds[i][lane];
    WaveLdsFence();
    uint2* at = reinterpret_cast<uint2*>(lds) + (rest - sum);
    uint32_t level = lane | kPoolWorld << kPoolInstShift, limit = top_total;
    const uint32_t in = lane | (inst == kInvalid ? kPoolWorld : inst) << kPoolInstShift;
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
        __builtin_amdgcn_sched_barrier(0);
        if ((uint32_t)i < entries) {
            const bool sentinel = row[i] == kTopLevelSentinel;
            at[i] = make_uint2(row[i] < limit ? row[i] : kInvalid, level | (uint32_t)i << kPoolSlotBits);
            if (sentinel) {
                level = in;
                limit = cur_total;
            }
        }
    }
    at += entries;
    const uint32_t word = in | entries << kPoolSlotBits;
    const uint32_t top = node == kTopLevelSentinel ? kInvalid : node;
    if (rid != kInvalid && node != kInvalid && (leaf != kInvalid || !lead)) *at++ = make_uint2(top, word);
    if (rid != kInvalid && leaf != kInvalid && !lead) *at = make_uint2(leaf, word);
    if (lead) reinterpret_cast<uint2*>(lds)[total - 1 - RankIn(leads)] = make_uint2(leaf != kInvalid ? leaf : top, word);
    WaveLdsFence();
    return total;
}

struct PoolScene {
    const BvhNode* nodes;
    const Transform* xforms;
    const uint64_t* blas_table;
    uint32_t total, prims;
};

template <bool ANY, int DEPTH>
__device__ __forceinline__ void PoolTraverse2L(uint2* pool, uint32_t count, const PoolScene& top, const float (*world)[kBlock],
                                               float tmin, float& best_t, float& hit_t, float& bu, float& bv,
                                               uint32_t& best_prim, uint32_t& best_inst, uint32_t* first, uint32_t* err) {
    const uint32_t lane = __lane_id();
    uint32_t step = 0;
    if (ANY) {
        first[lane] = 0;
        WaveLdsFence();
    }
    const uint32_t wave0 = threadIdx.x & ~63u;
    constexpr uint32_t kRoom = kPoolCapacity<DEPTH> - kPoolReserve;
    constexpr uint32_t kSlotMask = (1u << kPoolSlotBits) - 1, kDepthMask = (1u << kPoolDepthBits) - 1;
    while (count) {
        const uint32_t take = min(min(count, 64u), count < kRoom ? kRoom - count : 1u);
        count -= take;
        uint2 e = make_uint2(kInvalid, lane);
        if (lane < take) e = pool[count + take - 1 - lane];
        WaveLdsFence();
        const int slot = (int)(e.y & kSlotMask);
        const uint32_t inst = e.y >> kPoolInstShift;
        const uint32_t w = wave0 + (uint32_t)slot;
        RayState r;
        r.tmin = __shfl(tmin, slot, 64);
        const float tbest = __shfl(best_t, slot, 64);
        float4 q0, q1, q2, q3;
        uint32_t near = kInvalid, far = kInvalid, next = e.y;  // next: level of the children
        bool hit = false;
        TriHit h;
        if (e.x != kInvalid) {
            uint32_t total = top.total, flags = 0;
            r.ox = world[0][w]; r.oy = world[1][w]; r.oz = world[2][w];
            if (inst != kPoolWorld) {
                const float4* xp = reinterpret_cast<const float4*>(top.xforms + 2 * (size_t)inst);
                const float4 x0 = LdG4(xp), x1 = LdG4(xp + 1), x2 = LdG4(xp + 2);
                const uint8_t* blas = reinterpret_cast<const uint8_t*>(LdG(top.blas_table + inst));
                const AccelHeader* bh = reinterpret_cast<const AccelHeader*>(blas);
                total = LdG(&bh->node_count);
                flags = LdG(&bh->flags);
                const uint64_t offset = LdG(&bh->nodes_offset);
                // The builders put the nodes right behind the header: fetched
                // together with it, and again only if it says that they lie
                // further on (so the first read is inside the buffer too).
                LoadNode(reinterpret_cast<const BvhNode*>(blas + sizeof(AccelHeader)), e.x, q0, q1, q2, q3);
                if (offset != sizeof(AccelHeader)) LoadNode(reinterpret_cast<const BvhNode*>(blas + offset), e.x, q0, q1, q2, q3);
                const float wox = r.ox, woy = r.oy, woz = r.oz;
                const float wdx = world[3][w], wdy = world[4][w], wdz = world[5][w];
                const float ox = ((x0.x * wox + x0.y * woy) + x0.z * woz) + x0.w;
                const float oy = ((x1.x * wox + x1.y * woy) + x1.z * woz) + x1.w;
                const float oz = ((x2.x * wox + x2.y * woy) + x2.z * woz) + x2.w;
                const float dx = (x0.x * wdx + x0.y * wdy) + x0.z * wdz;
                const float dy = (x1.x * wdx + x1.y * wdy) + x1.z * wdz;
                const float dz = (x2.x * wdx + x2.y * wdy) + x2.z * wdz;
                SetupRay(r, ox, oy, oz, r.tmin, dx, dy, dz);
            } else {
                LoadNode(top.nodes, e.x, q0, q1, q2, q3);
                r.ix = world[6][w]; r.iy = world[7][w]; r.iz = world[8][w];
            }
            const uint32_t c0 = __float_as_uint(q0.w), c1 = __float_as_uint(q1.w);
            if (c0 != kInvalid) {
                float ta, tb;
                const float limit = WidenLimit(tbest);
                const bool h0 = SlabTest(r, limit, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, ta) && c0 < total;
                const bool h1 = SlabTest(r, limit, q2.x, q2.y, q2.z, q3.x, q3.y, q3.z, tb) && c1 < total;
                const bool c1first = h1 && (!h0 || ta > tb);
                if (h0 || h1) near = c1first ? c1 : c0;
                if (h0 && h1) {
                    far = c1first ? c0 : c1;
                    next += 1u << kPoolSlotBits;
                }
            } else if (inst == kPoolWorld) {
                // Instance leaf: its geometry's root, above the sentinel.
                if (c1 < top.prims) {
                    const AccelHeader* bh = reinterpret_cast<const AccelHeader*>(LdG(top.blas_table + c1));
                    if (bh && LdG(&bh->node_count) != 0) {
                        near = 0;
                        next = (e.y & ((1u << kPoolInstShift) - 1)) + (1u << kPoolSlotBits) + (c1 << kPoolInstShift);
                    }
                }
            } else {
                hit = LeafTest((flags & kAccelFlagAabbs) != 0, r, tbest, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, q2.x, q2.y, q2.z,
                               h) && h.t >= r.tmin && h.t <= tbest;
            }
            if (near != kInvalid && next != e.y && ((e.y >> kPoolSlotBits) & kDepthMask) >= (uint32_t)kStackCapacity) {
                // Deeper than the stack: reported, and this part of the ray ends.
                if (err) StG(err + kErrStackOverflow, 1u);
                near = far = kInvalid;
            }
        }
        uint64_t cancelled = 0;  // any hit: slots whose later entries end
        for (uint64_t m = __ballot(hit); m;) {
            const int f = __builtin_ctzll(m);
            const int o = __builtin_amdgcn_readlane(slot, f);
            const float ft = ReadLaneF(h.t, f);
            const float fu = ReadLaneF(h.V, f), fv = ReadLaneF(h.W, f), fd = ReadLaneF(h.det, f);
            const uint32_t fp = (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(q1.w), f);
            const uint32_t fi = (uint32_t)__builtin_amdgcn_readlane((int)inst, f);
            if ((int)lane == o && (ANY || CloserHit(ft, fi, fp, best_t, best_inst, best_prim))) {
                if (ANY) hit_t = ft;
                else best_t = ft;
                best_prim = fp;
                best_inst = fi;
                bu = fu / fd;
                bv = fv / fd;
            }
            m &= m - 1;
            if (ANY) {
                // Lanes above f hold later entries.
                if ((int)lane > f && slot == o) {
                    hit = false;
                    near = far = kInvalid;
                }
                cancelled |= 1ull << o;
                m &= __ballot(hit);
            }
        }
        if (ANY && cancelled) {
            for (uint32_t i = lane; i < count; i += 64)
                if ((cancelled >> (pool[i].y & kSlotMask)) & 1ull) pool[i].x = kInvalid;
            WaveLdsFence();
        }
        PoolPush<!ANY>(pool, count, kPoolWide<DEPTH>, first, ++step, slot, near, next, far, e.y);
    }
}

template <bool ANY, int OUT, int DEPTH>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(DEPTH <= 16 ? 6 : 4))) void TracePersistent2LKernel(const uint8_t* __restrict__ accel,
                                                                  const float4* __restrict__ rays, uint32_t ray_count,
                                                                  const uint32_t* __restrict__ indirect,
                                                                  void* __restrict__ hits,
                                                                  uint32_t* __restrict__ scratch, uint32_t min_busy,
                                                                  uint32_t fetch, uint32_t lone, uint32_t init_queues, uint32_t* err) {
    __shared__ uint32_t s_stack[kBlock / 64][kPoolRows<DEPTH>][64];
    // Each lane's world ray: origin xyz, direction xyz and reciprocal
    // direction, restored without divisions when the lane leaves an
    // instance.  The TLAS level only tests boxes (instance leaves are entered
    // with a fresh set-up), so the watertight shear and axis permutation of
    // the world ray are not kept.
    __shared__ float s_world[9][kBlock];
    __shared__ uint32_t s_first[kBlock / 64][64];  // PoolPush
    uint32_t n = ray_count;
    if (indirect) n = min(n, *indirect);
    if (init_queues) InitQueues(scratch, n);
    const AccelHeader* hdr = reinterpret_cast<const AccelHeader*>(accel);
    if (!HeaderIs(hdr, kAccelTlas, err)) return;
    const uint32_t top_total = hdr->node_count;
    const uint32_t top_prims = hdr->prim_count;
    const uint32_t top_int = top_prims ? top_prims - 1 : 0;
    const BvhNode* top_nodes = reinterpret_cast<const BvhNode*>(accel + hdr->nodes_offset);
    const Transform* xforms = reinterpret_cast<const Transform*>(accel + hdr->transforms_offset);
    const uint64_t* blas_table = reinterpret_cast<const uint64_t*>(accel + hdr->blas_table_offset);
    uint32_t* counters = scratch;
    const uint32_t part = (n + kQueues - 1) / kQueues;

    // Wave-uniform queue state.
    RayQueue rq;
    const bool pools = top_prims < kPoolWorld;
    const bool fixed = StartQueue(rq, n, part, fetch, pools, lone);
    bool pooled = false;  // the wave's last rays go on in a pool

    // Lane state: the ray of the level being traversed (the world ray waits
    // in LDS), the best hit (best_t is the ray's t_max until a hit), and the
    // level (inst == kInvalid at the top).
    uint32_t rid = kInvalid;
    RayState r;
    float best_t = 0.0f, bu = 0.0f, bv = 0.0f;  // the culling limit is WidenLimit(best_t), recomputed per node
    uint32_t best_prim = kInvalid, best_inst = kInvalid;
    uint32_t node = kInvalid, leaf = kInvalid;
    uint32_t inst = kInvalid;
    const BvhNode* cur = top_nodes;
    uint32_t cur_int = top_int, cur_total = top_total;
    bool boxes = false;
    LaneStack<DEPTH> st{s_stack[threadIdx.x / 64], scratch + kQueueHeadWords + SpillStart(fixed, rq.next), err, 0, 0};

    for (;;) {
        // Refill idle lanes.
        const uint64_t idle = __ballot(rid == kInvalid);
        if (idle && !rq.drained) {
            if (rq.next == rq.end) TakeRays(rq, counters, n, part);
            const uint32_t take = min((uint32_t)__popcll(idle), rq.end - rq.next);
            const uint32_t rank = RankIn(idle);
            if (rid == kInvalid && rank < take) {
                rid = rq.next + rank;
                const RayIn ray = LoadRay(rays, rid);
                s_world[0][threadIdx.x] = ray.a.x; s_world[1][threadIdx.x] = ray.a.y; s_world[2][threadIdx.x] = ray.a.z;
                s_world[3][threadIdx.x] = ray.b.x; s_world[4][threadIdx.x] = ray.b.y; s_world[5][threadIdx.x] = ray.b.z;
                SetupRay(r, ray.a.x, ray.a.y, ray.a.z, ray.a.w, ray.b.x, ray.b.y, ray.b.z);
                s_world[6][threadIdx.x] = r.ix; s_world[7][threadIdx.x] = r.iy; s_world[8][threadIdx.x] = r.iz;
                best_t = ray.b.w;
                best_prim = kInvalid;
                best_inst = kInvalid;
                bu = 0.0f; bv = 0.0f;
                st.clear();
                inst = kInvalid;
                cur = top_nodes;
                cur_int = top_int;
                cur_total = top_total;
                boxes = false;
                node = top_total ? 0u : kInvalid;
                leaf = kInvalid;
            }
            rq.next += take;
            if (fixed) rq.drained = true;  // a share is at most one ray per lane
        }
        if (__ballot(rid != kInvalid) == 0) {
            if (rq.drained) break;
            continue;
        }
        if (rq.drained && pools && PoolFits<false>(st, node, leaf, rid)) {
            pooled = true;
            break;
        }
        if (rid == kInvalid) continue;
        const uint64_t entered = __ballot(1);

        for (;;) {
            // Phase A: inner nodes, instance entries and exits, until every
            // traversing lane has postponed a leaf or too few still traverse.
            for (;;) {
                if (node < cur_int) {
                    float4 q0, q1, q2, q3;
                    LoadNode(cur, node, q0, q1, q2, q3);
                    const uint32_t c0 = __float_as_uint(q0.w);
                    const uint32_t c1 = __float_as_uint(q1.w);
                    float ta, tb;
                    const float limit = WidenLimit(best_t);
                    const bool h0 = SlabTest(r, limit, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, ta);
                    const bool h1 = SlabTest(r, limit, q2.x, q2.y, q2.z, q3.x, q3.y, q3.z, tb);
                    if (h0 || h1) {
                        const bool c1first = h1 && (!h0 || ta > tb);
                        if (h0 && h1) st.push(c1first ? c0 : c1);
                        node = c1first ? c1 : c0;
                    } else {
                        node = st.empty() ? kInvalid : st.pop();
                    }
                } else if (inst == kInvalid && node < cur_total) {
                    // Instance leaf: enter it (isect_2l.comp:222-237).
                    // The transform is fetched with the BLAS address, and the BLAS
                    // header's three fields together: two dependent round trips.
                    const uint32_t id = __float_as_uint(LdG4(&top_nodes[node].a0_max_or_v1).w);
                    const uint8_t* blas = nullptr;
                    float4 x0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), x1 = x0, x2 = x0;
                    uint32_t bn = 0, bflags = 0;
                    uint64_t boff = 0;
                    if (id < top_prims) {
                        const float4* xp = reinterpret_cast<const float4*>(xforms + 2 * (size_t)id);
                        x0 = LdG4(xp); x1 = LdG4(xp + 1); x2 = LdG4(xp + 2);
                        blas = reinterpret_cast<const uint8_t*>(LdG(blas_table + id));
                        if (blas) {
                            const AccelHeader* bh = reinterpret_cast<const AccelHeader*>(blas);
                            bn = LdG(&bh->node_count);
                            boff = LdG(&bh->nodes_offset);
                            bflags = LdG(&bh->flags);
                        }
                    }
                    if (bn != 0) {
                        const float wox = s_world[0][threadIdx.x], woy = s_world[1][threadIdx.x], woz = s_world[2][threadIdx.x];
                        const float wdx = s_world[3][threadIdx.x], wdy = s_world[4][threadIdx.x], wdz = s_world[5][threadIdx.x];
                        const float ox = ((x0.x * wox + x0.y * woy) + x0.z * woz) + x0.w;
                        const float oy = ((x1.x * wox + x1.y * woy) + x1.z * woz) + x1.w;
                        const float oz = ((x2.x * wox + x2.y * woy) + x2.z * woz) + x2.w;
                        const float dx = (x0.x * wdx + x0.y * wdy) + x0.z * wdz;
                        const float dy = (x1.x * wdx + x1.y * wdy) + x1.z * wdz;
                        const float dz = (x2.x * wdx + x2.y * wdy) + x2.z * wdz;
                        SetupRay(r, ox, oy, oz, r.tmin, dx, dy, dz);
                        inst = id;
                        cur = reinterpret_cast<const BvhNode*>(blas + boff);
                        cur_total = bn;
                        cur_int = (bn - 1) / 2;
                        boxes = (bflags & kAccelFlagAabbs) != 0;
                        st.push(kTopLevelSentinel);
                        node = 0;
                    } else {
                        node = st.empty() ? kInvalid : st.pop();
                    }
                } else if (node == kTopLevelSentinel && leaf == kInvalid) {
                    // Leave the instance, restore the world ray (isect_2l.comp:278-286).
                    inst = kInvalid;
                    cur = top_nodes;
                    cur_int = top_int;
                    cur_total = top_total;
                    boxes = false;
                    r.ox = s_world[0][threadIdx.x]; r.oy = s_world[1][threadIdx.x]; r.oz = s_world[2][threadIdx.x];
                    r.ix = s_world[6][threadIdx.x]; r.iy = s_world[7][threadIdx.x]; r.iz = s_world[8][threadIdx.x];
                    node = st.empty() ? kInvalid : st.pop();
                } else if (inst != kInvalid && node < cur_total && leaf == kInvalid) {
                    leaf = node;
                    node = st.empty() ? kInvalid : st.pop();
                } else {
                    break;  // a second leaf or the sentinel behind a postponed leaf, or done
                }
                // An index past the level's nodes (corrupt buffer) ends the ray.
                if (node != kInvalid && node != kTopLevelSentinel && node >= cur_total) node = kInvalid;
                if (!__any(leaf == kInvalid) || (!rq.drained && (uint32_t)__popcll(__ballot(1)) < min_busy)) break;
            }
            // Phase B: the postponed leaf, then the leaves that follow it in order.
            if (leaf == kInvalid && inst != kInvalid && node >= cur_int && node < cur_total) {
                leaf = node;
                node = st.empty() ? kInvalid : st.pop();
                if (node != kInvalid && node != kTopLevelSentinel && node >= cur_total) node = kInvalid;
            }
            bool finished = false;
            while (leaf != kInvalid) {
                float4 q0, q1, q2, q3;
                LoadNode(cur, leaf, q0, q1, q2, q3);
                const uint32_t prim = __float_as_uint(q1.w);
                TriHit h;
                if (LeafTest(boxes, r, best_t, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, q2.x, q2.y, q2.z, h) &&
                    h.t >= r.tmin && h.t <= best_t) {
                    if (ANY) {
                        best_t = h.t; best_prim = prim; best_inst = inst;
                        if (OUT != kOutInstanceId) { bu = h.V / h.det; bv = h.W / h.det; }
                        finished = true;
                        break;
                    }
                    if (CloserHit(h.t, inst, prim, best_t, best_inst, best_prim)) {
                        best_t = h.t; best_prim = prim; best_inst = inst;
                        if (OUT != kOutInstanceId) { bu = h.V / h.det; bv = h.W / h.det; }
                    }
                }
                leaf = kInvalid;
                if (node >= cur_int && node < cur_total) {
                    leaf = node;
                    node = st.empty() ? kInvalid : st.pop();
                    if (node != kInvalid && node != kTopLevelSentinel && node >= cur_total) node = kInvalid;
                }
            }
            if (finished || (node == kInvalid && leaf == kInvalid)) {
                const bool hit = best_prim != kInvalid;
                WriteHit<OUT, true>(hits, rid, hit, bu, bv, best_inst,
                                    best_prim, best_t, best_t);
                rid = kInvalid;
                node = kInvalid;
                leaf = kInvalid;
                break;
            }
            if (!rq.drained && (uint32_t)__popcll(__ballot(1)) < min_busy) break;  // refill (nothing left once rq.drained)
            // Drained, but the pool had no room: try again once a lane is done.
            if (rq.drained && pools && __ballot(1) != entered) break;
        }
    }
    // The wave's last rays.
    if (pooled) {
        const uint32_t count = PoolFromStacks2L<DEPTH>(st.lds, (uint32_t)st.sp, node, leaf, rid, inst, top_total,
                                                      cur_total);
        float hit_t = best_t;
        PoolTraverse2L<ANY, DEPTH>(reinterpret_cast<uint2*>(st.lds), count,
                                   PoolScene{top_nodes, xforms, blas_table, top_total, top_prims}, s_world, r.tmin, best_t,
                                   hit_t, bu, bv, best_prim, best_inst, s_first[threadIdx.x / 64], err);
        if (rid != kInvalid)
            WriteHit<OUT, true>(hits, rid, best_prim != kInvalid, bu, bv, best_inst, best_prim, ANY ? hit_t : best_t, best_t);
    }
}

template <bool ANY, bool TWO_LEVEL, bool STATS>
void LaunchOut(OutputKind out, dim3 g, hipStream_t s, const uint8_t* accel, const float4* rays, uint32_t count,
               const uint32_t* indirect, void* hits, uint32_t* scratch, uint32_t* stats) {
    uint32_t* err = DeviceErrorWords();
    switch (out) {
        case kOutFullHit:
            TraceKernel<ANY, kOutFullHit, TWO_LEVEL, STATS><<<g, kBlock, 0, s>>>(accel, rays, count, indirect, hits, scratch, stats, err);
            break;
        case kOutInstanceId:
            TraceKernel<ANY, kOutInstanceId, TWO_LEVEL, STATS><<<g, kBlock, 0, s>>>(accel, rays, count, indirect, hits, scratch, stats, err);
            break;
        default:
            TraceKernel<ANY, kOutFullHitT, TWO_LEVEL, STATS><<<g, kBlock, 0, s>>>(accel, rays, count, indirect, hits, scratch, stats, err);
            break;
    }
}

// ---------------------------------------------------------------------------
// Batched traversal: one persistent launch per level over many requests.
// The host orders the request table as: requests whose address the context
// recorded as a geometry, requests it has no record of, requests recorded as
// a scene.  The geometry kernel walks the chunks of the first two groups and
// the two-level kernel those of the last two; waves take 64-ray chunks from
// the kernel's counter, a chunk belongs to one request (found by binary
// search over first_chunk), and each lane carries its own request's BVH,
// query and output, so lanes of a wave may serve different requests.  An
// unrecorded request's level is read from its header when a wave takes one
// of its chunks, and a request of the other level is skipped whole; a
// recorded request whose header names the other level (the caller put
// another buffer at that address) is reported as a bad buffer and answered
// with misses.  No kernel beyond the two traversals and a one-wave init
// runs per batch: with several streams in flight, a wider helper kernel
// waits for another stream's persistent launch to leave the CUs.

// Each batch kernel's chunk range is cut into kQueues contiguous parts, one
// per XCD as the persistent kernels' rays are: a wave starts on part
// blockIdx % kQueues and moves to the next part once its own is drained, so
// the chunk atomics of different XCDs land on different words (one 128-byte
// line each; kBatch2LCounterWord is the two-level kernel's first, all
// inside the table offset).  One counter for the whole range took every
// wave's atomic on the same address.
constexpr uint32_t kBatchCounterWord = 0, kBatch2LCounterWord = kQueues * kQueueStride;
static_assert(2 * kQueues * kQueueStride * 4 <= kBatchTableOffset, "batch counters inside the head");

// Next chunk of this kernel's range [first, first + count) of the table's
// chunks, as [q_next, q_end) of request q_req; false once every part is
// drained.  `part` is the part the wave takes chunks from and `tries` how many
// parts it found drained; a drained part is never revisited, since its counter
// only grows.  The first chunks of a part go to the waves that start on it,
// one each (`started`), without an atomic and, when there are no more, without
// asking every part for some at the end (2,048 requests of 256 rays, whole
// frame 925 -> 909 us); counters[part * kQueueStride] counts those behind.  An
// unrecorded request (kBatchFlagCheckLevel) of the other level moves the
// part's counter past its chunks, up to the part's end, with one atomicMax.
// The loop ends because every counter only grows.  Wave-uniform: every lane
// calls it.
template <bool TWO_LEVEL>
__device__ __forceinline__ bool NextBatchChunk(const BatchRequest* __restrict__ table, uint32_t requests,
                                               uint32_t chunk, uint32_t first, uint32_t count, uint32_t* counters,
                                               uint32_t lane, bool& started, uint32_t& part, uint32_t& tries,
                                               uint32_t& q_req, uint32_t& q_next, uint32_t& q_end) {
    for (;;) {
        // Part `part` holds chunks [first + p_lo, first + p_hi).
        const uint32_t p_lo = (uint32_t)((uint64_t)count * part / kQueues);
        const uint32_t p_hi = (uint32_t)((uint64_t)count * (part + 1) / kQueues);
        const uint32_t waves = QueueFirst(part, 1, gridDim.x);
        uint32_t* counter = counters + part * kQueueStride;
        uint32_t c = 0;
        if (!started) {
            c = blockIdx.x / kQueues * (kBlock / 64) + threadIdx.x / 64;
            started = true;
        } else if (p_hi - p_lo > waves) {
            if (lane == 0) c = atomicAdd(counter, 1u);
            c = (uint32_t)__builtin_amdgcn_readfirstlane((int)c) + waves;
        } else {
            c = p_hi - p_lo;  // nothing behind the first chunks
        }
        if (c >= p_hi - p_lo) {
            if (++tries == kQueues) return false;
            part = part + 1 == kQueues ? 0 : part + 1;
            continue;
        }
        c += first + p_lo;
        // The last request with first_chunk <= c: each lane looks at one of 64
        // in the range left, so two loads in turn find it among 4,096.
        uint32_t lo = 0, hi = requests;
        while (hi - lo > 1) {
            const uint32_t stride = (hi - lo + 63) / 64;
            const uint32_t at = lo + lane * stride;
            const uint64_t before = __ballot(at < hi && table[at < hi ? at : lo].first_chunk <= c);
            const uint32_t k = before ? (uint32_t)(__popcll(before) - 1) : 0u;
            hi = min(hi, lo + (k + 1) * stride);
            lo += k * stride;
        }
        lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
        if (table[lo].flags & kBatchFlagCheckLevel) {
            const AccelHeader* hdr = reinterpret_cast<const AccelHeader*>(table[lo].accel);
            const bool scene = LdG(&hdr->magic) == kAccelMagic && LdG(&hdr->kind) == kAccelTlas;
            if (scene != TWO_LEVEL) {
                const uint32_t next = lo + 1 < requests ? table[lo + 1].first_chunk : first + count;
                const uint32_t to = min(next, first + p_hi) - (first + p_lo);
                if (lane == 0 && to > waves) atomicMax(counter, to - waves);
                continue;
            }
        }
        q_req = lo;
        q_next = (c - table[lo].first_chunk) * chunk;
        q_end = min(q_next + chunk, table[lo].ray_count);
        return true;
    }
}

// The output record of ray `i` of request `req`.
template <bool TWO_LEVEL>
__device__ __forceinline__ void WriteBatchHit(const BatchRequest* __restrict__ table, uint32_t req, uint32_t flags, uint32_t i,
                                              bool hit, float u, float v, uint32_t inst, uint32_t prim, float t, float tmax) {
    void* out = reinterpret_cast<void*>(table[req].hits);
    switch ((flags >> 1) & 3u) {
        case kOutFullHit: WriteHit<kOutFullHit, TWO_LEVEL>(out, i, hit, u, v, inst, prim, t, tmax); break;
        case kOutInstanceId: WriteHit<kOutInstanceId, TWO_LEVEL>(out, i, hit, u, v, inst, prim, t, tmax); break;
        default: WriteHit<kOutFullHitT, TWO_LEVEL>(out, i, hit, u, v, inst, prim, t, tmax); break;
    }
}

__global__ __launch_bounds__(kBlock) void TraceBatchKernel(const BatchRequest* __restrict__ table, uint32_t requests,
                                                           uint32_t first_chunk, uint32_t chunk_count,
                                                           uint32_t* __restrict__ head, uint32_t* __restrict__ spill,
                                                           uint32_t min_busy, uint32_t chunk, uint32_t* err) {
    __shared__ uint32_t s_stack[kBlock / 64][kLdsStackEntries][64];
    __shared__ PoolHits s_best[kBlock / 64];
    uint32_t* counter = head + kBatchCounterWord;
    const uint32_t lane = __lane_id();

    // Wave-uniform queue: rays [q_next, q_end) of request q_req.
    uint32_t q_req = 0, q_next = 0, q_end = 0;
    uint32_t part = blockIdx.x % kQueues, tries = 0;  // this wave's chunk part, parts found drained
    bool started = false;
    bool drained = false, pooled = false;  // pooled: the wave's last rays go on in a pool

    // Lane state.
    uint32_t rid = kInvalid, lreq = 0, lflags = 0, n_int = 0, total = 0;
    bool boxes = false;
    const BvhNode* nodes = nullptr;
    RayState r;
    float best_t = 0.0f, bu = 0.0f, bv = 0.0f;  // best_t is t_max until a hit; culling limit WidenLimit(best_t)
    uint32_t best_prim = kInvalid;
    uint32_t node = kInvalid, leaf = kInvalid;
    LaneStack<> st{s_stack[threadIdx.x / 64], spill + (size_t)(blockIdx.x * kBlock + (threadIdx.x & ~63u)) * kSpillEntries, err, 0, 0};

    for (;;) {
        const uint64_t idle = __ballot(rid == kInvalid);
        if (idle && !drained) {
            if (q_next == q_end)
                drained = !NextBatchChunk<false>(table, requests, chunk, first_chunk, chunk_count, counter, lane, started, part, tries,
                                                 q_req, q_next, q_end);
            const uint32_t take = drained ? 0u : min((uint32_t)__popcll(idle), q_end - q_next);
            const uint32_t rank = RankIn(idle);
            if (rid == kInvalid && rank < take) {
                rid = q_next + rank;
                lreq = q_req;
                const BatchRequest& rq = table[q_req];
                lflags = rq.flags;
                const uint8_t* accel = reinterpret_cast<const uint8_t*>(rq.accel);
                const AccelHeader* hdr = reinterpret_cast<const AccelHeader*>(accel);
                total = LdG(&hdr->node_count);
                if (LdG(&hdr->magic) != kAccelMagic || LdG(&hdr->kind) != kAccelBlas) {
                    // Not a geometry (no valid header, or a scene at an
                    // address recorded as a geometry): report it, answer misses.
                    if (err) StG(err + kErrBadAccel, 1u);
                    total = 0;
                }
                const uint32_t prims = LdG(&hdr->prim_count);
                n_int = (prims && total) ? prims - 1 : 0;
                nodes = reinterpret_cast<const BvhNode*>(accel + LdG(&hdr->nodes_offset));
                boxes = (LdG(&hdr->flags) & kAccelFlagAabbs) != 0;
                const RayIn ray = LoadRay(reinterpret_cast<const float4*>(rq.rays), rid);
                SetupRay(r, ray.a.x, ray.a.y, ray.a.z, ray.a.w, ray.b.x, ray.b.y, ray.b.z);
                best_t = ray.b.w;
                best_prim = kInvalid;
                bu = 0.0f; bv = 0.0f;
                st.clear();
                node = total ? 0u : kInvalid;
                leaf = kInvalid;
            }
            q_next += take;
        }
        if (__ballot(rid != kInvalid) == 0) {
            if (drained) break;
            continue;
        }
        if (drained && PoolFits<false>(st, node, leaf, rid)) {
            pooled = true;
            break;
        }
        if (rid == kInvalid) continue;
        const uint64_t entered = __ballot(1);

        const bool any = (lflags & 1u) != 0;
        for (;;) {
            while (node < n_int) {
                float4 q0, q1, q2, q3;
                LoadNode(nodes, node, q0, q1, q2, q3);
                const uint32_t c0 = __float_as_uint(q0.w);
                const uint32_t c1 = __float_as_uint(q1.w);
                float ta, tb;
                const float limit = WidenLimit(best_t);
                const bool h0 = SlabTest(r, limit, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, ta);
                const bool h1 = SlabTest(r, limit, q2.x, q2.y, q2.z, q3.x, q3.y, q3.z, tb);
                if (h0 || h1) {
                    const bool c1first = h1 && (!h0 || ta > tb);
                    if (h0 && h1) st.push(c1first ? c0 : c1);
                    node = c1first ? c1 : c0;
                } else {
                    node = st.empty() ? kInvalid : st.pop();
                }
                if (node >= total && node != kInvalid) node = kInvalid;
                if (node != kInvalid && node >= n_int && leaf == kInvalid) {
                    leaf = node;
                    node = st.empty() ? kInvalid : st.pop();
                }
                if (!__any(leaf == kInvalid) || (!drained && (uint32_t)__popcll(__ballot(1)) < min_busy)) break;
            }
            if (leaf == kInvalid && node != kInvalid && node >= n_int) {
                leaf = node < total ? node : kInvalid;  // corrupt index: dropped
                node = st.empty() ? kInvalid : st.pop();
            }
            bool finished = false;
            while (leaf != kInvalid) {
                float4 q0, q1, q2, q3;
                LoadNode(nodes, leaf, q0, q1, q2, q3);
                const uint32_t prim = __float_as_uint(q1.w);
                TriHit h;
                if (LeafTest(boxes, r, best_t, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, q2.x, q2.y, q2.z, h) &&
                    h.t >= r.tmin && h.t <= best_t) {
                    if (any) {
                        best_t = h.t; best_prim = prim;
                        bu = h.V / h.det; bv = h.W / h.det;
                        finished = true;
                        break;
                    }
                    if (CloserHit(h.t, 0u, prim, best_t, 0u, best_prim)) {
                        best_t = h.t; best_prim = prim;
                        bu = h.V / h.det; bv = h.W / h.det;
                    }
                }
                leaf = kInvalid;
                if (node != kInvalid && node >= n_int && node < total) {
                    leaf = node;
                    node = st.empty() ? kInvalid : st.pop();
                }
            }
            if (finished || (node == kInvalid && leaf == kInvalid)) {
                const bool hit = best_prim != kInvalid;
                WriteBatchHit<false>(table, lreq, lflags, rid, hit, bu, bv, 0u, best_prim, best_t, best_t);  // a miss leaves best_t at t_max
                rid = kInvalid;
                node = kInvalid;
                leaf = kInvalid;
                break;
            }
            if (!drained && (uint32_t)__popcll(__ballot(1)) < min_busy) break;  // refill (nothing left once drained)
            // Drained, but the pool had no room: try again once a lane is done.
            if (drained && __ballot(1) != entered) break;
        }
    }
    // The wave's last rays.
    if (pooled) {
        const uint32_t count = PoolFromStacks<false>(st, node, leaf, rid);
        PoolHits& best = s_best[threadIdx.x / 64];
        best.u[lane] = bu;
        best.v[lane] = bv;
        best.prim[lane] = best_prim;
        WaveLdsFence();
        PoolTraverse<kPoolPerLane, kLdsStackEntries>(reinterpret_cast<uint2*>(st.lds), count,
                                                     PoolBvh{nodes, n_int, total, boxes, (lflags & 1u) != 0}, r, best_t,
                                                     best, best.first, err);
        if (rid != kInvalid) {
            best_prim = best.prim[lane];
            const bool hit = best_prim != kInvalid;
            WriteBatchHit<false>(table, lreq, lflags, rid, hit, hit ? best.u[lane] : 0.0f, hit ? best.v[lane] : 0.0f, 0u,
                                 best_prim, (lflags & 1u) && hit ? best.t[lane] : best_t, best_t);
        }
    }
}

// The two-level batch kernel: the scene requests of the table, with the
// persistent two-level kernel's loop (instances entered at once, the world
// ray in LDS, postponed leaves, the sentinel never popped while a leaf is
// postponed), so each request's hits equal a TracePersistent2LKernel launch
// of its own.  Per lane: the request's TLAS (its header is re-read on
// instance entry and exit, which are rare next to node visits), query and
// output.
__global__ __launch_bounds__(kBlock) void TraceBatch2LKernel(const BatchRequest* __restrict__ table, uint32_t requests,
                                                             uint32_t first_chunk, uint32_t chunk_count,
                                                             uint32_t* __restrict__ head, uint32_t* __restrict__ spill,
                                                             uint32_t min_busy, uint32_t chunk, uint32_t* err) {
    __shared__ uint32_t s_stack[kBlock / 64][kLdsStackEntries][64];
    __shared__ float s_world[9][kBlock];  // world ray: origin, direction, reciprocal direction
    uint32_t* counter = head + kBatch2LCounterWord;
    const uint32_t lane = __lane_id();

    // Wave-uniform queue: rays [q_next, q_end) of request q_req.
    uint32_t q_req = 0, q_next = 0, q_end = 0;
    uint32_t part = blockIdx.x % kQueues, tries = 0;  // this wave's chunk part, parts found drained
    bool started = false;
    bool drained = false;

    // Lane state.
    uint32_t rid = kInvalid, lreq = 0, lflags = 0;
    const AccelHeader* top = nullptr;  // this lane's scene
    uint32_t top_int = 0, top_total = 0;
    const BvhNode* cur = nullptr;
    uint32_t cur_int = 0, cur_total = 0, inst = kInvalid;
    bool boxes = false;
    RayState r;
    float best_t = 0.0f, bu = 0.0f, bv = 0.0f;  // best_t is t_max until a hit; culling limit WidenLimit(best_t)
    uint32_t best_prim = kInvalid, best_inst = kInvalid;
    uint32_t node = kInvalid, leaf = kInvalid;
    LaneStack<> st{s_stack[threadIdx.x / 64], spill + (size_t)(blockIdx.x * kBlock + (threadIdx.x & ~63u)) * kSpillEntries, err, 0, 0};

    for (;;) {
        const uint64_t idle = __ballot(rid == kInvalid);
        if (idle && !drained) {
            if (q_next == q_end)
                drained = !NextBatchChunk<true>(table, requests, chunk, first_chunk, chunk_count, counter, lane, started, part, tries,
                                                q_req, q_next, q_end);
            const uint32_t take = drained ? 0u : min((uint32_t)__popcll(idle), q_end - q_next);
            const uint32_t rank = RankIn(idle);
            if (rid == kInvalid && rank < take) {
                rid = q_next + rank;
                lreq = q_req;
                const BatchRequest& rq = table[q_req];
                lflags = rq.flags;
                top = reinterpret_cast<const AccelHeader*>(rq.accel);
                top_total = LdG(&top->node_count);
                if (LdG(&top->magic) != kAccelMagic || LdG(&top->kind) != kAccelTlas) {
                    // A geometry (or no valid header) at an address recorded
                    // as a scene: report it, answer misses.
                    if (err) StG(err + kErrBadAccel, 1u);
                    top_total = 0;
                }
                const uint32_t prims = LdG(&top->prim_count);
                top_int = (prims && top_total) ? prims - 1 : 0;
                const RayIn ray = LoadRay(reinterpret_cast<const float4*>(rq.rays), rid);
                s_world[0][threadIdx.x] = ray.a.x; s_world[1][threadIdx.x] = ray.a.y; s_world[2][threadIdx.x] = ray.a.z;
                s_world[3][threadIdx.x] = ray.b.x; s_world[4][threadIdx.x] = ray.b.y; s_world[5][threadIdx.x] = ray.b.z;
                SetupRay(r, ray.a.x, ray.a.y, ray.a.z, ray.a.w, ray.b.x, ray.b.y, ray.b.z);
                s_world[6][threadIdx.x] = r.ix; s_world[7][threadIdx.x] = r.iy; s_world[8][threadIdx.x] = r.iz;
                best_t = ray.b.w;
                best_prim = kInvalid;
                best_inst = kInvalid;
                bu = 0.0f; bv = 0.0f;
                st.clear();
                inst = kInvalid;
                cur = reinterpret_cast<const BvhNode*>(reinterpret_cast<const uint8_t*>(top) + LdG(&top->nodes_offset));
                cur_int = top_int;
                cur_total = top_total;
                boxes = false;
                node = top_total ? 0u : kInvalid;
                leaf = kInvalid;
            }
            q_next += take;
        }
        if (__ballot(rid != kInvalid) == 0) {
            if (drained) break;
            continue;
        }
        if (rid == kInvalid) continue;

        const bool any = (lflags & 1u) != 0;
        for (;;) {
            // Phase A: inner nodes, instance entries and exits.
            for (;;) {
                if (node < cur_int) {
                    float4 q0, q1, q2, q3;
                    LoadNode(cur, node, q0, q1, q2, q3);
                    const uint32_t c0 = __float_as_uint(q0.w);
                    const uint32_t c1 = __float_as_uint(q1.w);
                    float ta, tb;
                    const float limit = WidenLimit(best_t);
                    const bool h0 = SlabTest(r, limit, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, ta);
                    const bool h1 = SlabTest(r, limit, q2.x, q2.y, q2.z, q3.x, q3.y, q3.z, tb);
                    if (h0 || h1) {
                        const bool c1first = h1 && (!h0 || ta > tb);
                        if (h0 && h1) st.push(c1first ? c0 : c1);
                        node = c1first ? c1 : c0;
                    } else {
                        node = st.empty() ? kInvalid : st.pop();
                    }
                } else if (inst == kInvalid && node < cur_total) {
                    // Instance leaf: enter it (isect_2l.comp:222-237).
                    const uint8_t* base = reinterpret_cast<const uint8_t*>(top);
                    const uint32_t id = __float_as_uint(LdG4(&cur[node].a0_max_or_v1).w);
                    const uint8_t* blas = nullptr;
                    float4 x0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), x1 = x0, x2 = x0;
                    uint32_t bn = 0, bflags = 0;
                    uint64_t boff = 0;
                    if (id < LdG(&top->prim_count)) {
                        const Transform* xforms = reinterpret_cast<const Transform*>(base + LdG(&top->transforms_offset));
                        const uint64_t* blas_table = reinterpret_cast<const uint64_t*>(base + LdG(&top->blas_table_offset));
                        const float4* xp = reinterpret_cast<const float4*>(xforms + 2 * (size_t)id);
                        x0 = LdG4(xp); x1 = LdG4(xp + 1); x2 = LdG4(xp + 2);
                        blas = reinterpret_cast<const uint8_t*>(LdG(blas_table + id));
                        if (blas) {
                            const AccelHeader* bh = reinterpret_cast<const AccelHeader*>(blas);
                            bn = LdG(&bh->node_count);
                            boff = LdG(&bh->nodes_offset);
                            bflags = LdG(&bh->flags);
                        }
                    }
                    if (bn != 0) {
                        const float wox = s_world[0][threadIdx.x], woy = s_world[1][threadIdx.x], woz = s_world[2][threadIdx.x];
                        const float wdx = s_world[3][threadIdx.x], wdy = s_world[4][threadIdx.x], wdz = s_world[5][threadIdx.x];
                        const float ox = ((x0.x * wox + x0.y * woy) + x0.z * woz) + x0.w;
                        const float oy = ((x1.x * wox + x1.y * woy) + x1.z * woz) + x1.w;
                        const float oz = ((x2.x * wox + x2.y * woy) + x2.z * woz) + x2.w;
                        const float dx = (x0.x * wdx + x0.y * wdy) + x0.z * wdz;
                        const float dy = (x1.x * wdx + x1.y * wdy) + x1.z * wdz;
                        const float dz = (x2.x * wdx + x2.y * wdy) + x2.z * wdz;
                        SetupRay(r, ox, oy, oz, r.tmin, dx, dy, dz);
                        inst = id;
                        cur = reinterpret_cast<const BvhNode*>(blas + boff);
                        cur_total = bn;
                        cur_int = (bn - 1) / 2;
                        boxes = (bflags & kAccelFlagAabbs) != 0;
                        st.push(kTopLevelSentinel);
                        node = 0;
                    } else {
                        node = st.empty() ? kInvalid : st.pop();
                    }
                } else if (node == kTopLevelSentinel && leaf == kInvalid) {
                    // Leave the instance, restore the world ray (isect_2l.comp:278-286).
                    inst = kInvalid;
                    cur = reinterpret_cast<const BvhNode*>(reinterpret_cast<const uint8_t*>(top) + LdG(&top->nodes_offset));
                    cur_int = top_int;
                    cur_total = top_total;
                    boxes = false;
                    r.ox = s_world[0][threadIdx.x]; r.oy = s_world[1][threadIdx.x]; r.oz = s_world[2][threadIdx.x];
                    r.ix = s_world[6][threadIdx.x]; r.iy = s_world[7][threadIdx.x]; r.iz = s_world[8][threadIdx.x];
                    node = st.empty() ? kInvalid : st.pop();
                } else if (inst != kInvalid && node < cur_total && leaf == kInvalid) {
                    leaf = node;
                    node = st.empty() ? kInvalid : st.pop();
                } else {
                    break;  // a second leaf or the sentinel behind a postponed leaf, or done
                }
                // An index past the level's nodes (corrupt buffer) ends the ray.
                if (node != kInvalid && node != kTopLevelSentinel && node >= cur_total) node = kInvalid;
                if (!__any(leaf == kInvalid) || (!drained && (uint32_t)__popcll(__ballot(1)) < min_busy)) break;
            }
            // Phase B: the postponed leaf, then the leaves that follow it in order.
            if (leaf == kInvalid && inst != kInvalid && node >= cur_int && node < cur_total) {
                leaf = node;
                node = st.empty() ? kInvalid : st.pop();
                if (node != kInvalid && node != kTopLevelSentinel && node >= cur_total) node = kInvalid;
            }
            bool finished = false;
            while (leaf != kInvalid) {
                float4 q0, q1, q2, q3;
                LoadNode(cur, leaf, q0, q1, q2, q3);
                const uint32_t prim = __float_as_uint(q1.w);
                TriHit h;
                if (LeafTest(boxes, r, best_t, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, q2.x, q2.y, q2.z, h) &&
                    h.t >= r.tmin && h.t <= best_t) {
                    if (any) {
                        best_t = h.t; best_prim = prim; best_inst = inst;
                        bu = h.V / h.det; bv = h.W / h.det;
                        finished = true;
                        break;
                    }
                    if (CloserHit(h.t, inst, prim, best_t, best_inst, best_prim)) {
                        best_t = h.t; best_prim = prim; best_inst = inst;
                        bu = h.V / h.det; bv = h.W / h.det;
                    }
                }
                leaf = kInvalid;
                if (node >= cur_int && node < cur_total) {
                    leaf = node;
                    node = st.empty() ? kInvalid : st.pop();
                    if (node != kInvalid && node != kTopLevelSentinel && node >= cur_total) node = kInvalid;
                }
            }
            if (finished || (node == kInvalid && leaf == kInvalid)) {
                const bool hit = best_prim != kInvalid;
                WriteBatchHit<true>(table, lreq, lflags, rid, hit, bu, bv, best_inst, best_prim, best_t, best_t);  // a miss leaves best_t at t_max
                rid = kInvalid;
                node = kInvalid;
                leaf = kInvalid;
                break;
            }
            if (!drained && (uint32_t)__popcll(__ballot(1)) < min_busy) break;  // refill (nothing left once drained)
        }
    }
}


__global__ void BatchInitKernel(uint32_t* head) {
    if (threadIdx.x < kQueues) {
        head[kBatchCounterWord + threadIdx.x * kQueueStride] = 0;
        head[kBatch2LCounterWord + threadIdx.x * kQueueStride] = 0;
    }
}

}  // namespace

// Spill slots for every lane the launch can have: the persistent kernel runs
// ceil(ray_count / kBlock) blocks at most and hands rays to any of their
// lanes, so the slots are indexed by lane (up to ray_count rounded up to
// kBlock), not by ray.
size_t TraceScratchBytes(uint32_t ray_count) {
    return AlignUp((size_t)kQueueHeadWords * 4 + AlignUp((size_t)ray_count, kBlock) * kSpillEntries * 4, 256);
}

static std::atomic<uint32_t> g_min_busy{0};
uint32_t MinBusyLanes() {
    uint32_t m = g_min_busy.load(std::memory_order_relaxed);
    if (!m) {
        const char* e = std::getenv("RR_TRACE_MIN_BUSY");
        const int v = e ? std::atoi(e) : 0;
        uint32_t expected = 0;
        m = (v >= 1 && v <= 64) ? (uint32_t)v : kDefaultMinBusy;
        if (!g_min_busy.compare_exchange_strong(expected, m, std::memory_order_relaxed)) m = expected;
    }
    return m;
}
void SetMinBusyLanes(uint32_t v) { g_min_busy.store((v >= 1 && v <= 64) ? v : kDefaultMinBusy, std::memory_order_relaxed); }

static std::atomic<uint32_t> g_fetch{kDefaultFetch};
static std::atomic<uint32_t> g_depth{kDefaultLdsStack};
uint32_t RaysPerFetch() { return g_fetch.load(std::memory_order_relaxed); }
bool SetRaysPerFetch(uint32_t v) {
    if (v != 32 && v != 64 && v != 128) return false;
    g_fetch.store(v, std::memory_order_relaxed);
    return true;
}

static std::atomic<uint32_t> g_min_busy_2l{kDefaultMinBusy2L};
static std::atomic<uint32_t> g_fetch_2l{kDefaultFetch2L};
uint32_t MinBusyLanes2L() { return g_min_busy_2l.load(std::memory_order_relaxed); }
bool SetMinBusyLanes2L(uint32_t v) {
    if (v < 1 || v > 64) return false;
    g_min_busy_2l.store(v, std::memory_order_relaxed);
    return true;
}
static std::atomic<uint32_t> g_min_busy_batch{kDefaultMinBusyBatch};
uint32_t MinBusyLanesBatch() { return g_min_busy_batch.load(std::memory_order_relaxed); }
bool SetMinBusyLanesBatch(uint32_t v) {
    if (v < 1 || v > 64) return false;
    g_min_busy_batch.store(v, std::memory_order_relaxed);
    return true;
}
uint32_t RaysPerFetch2L() { return g_fetch_2l.load(std::memory_order_relaxed); }
bool SetRaysPerFetch2L(uint32_t v) {
    if (v != 32 && v != 64 && v != 128) return false;
    g_fetch_2l.store(v, std::memory_order_relaxed);
    return true;
}
uint32_t LdsStackDepth() { return g_depth.load(std::memory_order_relaxed); }
bool SetLdsStackDepth(uint32_t v) {
    if (v != 8 && v != 16 && v != 32) return false;
    g_depth.store(v, std::memory_order_relaxed);
    return true;
}

static std::atomic<uint32_t> g_rays_per_lane{kDefaultRaysPerLane};
uint32_t RaysPerLane() { return g_rays_per_lane.load(std::memory_order_relaxed); }
bool SetRaysPerLane(uint32_t v) {
    if (v > 64) return false;
    g_rays_per_lane.store(v, std::memory_order_relaxed);
    return true;
}

static std::atomic<int> g_trace_mode{-1};
int TraceMode() {
    int m = g_trace_mode.load(std::memory_order_relaxed);
    if (m < 0) {
        const char* e = std::getenv("RR_TRACE_MODE");
        m = (e && std::strcmp(e, "plain") == 0) ? kTraceModePlain : kTraceModePersistent;
        int expected = -1;
        if (!g_trace_mode.compare_exchange_strong(expected, m, std::memory_order_relaxed)) m = expected;
    }
    return m;
}
void SetTraceMode(int mode) { g_trace_mode.store(mode, std::memory_order_relaxed); }

namespace {

// Resident waves of the persistent kernel (queried once per device).
// Resident blocks of `kernel` on the current device (cached per device;
// which = 0 for the single-request kernel, 1 for the batch kernel).
uint32_t ResidentBlocks(const void* kernel, int which) {
    static std::atomic<uint32_t> blocks[8][64];
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (dev < 0 || dev >= 64) dev = 0;
    uint32_t b = blocks[which][dev].load(std::memory_order_relaxed);
    if (!b) {
        int per_cu = 0, cus = 0;
        (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBlock, 0);
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        b = (uint32_t)std::max(1, per_cu * std::max(1, cus));
        blocks[which][dev].store(b, std::memory_order_relaxed);
    }
    return b;
}

// Resident blocks of the single- or two-level persistent kernel with the
// current LDS stack depth (the occupancy depends on its LDS).
uint32_t PersistentBlocks(bool two) {
    if (two) {
        switch (LdsStackDepth()) {
            case 8: return ResidentBlocks(reinterpret_cast<const void*>(&TracePersistent2LKernel<false, kOutFullHit, 8>), 4);
            case 32: return ResidentBlocks(reinterpret_cast<const void*>(&TracePersistent2LKernel<false, kOutFullHit, 32>), 5);
            default: return ResidentBlocks(reinterpret_cast<const void*>(&TracePersistent2LKernel<false, kOutFullHit, 16>), 6);
        }
    }
    switch (LdsStackDepth()) {
        case 8: return ResidentBlocks(reinterpret_cast<const void*>(&TracePersistentKernel<false, kOutFullHit, 8>), 2);
        case 32: return ResidentBlocks(reinterpret_cast<const void*>(&TracePersistentKernel<false, kOutFullHit, 32>), 3);
        default: return ResidentBlocks(reinterpret_cast<const void*>(&TracePersistentKernel<false, kOutFullHit, 16>), 0);
    }
}

// Workgroups a single query of n rays asks for (the caller takes the minimum
// with the resident grid).
//
// shares (queries of their own): up to 64 rays for each of kSharedWaves
// waves per CU, every wave gets an equal share, as few as one, and pools it
// at once (StartQueue, PoolTraverse): rays end after as many steps as the
// tree is deep, so more waves with fewer rays each are faster until the
// SIMDs are full.  Closest / any in microseconds, 65,536-triangle soup,
// rays from inside, one ray per lane before -> equal shares: 1,000 rays
// 202/228 -> 30/31, 16,000 222/287 -> 53/49, 131,072 349/416 -> 129/122;
// 1M-triangle terrain, 131,072 rays 190/206 -> 46/47.  16 waves per CU
// against 24: 262,144 rays from inside the soup 198 against 246, camera rays
// 183 against 150 (terrain: 60 against 63, 145 against 144); 64 rays each
// for up to 28 waves gains as much on some queries (393,216 rays, terrain:
// from inside 112 -> 83) as it loses on others (camera 168 -> 188).  A
// scene's rays are longer: 24 waves per CU (1,000 instances built and
// 262,144 rays traced: 1074 -> 945 us; 300 instances, 180,000 rays: 148 ->
// 118).  The grid may have more lanes than rays (SpillStart); a scene too large
// to pool uses it only for shares of a few rays (kLoneShare).
//
// Otherwise never more than one ray per lane and never more
// than four workgroups per CU (four waves per SIMD) unless 512 x k rays per
// workgroup need more, k the tuned rays per lane (default 2).  Below that
// the single-level kernel takes a workgroup per 256 x k rays, at least one
// per CU; the two-level kernel, whose rays are four times longer, keeps one
// ray per lane.  k = 0: the full grid whenever the rays fill it.
constexpr uint32_t kSharedWaves = 16, kSharedWaves2L = 24;
uint32_t QueryBlocks(uint64_t n, bool two, bool shares = false) {
    const uint64_t one_per_lane = std::max<uint64_t>(1, (n + kBlock - 1) / kBlock);
    const uint32_t k = RaysPerLane();
    if (k == 0) return (uint32_t)std::min<uint64_t>(one_per_lane, UINT32_MAX);
    static std::atomic<uint32_t> cus_of[64];
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (dev < 0 || dev >= 64) dev = 0;
    uint32_t cus = cus_of[dev].load(std::memory_order_relaxed);
    if (!cus) {
        int c = 0;
        (void)hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev);
        cus = (uint32_t)std::max(1, c);
        cus_of[dev].store(cus, std::memory_order_relaxed);
    }
    const uint64_t shared_waves = (uint64_t)cus * (two ? kSharedWaves2L : kSharedWaves);
    if (shares && n <= shared_waves * 64) return (uint32_t)std::min<uint64_t>((n + 3) / 4, shared_waves / 4);
    const uint64_t lo = two ? one_per_lane : (n + (uint64_t)kBlock * k - 1) / ((uint64_t)kBlock * k);
    const uint64_t hi = (n + (uint64_t)kBlock * 2 * k - 1) / ((uint64_t)kBlock * 2 * k);
    const uint64_t b = std::max<uint64_t>({cus, std::min<uint64_t>(4ull * cus, lo), hi});
    return (uint32_t)std::min<uint64_t>({b, one_per_lane, UINT32_MAX});
}

uint32_t BatchBlocks() { return ResidentBlocks(reinterpret_cast<const void*>(&TraceBatchKernel), 1); }
uint32_t Batch2LBlocks() { return ResidentBlocks(reinterpret_cast<const void*>(&TraceBatch2LKernel), 7); }

uint32_t FetchFor(uint32_t n, uint32_t blocks, bool two) {
    return PieceRays(n, blocks, two ? RaysPerFetch2L() : RaysPerFetch());
}

template <bool ANY, bool TWO, int OUT, int DEPTH>
void LaunchPersistentKernel(uint32_t blocks, hipStream_t s, const uint8_t* a, const float4* r, uint32_t n,
                            const uint32_t* ind, void* hits, uint32_t* sc, uint32_t mb, uint32_t f, uint32_t lone,
                            uint32_t init) {
    uint32_t* err = DeviceErrorWords();
    if (TWO) TracePersistent2LKernel<ANY, OUT, DEPTH><<<blocks, kBlock, 0, s>>>(a, r, n, ind, hits, sc, mb, f, lone, init, err);
    else TracePersistentKernel<ANY, OUT, DEPTH><<<blocks, kBlock, 0, s>>>(a, r, n, ind, hits, sc, mb, f, init, err);
}

template <bool ANY, bool TWO, int DEPTH>
void LaunchPersistentDepth(OutputKind out, uint32_t blocks, hipStream_t s, const uint8_t* a, const float4* r,
                           uint32_t n, const uint32_t* ind, void* hits, uint32_t* sc, uint32_t init) {
    // Equal shares take no pieces, unless the scene is too large for a pool.
    const uint32_t lone = TWO ? std::min(blocks, QueryBlocks(n, true)) : blocks;
    const uint32_t mb = TWO ? MinBusyLanes2L() : MinBusyLanes(), f = FetchFor(n, lone, TWO);
    switch (out) {
        case kOutFullHit: LaunchPersistentKernel<ANY, TWO, kOutFullHit, DEPTH>(blocks, s, a, r, n, ind, hits, sc, mb, f, lone, init); break;
        case kOutInstanceId: LaunchPersistentKernel<ANY, TWO, kOutInstanceId, DEPTH>(blocks, s, a, r, n, ind, hits, sc, mb, f, lone, init); break;
        default: LaunchPersistentKernel<ANY, TWO, kOutFullHitT, DEPTH>(blocks, s, a, r, n, ind, hits, sc, mb, f, lone, init); break;
    }
}

// init: this launch (one block) sets the queues up first (see InitQueues).
template <bool ANY, bool TWO>
void LaunchPersistent(OutputKind out, uint32_t blocks, hipStream_t s, const uint8_t* a, const float4* r, uint32_t n,
                      const uint32_t* ind, void* hits, uint32_t* sc, bool init) {
    const uint32_t i = init ? 1u : 0u;
    switch (LdsStackDepth()) {
        case 8: LaunchPersistentDepth<ANY, TWO, 8>(out, blocks, s, a, r, n, ind, hits, sc, i); break;
        case 32: LaunchPersistentDepth<ANY, TWO, 32>(out, blocks, s, a, r, n, ind, hits, sc, i); break;
        default: LaunchPersistentDepth<ANY, TWO, 16>(out, blocks, s, a, r, n, ind, hits, sc, i); break;
    }
}

}  // namespace

void Trace(const void* accel, AccelKind kind, QueryKind query, OutputKind output, const void* rays, uint32_t ray_count,
           const uint32_t* indirect, void* hits, void* scratch, hipStream_t s) {
    if (ray_count == 0) return;
    const uint8_t* a = static_cast<const uint8_t*>(accel);
    const float4* r = static_cast<const float4*>(rays);
    uint32_t* sc = static_cast<uint32_t*>(scratch);
    // Both levels are launched every time: each kernel reads the level from
    // the buffer's header and the one for the other level returns at once.
    // `kind` is the level the context recorded when it built this address;
    // it is only a hint, because the caller may have freed that buffer and
    // put another one (a copy, a build elsewhere) at the same address, so it
    // decides which persistent kernel gets the full grid and which gets one
    // block (all that an exiting kernel needs; a persistent kernel with one
    // block still traces every ray, slowly, if the hint was stale).
    if (TraceMode() != kTraceModePlain) {
        // At most ceil(ray_count / kBlock) blocks: TraceScratchBytes holds
        // spill slots for that many lanes.  The queues are set up once: a
        // kernel of the wrong level returns before touching them.
        // With a recorded level the one-block launch (first) sets the queues
        // up; with none, both grids are full and a QueueInitKernel does.
        const bool recorded = kind != kAccelUnknown;
        if (!recorded) QueueInitKernel<<<1, 64, 0, s>>>(sc, ray_count, indirect);
        const uint32_t b1 = kind == kAccelTlas ? 1u : std::min(PersistentBlocks(false), QueryBlocks(ray_count, false, true));
        const uint32_t b2 = kind == kAccelBlas ? 1u : std::min(PersistentBlocks(true), QueryBlocks(ray_count, true, true));
        // The one-block launch goes first: with other streams' persistent
        // launches holding the CUs it waits as long as the full launch
        // behind it would, instead of delaying the query's end.
        const bool single_first = kind == kAccelTlas;
        for (int k = 0; k < 2; ++k) {
            const bool two = (k == 0) != single_first;
            const uint32_t b = two ? b2 : b1;
            const bool init = recorded && k == 0;
            if (query == kQueryAny) {
                if (two) LaunchPersistent<true, true>(output, b, s, a, r, ray_count, indirect, hits, sc, init);
                else LaunchPersistent<true, false>(output, b, s, a, r, ray_count, indirect, hits, sc, init);
            } else {
                if (two) LaunchPersistent<false, true>(output, b, s, a, r, ray_count, indirect, hits, sc, init);
                else LaunchPersistent<false, false>(output, b, s, a, r, ray_count, indirect, hits, sc, init);
            }
        }
        return;
    }
    // One lane per ray: both grids cover every ray.
    const dim3 g((ray_count + kBlock - 1) / kBlock);
    if (query == kQueryAny) {
        LaunchOut<true, false, false>(output, g, s, a, r, ray_count, indirect, hits, sc, nullptr);
        LaunchOut<true, true, false>(output, g, s, a, r, ray_count, indirect, hits, sc, nullptr);
    } else {
        LaunchOut<false, false, false>(output, g, s, a, r, ray_count, indirect, hits, sc, nullptr);
        LaunchOut<false, true, false>(output, g, s, a, r, ray_count, indirect, hits, sc, nullptr);
    }
}

void TraceWithStats(const void* accel, AccelKind kind, QueryKind query, const void* rays, uint32_t ray_count, void* hits,
                    void* scratch, uint32_t* stats, hipStream_t s) {
    if (ray_count == 0) return;
    const dim3 g((ray_count + kBlock - 1) / kBlock);
    const uint8_t* a = static_cast<const uint8_t*>(accel);
    const float4* r = static_cast<const float4*>(rays);
    uint32_t* sc = static_cast<uint32_t*>(scratch);
    (void)kind;  // a hint only (see Trace): both levels run, the other one returns at once
    uint32_t* err = DeviceErrorWords();
    if (query == kQueryAny) {
        TraceKernel<true, kOutFullHitT, false, true><<<g, kBlock, 0, s>>>(a, r, ray_count, nullptr, hits, sc, stats, err);
        TraceKernel<true, kOutFullHitT, true, true><<<g, kBlock, 0, s>>>(a, r, ray_count, nullptr, hits, sc, stats, err);
    } else {
        TraceKernel<false, kOutFullHitT, false, true><<<g, kBlock, 0, s>>>(a, r, ray_count, nullptr, hits, sc, stats, err);
        TraceKernel<false, kOutFullHitT, true, true><<<g, kBlock, 0, s>>>(a, r, ray_count, nullptr, hits, sc, stats, err);
    }
}

size_t TraceBatchScratchBytes(uint32_t requests, uint64_t total_rays) {
    // The launch has at most one lane per chunked ray, and the chunks of at
    // most kBatchChunkLarge rays number fewer than total_rays / chunk + requests.
    const uint64_t lanes = std::min<uint64_t>((uint64_t)std::max(BatchBlocks(), Batch2LBlocks()) * kBlock,
                                              AlignUp(total_rays + (uint64_t)requests * kBatchChunkLarge, kBlock));
    return kBatchTableOffset + BatchTableBytes(requests) + AlignUp((size_t)lanes * kSpillEntries * 4, 256);
}

void TraceBatch(const BatchRequest* table, uint32_t requests, uint32_t chunk, uint32_t geo_chunks, uint32_t unrecorded_chunks,
                uint32_t scene_chunks, void* scratch, hipStream_t s) {
    if (requests == 0 || geo_chunks + unrecorded_chunks + scene_chunks == 0) return;
    uint8_t* base = static_cast<uint8_t*>(scratch);
    uint32_t* head = reinterpret_cast<uint32_t*>(base);
    auto* spill = reinterpret_cast<uint32_t*>(base + kBatchTableOffset + BatchTableBytes(requests));
    const uint32_t mb = MinBusyLanesBatch();
    BatchInitKernel<<<1, 64, 0, s>>>(head);
    // The geometry kernel takes chunks [0, geo + unrecorded), the two-level
    // kernel [geo, geo + unrecorded + scene); a kernel with no chunk is not
    // launched.  The geometry kernel has a wave per chunk, up to the resident
    // grid: a chunk is pooled by its wave at once, so more waves with fewer
    // chunks each are faster (500 meshes refitted, 256 rays each: 1,024 waves
    // 294 us, 2,000 waves 256; 2,048 meshes and 32 large requests the same
    // either way).  The two-level kernel's is a single query's of the chunks'
    // lanes.
    const uint32_t n1 = geo_chunks + unrecorded_chunks, n2 = unrecorded_chunks + scene_chunks;
    if (n1) {
        const uint32_t b = std::min(BatchBlocks(), (n1 + kBlock / 64 - 1) / (kBlock / 64));
        TraceBatchKernel<<<b, kBlock, 0, s>>>(table, requests, 0u, n1, head, spill, mb, chunk, DeviceErrorWords());
    }
    if (n2) {
        const uint32_t b = std::min(Batch2LBlocks(), QueryBlocks((uint64_t)n2 * chunk, true));
        TraceBatch2LKernel<<<b, kBlock, 0, s>>>(table, requests, geo_chunks, n2, head, spill, MinBusyLanes2L(), chunk,
                                                DeviceErrorWords());
    }
}

}  // namespace rr
