// tree_device.h — the radix tree over sorted Morton codes, built together with
// its boxes, for the single-mesh, batched and scene builders.
//
// The tree is Karras's ("Maximizing Parallelism in the Construction of BVHs,
// Octrees, and k-d Trees", HPG 2012; the reference builds it top-down, one
// binary search per node, lbvh_emit_hierarchy_mesh.comp:85-217, and refits
// it in a second pass, lbvh_fit_aabb_mesh.comp:122-205).  Here it is built
// from its gaps: the gap before key k shares a prefix of delta(k - 1, k)
// bits, each gap is where one node splits, and that node reaches to the next
// gap on either side that shares less (it is the Cartesian tree of the
// deltas).  Its index is the end of its range on the side that its parent
// splits (its last key if it is a left child, its first if it is a right
// one; the root is 0), which is Karras's numbering.
//
// A workgroup takes kTreeWindow consecutive leaves.  Each thread owns a gap,
// finds its node's range in LDS (minima over 1, 2, 4 ... gaps) and reads its
// children's boxes from unions over 1, 2, 4 ... entries: no thread waits for
// another's merge, so the chain up the tree, which bounds a climb (a wave
// passes as often as its longest climb, and each pass is six dependent LDS
// accesses), is gone.  Nodes and leaves go to memory whole and in order
// through LDS.  The few subtrees whose sibling lies outside (about ten per
// window) are published in key order, and the last workgroup of kTreeGroup
// windows does the same with those, and so on up: as many hand-offs between
// workgroups as the logarithm of the windows to base kTreeGroup, rounded up
// (none for one window, one for up to 24,576 leaves, two for up to 1.18M,
// three for up to 56.6M).  Boxes are min and max, so the result does not
// depend on which workgroup merges what.
#pragma once
#include <hip/hip_runtime.h>

#include "build.h"
#include "build_device.h"
#include "rr_device.h"

namespace rr {

constexpr int kTreeWindow = 512;  // threads of a workgroup: one leaf, or one published subtree, each
constexpr uint32_t kTreeGroup = 48;  // about ten published subtrees of each fill a workgroup
// One wave scans a group's counts and gives the sum in one entry more.
static_assert(kTreeGroup < 64, "group_first[children] is written by lane `children`");
// A contiguous run of keys leaves at most this many subtrees unmerged: those
// on one side have strictly decreasing prefixes with what lies beyond, and
// there are at most 60 prefix lengths (30 code bits, then the key position's
// 30).
constexpr uint32_t kTreePending = 128;

// A published subtree: its key range and box.
struct TreePending {
    uint32_t first, last;
    float lo[3], hi[3];
};
static_assert(sizeof(TreePending) == 32, "two 16-byte accesses");

__host__ __device__ inline uint32_t TreeWindows(uint32_t n) { return (n + kTreeWindow - 1) / kTreeWindow; }
// Publishing runs of all levels: windows, groups of windows, groups of those ...
__host__ __device__ inline uint32_t TreeRuns(uint32_t windows) {
    uint32_t t = 0;
    for (uint32_t w = windows; w > 1; w = (w + kTreeGroup - 1) / kTreeGroup) t += w;
    return t + 1;
}
// Scratch of a tree of n leaves: per run an arrival counter (zero before the
// build), an entry count, and its published subtrees.
struct TreeScratch {
    TreePending* pending;
    uint32_t* arrived;
    uint32_t* count;
};
__host__ __device__ inline size_t TreeHeadWords(uint32_t runs) { return AlignUp(size_t(runs), 64); }
inline size_t TreeScratchBytes(uint32_t n) {
    const uint32_t runs = TreeRuns(TreeWindows(n));
    return runs <= 1 ? 0 : TreeHeadWords(runs) * 8 + size_t(runs) * kTreePending * sizeof(TreePending);
}
__host__ __device__ inline TreeScratch CarveTreeScratch(void* base, uint32_t runs) {
    uint32_t* words = static_cast<uint32_t*>(base);
    return TreeScratch{reinterpret_cast<TreePending*>(words + 2 * TreeHeadWords(runs)), words, words + TreeHeadWords(runs)};
}

__device__ __forceinline__ void StoreAgent4(void* p, uint32_t x, uint32_t y, uint32_t z, uint32_t w) {
    RrFloat4V v;
    v.x = __uint_as_float(x); v.y = __uint_as_float(y); v.z = __uint_as_float(z); v.w = __uint_as_float(w);
    asm volatile("global_store_dwordx4 %0, %1, off sc1" RR_STORE_WAIT_STATES : : "v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ TreePending LoadPendingAgent(const TreePending* p) {
    RrFloat4V a, b;
    asm volatile("global_load_dwordx4 %0, %2, off sc1\n\tglobal_load_dwordx4 %1, %2, off offset:16 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(a), "=&v"(b)
                 : "v"(p)
                 : "memory");
    TreePending e;
    e.first = __float_as_uint(a.x); e.last = __float_as_uint(a.y);
    e.lo[0] = a.z; e.lo[1] = a.w; e.lo[2] = b.x;
    e.hi[0] = b.y; e.hi[1] = b.z; e.hi[2] = b.w;
    return e;
}

constexpr int kTreeLevels = 9;  // log2(kTreeWindow)
struct TreeLds {
    // delta_min[k][g]: 1 + the shortest prefix among gaps g .. g + 2^k - 1
    // (0: outside the tree).  Gap g lies before entry g; gap kTreeWindow
    // after the last.
    uint8_t delta_min[kTreeLevels + 1][kTreeWindow + 8];
    // Unions over 2^k entries from entry t, two levels at a time; then the
    // nodes and the leaves on their way to memory.
    union {
        struct {
            float4 lo[2][kTreeWindow], hi[2][kTreeWindow];
        };
        float4 quads[4 * kTreeWindow];
    };
    uint32_t index[kTreeWindow + 1];             // the node split at gap g, kInvalid if it reaches outside
    uint32_t first[kTreeWindow], last[kTreeWindow];  // keys of published subtree t
    uint8_t state[kTreeWindow];                  // of the quads of slot t: 0 none, 1 whole, 2 without the parent link
    uint64_t slot_nodes[kTreeWindow / 64];       // of each 64 slots: address of node 0 of their tree, less the first key
    uint32_t slot_leaves[kTreeWindow / 64];      // ... and leaves less one
    uint32_t wave_pending[kTreeWindow / 64];
    uint32_t group_first[64];
    uint32_t go;
};

// A subtree: entries [a, b] and box.
struct TreeRun {
    uint32_t first, last;
    float lo[3], hi[3];
};
// What a thread's gap splits.
struct TreeNode {
    uint32_t index, a, b, parent;  // parent: kInvalid for the root or if it is not known here
    float4 lo0, hi0, lo1, hi1;     // children's boxes
    bool whole, waits;             // the node lies inside; ... and its parent does not
};

__device__ __forceinline__ float4 Min4(const float4& a, const float4& b) {
    return make_float4(fminf(a.x, b.x), fminf(a.y, b.y), fminf(a.z, b.z), 0.0f);
}
__device__ __forceinline__ float4 Max4(const float4& a, const float4& b) {
    return make_float4(fmaxf(a.x, b.x), fmaxf(a.y, b.y), fmaxf(a.z, b.z), 0.0f);
}

// The gap whose node is the parent of the subtree over entries [a, b]: the
// one beside it that shares more; false for a whole tree.
__device__ __forceinline__ bool ParentGap(const TreeLds& s, uint32_t a, uint32_t b, uint32_t& gap) {
    const uint32_t dl = s.delta_min[0][a], dr = s.delta_min[0][b + 1];
    gap = dl > dr ? a : b + 1;
    return (dl | dr) != 0;
}

// All threads: the node that gap threadIdx.x splits, from the prefixes in
// delta_min[0] and this thread's entry's box (active: it has an entry).  end:
// the last gap whose prefix is set; a node that reaches past it lies outside.
// first(t), last(t): first and last key of entry t.  index[] holds every
// gap's node afterwards.
template <typename First, typename Last>
__device__ __forceinline__ TreeNode FindNode(bool active, uint32_t end, const float lo[3], const float hi[3], const First& first,
                                             const Last& last, TreeLds& s) {
    const uint32_t t = threadIdx.x;
    s.lo[0][t] = make_float4(lo[0], lo[1], lo[2], 0.0f);
    s.hi[0][t] = make_float4(hi[0], hi[1], hi[2], 0.0f);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTreeLevels; ++k) {
        const uint32_t o = t + (1u << k);
        // Past the last gap: nothing is looked up there.
        const uint8_t m = s.delta_min[k][t], y = o <= (uint32_t)kTreeWindow ? s.delta_min[k][o] : (uint8_t)0;
        s.delta_min[k + 1][t] = m < y ? m : y;
        if (t == 0) s.delta_min[k + 1][kTreeWindow] = 0;
        __syncthreads();
    }
    TreeNode nd{};
    const uint32_t d = s.delta_min[0][t];
    // The gaps on either side that share less; none found: the node reaches outside.
    uint32_t l = t, r = t + 1;
#pragma unroll
    for (int k = kTreeLevels - 1; k >= 0; --k) {
        const uint32_t w = 1u << k;
        if (l >= w && s.delta_min[k][l - w] > d) l -= w;
        if (r + w <= (uint32_t)kTreeWindow + 1 && s.delta_min[k][r] > d) r += w;
    }
    nd.whole = active && t > 0 && d != 0 && l > 0 && r <= end;
    nd.a = nd.whole ? l - 1 : t;
    nd.b = nd.whole ? r - 1 : t;
    uint32_t gap = 0;
    const bool has_parent = ParentGap(s, nd.a, nd.b, gap);
    nd.index = !nd.whole ? kInvalid : !has_parent ? 0u : gap == nd.a ? first(nd.a) : last(nd.b);
    s.index[t] = nd.index;
    if (t == 0) s.index[kTreeWindow] = kInvalid;
    // Children's boxes: two overlapping unions each.
    const uint32_t n0 = nd.whole ? t - nd.a : 0, n1 = nd.whole ? nd.b - t + 1 : 0;  // entries of the children
    const int k0 = 31 - __clz(n0 | 1u), k1 = 31 - __clz(n1 | 1u);
    int cur = 0;
#pragma unroll 1
    for (int k = 0;; ++k) {
        if (n0 && k == k0) {
            const uint32_t e = t - (1u << k);
            nd.lo0 = Min4(s.lo[cur][nd.a], s.lo[cur][e]);
            nd.hi0 = Max4(s.hi[cur][nd.a], s.hi[cur][e]);
        }
        if (n1 && k == k1) {
            const uint32_t e = nd.b + 1 - (1u << k);
            nd.lo1 = Min4(s.lo[cur][t], s.lo[cur][e]);
            nd.hi1 = Max4(s.hi[cur][t], s.hi[cur][e]);
        }
        if (k == kTreeLevels - 1) break;
        const uint32_t o = min(t + (1u << k), (uint32_t)kTreeWindow - 1);
        s.lo[cur ^ 1][t] = Min4(s.lo[cur][t], s.lo[cur][o]);
        s.hi[cur ^ 1][t] = Max4(s.hi[cur][t], s.hi[cur][o]);
        cur ^= 1;
        __syncthreads();
    }
    __syncthreads();
    nd.parent = has_parent ? s.index[gap] : kInvalid;
    nd.waits = nd.whole && has_parent && nd.parent == kInvalid;
    return nd;
}

// The links of node nd to its children: a leaf, or the node that ends (left)
// or starts (right) at the split.
__device__ __forceinline__ uint32_t LeftLink(uint32_t n, uint32_t first, uint32_t split) {
    return first == split ? n - 1 + split : split;
}
__device__ __forceinline__ uint32_t RightLink(uint32_t n, uint32_t split, uint32_t last) {
    return last == split + 1 ? n - 1 + last : split + 1;
}

// The quads of all slots with a state, in memory order.  leaves: the slots'
// leaves, else their internal nodes.
__device__ __forceinline__ void StoreQuads(bool leaves, const void* arg, TreeLds& s) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t q = (uint32_t)j * kTreeWindow + threadIdx.x, slot = q / 4, c = slot / 64;
        const uint32_t state = s.state[slot];
        if (state == 0) continue;
        float4* p = RebaseOn<float4>(arg, s.slot_nodes[c]) + 4 * (int64_t)slot + (q & 3u);
        if (leaves) p += 4 * (size_t)s.slot_leaves[c];
        const float4 v = s.quads[q];
        if (state == 2 && (q & 3u) == 2) {
            RrBox3 third;
            third.x = v.x; third.y = v.y; third.z = v.z;
            *reinterpret_cast<RrBox3*>(p) = third;
        } else {
            *p = v;
        }
    }
}

// A window: entry t of this workgroup is leaf `key` of the tree `nodes` of n
// leaves (active), whose quads are q (without the parent link) and whose box
// is lo, hi; slots without a leaf separate trees.  delta_min[0] is set.
// Gives the subtree of this thread that waits for one outside, if it has one.
// `arg`: any global-memory pointer of the launch.
__device__ __forceinline__ bool BuildWindow(BvhNode* nodes, uint32_t n, uint32_t key, bool active, float4 q[4],
                                            const float lo[3], const float hi[3], const void* arg, TreeRun& r, TreeLds& s) {
    const uint32_t t = threadIdx.x;
    s.state[t] = 0;
    if ((t & 63u) == 0) {
        s.slot_nodes[t / 64] = reinterpret_cast<uint64_t>(nodes) + 64 * ((uint64_t)key - t);
        s.slot_leaves[t / 64] = n - 1;
    }
    const uint32_t key0 = key - t;  // wraps; key0 + entry is the entry's key within this thread's tree
    auto at = [key0](uint32_t e) { return key0 + e; };
    const TreeNode nd = FindNode(active, kTreeWindow, lo, hi, at, at, s);
    // Internal nodes.
    if (nd.whole) {
        const uint32_t slot = nd.index - key0, split = key - 1;
        s.quads[4 * slot] = make_float4(nd.lo0.x, nd.lo0.y, nd.lo0.z, __uint_as_float(LeftLink(n, key0 + nd.a, split)));
        s.quads[4 * slot + 1] = make_float4(nd.hi0.x, nd.hi0.y, nd.hi0.z, __uint_as_float(RightLink(n, split, key0 + nd.b)));
        s.quads[4 * slot + 2] = make_float4(nd.lo1.x, nd.lo1.y, nd.lo1.z, __uint_as_float(nd.parent));
        s.quads[4 * slot + 3] = make_float4(nd.hi1.x, nd.hi1.y, nd.hi1.z, __uint_as_float(0u));
        s.state[slot] = nd.waits ? 2 : 1;
    }
    __syncthreads();
    StoreQuads(false, arg, s);
    __syncthreads();
    // Leaves.
    uint32_t gap = 0;
    bool leaf_waits = false;
    if (active) {
        const bool has_parent = ParentGap(s, t, t, gap);
        const uint32_t parent = has_parent ? s.index[gap] : kInvalid;
        leaf_waits = has_parent && parent == kInvalid;
        q[2].w = __uint_as_float(parent);
        for (int j = 0; j < 4; ++j) s.quads[4 * t + j] = q[j];
    }
    s.state[t] = !active ? 0 : leaf_waits ? 2 : 1;
    __syncthreads();
    StoreQuads(true, arg, s);
    r.first = leaf_waits ? key : key0 + nd.a;
    r.last = leaf_waits ? key : key0 + nd.b;
    if (!leaf_waits && nd.waits) {
        const float4 l = Min4(nd.lo0, nd.lo1), h = Max4(nd.hi0, nd.hi1);
        r.lo[0] = l.x; r.lo[1] = l.y; r.lo[2] = l.z;
        r.hi[0] = h.x; r.hi[1] = h.y; r.hi[2] = h.z;
    } else {
        for (int k = 0; k < 3; ++k) {
            r.lo[k] = lo[k];
            r.hi[k] = hi[k];
        }
    }
    return leaf_waits || nd.waits;
}

// Publishes the workgroup's waiting subtrees, in key order (a thread's
// subtree contains the thread's entry, and a thread has one at most), as run
// `run`; returns their number.  Every thread calls it (it holds barriers); the
// stores are complete when it returns.
__device__ __forceinline__ uint32_t PublishRun(bool waits, const TreeRun& r, const TreeScratch& ts, uint32_t run,
                                               TreeLds& s) {
    const uint64_t mask = __ballot(waits);
    const uint32_t wave = threadIdx.x / 64;
    if ((threadIdx.x & 63u) == 0) s.wave_pending[wave] = (uint32_t)__popcll(mask);
    __syncthreads();
    uint32_t k = RankIn(mask), total = 0;
    for (uint32_t w = 0; w < (uint32_t)kTreeWindow / 64; ++w) {
        if (w < wave) k += s.wave_pending[w];
        total += s.wave_pending[w];
    }
    total = min(total, kTreePending);  // more only from unsorted codes (a sort that was reported as failed)
    if (waits && k < kTreePending) {
        TreePending* p = ts.pending + (size_t)run * kTreePending + k;
        StoreAgent4(p, r.first, r.last, __float_as_uint(r.lo[0]), __float_as_uint(r.lo[1]));
        StoreAgent4(reinterpret_cast<float4*>(p) + 1, __float_as_uint(r.lo[2]), __float_as_uint(r.hi[0]),
                    __float_as_uint(r.hi[1]), __float_as_uint(r.hi[2]));
    }
    if (threadIdx.x == 0) __hip_atomic_store(ts.count + run, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    WaitStores();
    __syncthreads();
    return total;
}

// After a window (waits, r: BuildWindow's result): hand-offs up the levels.
// Window `window` of `windows` (> 1) of a tree of n leaves; code(k): sorted
// code k, in global memory.  Every thread of the workgroup calls it.
template <typename Code>
__device__ __forceinline__ void FinishTree(BvhNode* __restrict__ nodes, uint32_t n, const Code& code, bool waits, TreeRun& r,
                                           const TreeScratch& ts, uint32_t window, uint32_t windows, TreeLds& s) {
    const uint32_t t = threadIdx.x;
    uint32_t base = 0, runs = windows, run = window;  // this level's first run, its runs, this workgroup's
    PublishRun(waits, r, ts, base + run, s);
    for (;;) {
        // The last of a group's runs to arrive goes on.
        const uint32_t group = run / kTreeGroup;
        const uint32_t child0 = base + group * kTreeGroup;
        const uint32_t children = min(kTreeGroup, runs - group * kTreeGroup);
        const uint32_t parent = base + runs + group;
        if (t == 0)
            s.go = __hip_atomic_fetch_add(ts.arrived + parent, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == children;
        __syncthreads();
        if (!s.go) return;
        if (t < 64) {
            uint32_t c = 0;
            if (t < children) c = min(__hip_atomic_load(ts.count + child0 + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), kTreePending);
            uint32_t sum = c;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t y = __shfl_up(sum, o, 64);
                if (t >= (uint32_t)o) sum += y;
            }
            s.group_first[t] = sum - c;  // entries before run t; past the last run, all
        }
        __syncthreads();
        const uint32_t entries = s.group_first[children];
        // At most kTreeWindow entries at a time: those still unmerged of one
        // part lead the next.
        const bool top = parent == base + runs && children == runs;
        for (uint32_t done = 0, carry = 0; done < entries;) {
            const uint32_t m = min((uint32_t)kTreeWindow, carry + entries - done);
            TreePending e{};
            uint32_t d = 0;
            if (t < m) {
                const TreePending* p = ts.pending + (size_t)parent * kTreePending + t;
                if (t >= carry) {
                    const uint32_t k = done + t - carry;
                    uint32_t c = 0;
                    for (uint32_t step = 32; step >= 1; step /= 2)
                        if (c + step < children && s.group_first[c + step] <= k) c += step;
                    p = ts.pending + (size_t)(child0 + c) * kTreePending + (k - s.group_first[c]);
                }
                e = LoadPendingAgent(p);
                s.first[t] = e.first;
                s.last[t] = e.last;
                d = (uint32_t)(1 + DeltaOf(code, (int)n, (int)e.first, code((int)e.first), (int)e.first - 1));
                if (t + 1 == m)
                    s.delta_min[0][m] = (uint8_t)(1 + DeltaOf(code, (int)n, (int)e.last, code((int)e.last), (int)e.last + 1));
            }
            if (t != m) s.delta_min[0][t] = (uint8_t)d;
            const TreeNode nd = FindNode(
                t < m, m, e.lo, e.hi, [&s](uint32_t x) { return s.first[x]; }, [&s](uint32_t x) { return s.last[x]; }, s);
            if (nd.whole) {
                const uint32_t split = s.last[t - 1], first = s.first[nd.a], last = s.last[nd.b];
                const uint32_t c0 = LeftLink(n, first, split), c1 = RightLink(n, split, last);
                float4* q = reinterpret_cast<float4*>(nodes + nd.index);
                q[0] = make_float4(nd.lo0.x, nd.lo0.y, nd.lo0.z, __uint_as_float(c0));
                q[1] = make_float4(nd.hi0.x, nd.hi0.y, nd.hi0.z, __uint_as_float(c1));
                RrBox3 third;
                third.x = nd.lo1.x; third.y = nd.lo1.y; third.z = nd.lo1.z;
                *reinterpret_cast<RrBox3*>(&q[2]) = third;
                q[3] = make_float4(nd.hi1.x, nd.hi1.y, nd.hi1.z, __uint_as_float(0u));
                // A node's parent link is the one word written with the
                // parent's node, so no two workgroups write the same bytes.
                nodes[c0].parent = nd.index;
                nodes[c1].parent = nd.index;
                if (nd.index == 0 && !nd.waits && nd.parent == kInvalid) nodes[0].parent = kInvalid;
            }
            // This thread's entry, or the node its gap splits, may wait.
            uint32_t gap = 0;
            const bool entry_waits = t < m && ParentGap(s, t, t, gap) && s.index[gap] == kInvalid;
            waits = entry_waits || nd.waits;
            r.first = entry_waits ? e.first : s.first[nd.a];
            r.last = entry_waits ? e.last : s.last[nd.b];
            const float4 l = Min4(nd.lo0, nd.lo1), h = Max4(nd.hi0, nd.hi1);
            r.lo[0] = entry_waits ? e.lo[0] : l.x; r.lo[1] = entry_waits ? e.lo[1] : l.y; r.lo[2] = entry_waits ? e.lo[2] : l.z;
            r.hi[0] = entry_waits ? e.hi[0] : h.x; r.hi[1] = entry_waits ? e.hi[1] : h.y; r.hi[2] = entry_waits ? e.hi[2] : h.z;
            done += m - carry;
            if (top && done >= entries) break;
            carry = PublishRun(waits, r, ts, parent, s);
        }
        if (top) return;
        base += runs;
        run = group;
        runs = (runs + kTreeGroup - 1) / kTreeGroup;
    }
}

}  // namespace rr
