// Traversal kernels: closest-hit rays, closest / kNN / radius point queries, over
// binary (32 B) or 4-wide (128 B) nodes, for triangle, point and Gaussian leaves.
//
// A ray or query is walked by one lane, by four (quads), or by a group of 8 to 64
// lanes whose quads each open a node a round; the launchers at the end of the file
// choose by the set's size, leaf kind and k.  The pruning predicates are the
// reference's (src/gpu/raycast.cu:75-245, src/gpu/query.cu:52-637): padded slab
// test against the current best t for rays, box lower bound <= bound for
// closest / kNN (so equal-distance primitives with a smaller index are still
// reached), box lower bound <= r^2 for radius.  Every predicate only prunes
// subtrees that cannot hold a better (dist2, index) or a smaller t, so the result
// is the brute-force answer whatever the tree, node width, walk or visiting order -
// which is what makes binary, wide, LBVH, SAH and reordered runs bit-identical.
//
// Layout for gfx950:
//   * one lane: the depth-first stack lives in LDS ([depth][lane]); deeper entries
//     spill to scratch, which only very deep or very wide traversals touch;
//   * groups: one LDS stack per query, shared by its quads; a binary node is opened
//     together with its interior children, so both node widths feed four entries to
//     a quad; the k-best list is one entry per lane;
//   * leaf children are tested as soon as their parent is opened, against the live
//     bound, and only interior children go on the stack, nearest on top;
//   * closest is kNN with k = 1 (identical record and tie rule).
//
// Queries may be visited in a permuted order (Morton reordering): lane i works
// on query order[i] and writes its result straight to slot order[i], so no
// gather/scatter copies of queries or results are made.
#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "qr_traverse.h"

namespace qr {

namespace {

constexpr int kBlock = 256;
constexpr int kLdsDepth = 32;
constexpr int kSpill = 128;  // scratch entries beyond the LDS part (never reached by LBVH trees)

// ---- XCD-aware block numbering ------------------------------------------------------
// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.  The
// traversal kernels renumber their blocks so that XCD x walks one contiguous range
// of the (Morton-ordered) queries: neighbouring queries share most of their nodes,
// and those nodes then stay in one L2 instead of being fetched by all eight.
// Bijective on [0, gridDim.x): XCD x owns q + (x < r) blocks, q = g / 8, r = g % 8.
__device__ __forceinline__ int xcdBlock() {
    const int g = static_cast<int>(gridDim.x), i = static_cast<int>(blockIdx.x);
    const int x = i & 7, j = i >> 3;
    const int q = g >> 3, r = g & 7;
    return x * q + (x < r ? x : r) + j;
}

// Largest v over the wave, one atomic per wave (nothing when dst is null).
__device__ __forceinline__ void waveMaxAtomic(int* dst, int v) {
    if (dst == nullptr) return;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    if ((threadIdx.x & 63) == 0 && v > 0) atomicMax(dst + blockIdx.x % kMaxCopies, v);
}

// ---- stats -------------------------------------------------------------------------
// stats[0] node tests, [1] leaf tests, [2] stack overflows, [3] interior nodes opened.
// Pinned host word that any walk whose stack overflowed sets to 1 (the walk stops
// and its result is incomplete); the host checks it after every query call.  Null
// until armOverflowWord() has run on the device.
__device__ int* gOverflowWord = nullptr;

template <bool kStats>
__device__ __forceinline__ void flushStats(unsigned long long* stats, int nodeTests, int leafTests,
                                           int overflow, int opened) {
    if (overflow) {  // an incomplete walk: tell the host, whatever the build
        int* w = gOverflowWord;
        if (w) __hip_atomic_store(w, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (!kStats) return;
    unsigned long long a = static_cast<unsigned long long>(nodeTests);
    unsigned long long b = static_cast<unsigned long long>(leafTests);
    unsigned long long c = static_cast<unsigned long long>(overflow);
    unsigned long long d = static_cast<unsigned long long>(opened);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off, 64);
        b += __shfl_xor(b, off, 64);
        c += __shfl_xor(c, off, 64);
        d += __shfl_xor(d, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        unsigned long long* st = stats + 4 * (blockIdx.x % kStatCopies);
        if (a) atomicAdd(&st[0], a);
        if (b) atomicAdd(&st[1], b);
        if (c) atomicAdd(&st[2], c);
        if (d) atomicAdd(&st[3], d);
    }
}

// ---- per-lane stack: LDS first, scratch beyond ---------------------------------------
// The stack pointer and LDS column are plain registers; only the spill area (the
// part beyond the LDS depth) lives in scratch.  Both areas are accessed through
// volatile pointers: that keeps every LDS access a ds_read/ds_write (which one
// wave executes in order) and stops the compiler from merging the two branches
// of a pop into one generic (flat) load, which is not ordered behind the
// preceding ds_write pushes.
typedef __attribute__((address_space(3))) volatile int LdsInt;      // workgroup LDS
typedef __attribute__((address_space(5))) volatile int PrivateInt;  // per-lane scratch

template <int kS, int kD>
struct LaneStackT {
    static constexpr int kStride = kS;  // lanes per workgroup: distance between a lane's entries
    static constexpr int kDepth = kD;   // entries kept in LDS before spilling to scratch
    LdsInt* base;  // this lane's column of the workgroup's LDS stack
    int sp;
    __device__ __forceinline__ void init(int* lds) {
        base = (LdsInt*)(lds + threadIdx.x);
        sp = 0;
    }
    __device__ __forceinline__ bool empty() const { return sp == 0; }
    __device__ __forceinline__ bool room(int n) const { return sp + n <= kD + kSpill; }
};
using LaneStack = LaneStackT<kBlock, kLdsDepth>;

struct SpillArea {
    int v[kSpill];
    __device__ __forceinline__ PrivateInt* at(int i) {
        return (PrivateInt*)(&v[i]);
    }
};

#define QR_PUSH(st, spill, val)                               \
    do {                                                      \
        const int qrv_ = (val);                               \
        if ((st).sp < (st).kDepth) {                          \
            (st).base[(st).sp * (st).kStride] = qrv_;         \
        } else {                                              \
            *(spill).at((st).sp - (st).kDepth) = qrv_;        \
        }                                                     \
        ++(st).sp;                                            \
    } while (0)

#define QR_POP(st, spill, out)                                \
    do {                                                      \
        --(st).sp;                                            \
        if ((st).sp < (st).kDepth) {                          \
            (out) = (st).base[(st).sp * (st).kStride];        \
        } else {                                              \
            (out) = *(spill).at((st).sp - (st).kDepth);       \
        }                                                     \
    } while (0)

// Stack operations shared by the walks: the LDS/scratch stack above, and a stack
// whose top R entries live in registers (a shift register: static indices only, so
// it stays in VGPRs) with deeper entries in the lane's scratch spill area.
template <typename Stack>
__device__ __forceinline__ void stackPush(Stack& st, SpillArea& spill, int v) {
    QR_PUSH(st, spill, v);
}
template <typename Stack>
__device__ __forceinline__ int stackPop(Stack& st, SpillArea& spill) {
    int v;
    QR_POP(st, spill, v);
    return v;
}

template <int R>
struct RegStack {
    int r[R];  // r[0]: top
    int sp;    // entries; those beyond R sit in the spill area, deepest first
    __device__ __forceinline__ void init(int*) { sp = 0; }
    __device__ __forceinline__ bool empty() const { return sp == 0; }
    __device__ __forceinline__ bool room(int n) const { return sp + n <= R + kSpill; }
};
template <int R>
__device__ __forceinline__ void stackPush(RegStack<R>& st, SpillArea& spill, int v) {
    if (st.sp >= R) *spill.at(st.sp - R) = st.r[R - 1];
#pragma unroll
    for (int k = R - 1; k > 0; --k) st.r[k] = st.r[k - 1];
    st.r[0] = v;
    ++st.sp;
}
template <int R>
__device__ __forceinline__ int stackPop(RegStack<R>& st, SpillArea& spill) {
    const int v = st.r[0];
#pragma unroll
    for (int k = 0; k < R - 1; ++k) st.r[k] = st.r[k + 1];
    --st.sp;
    if (st.sp >= R) st.r[R - 1] = *spill.at(st.sp - R);
    return v;
}
constexpr int kRegStack = 8;

// Compare-exchange on (key, payload) pairs: ascending by key.
__device__ __forceinline__ void cx(float& ka, int& va, float& kb, int& vb) {
    const bool sw = kb < ka;
    const float tk = ka;
    const int tv = va;
    ka = sw ? kb : ka;
    va = sw ? vb : va;
    kb = sw ? tk : kb;
    vb = sw ? tv : vb;
}

// Sorts four (key, child) pairs ascending (5 compare-exchanges).
__device__ __forceinline__ void sort4(float (&k)[4], int (&c)[4]) {
    cx(k[0], c[0], k[1], c[1]);
    cx(k[2], c[2], k[3], c[3]);
    cx(k[0], c[0], k[2], c[2]);
    cx(k[1], c[1], k[3], c[3]);
    cx(k[1], c[1], k[2], c[2]);
}

__device__ __forceinline__ bool closer(float d, int id, float bd, int bid) {
    return d < bd || (d == bd && id < bid);
}

// A query with a NaN coordinate has no closest primitive (index -1) and is not walked (by
// groups of lanes: not beyond the root): its box distances are 0 and no distance of it ever
// bounds them, so every node would be opened.
__device__ __forceinline__ bool hasNaN(V3 p) { return (p.x != p.x) | (p.y != p.y) | (p.z != p.z); }

// ---- k best so far ------------------------------------------------------------------
// Capacity-K list sorted by (dist2, index) in registers, for any k <= K.  It keeps
// the K best seen so far and prunes with the K-th: the first k entries are then
// the exact k best (a subtree beyond the K-th best cannot hold one of the k best),
// and every index into the list is static, so it never leaves registers.  A
// candidate is inserted by one ascending compare-exchange sweep; the displaced
// worst drops off the end.  Semantics equal the reference's sorted table
// (src/gpu/query.cu:150-158) and, for k = 1, its closest-point rule
// (src/gpu/query.cu:83-90).
template <int K>
struct KnnList {
    float d[K];
    int id[K];
    int n;
    __device__ __forceinline__ void init() {
        n = 0;
#pragma unroll
        for (int s = 0; s < K; ++s) {
            d[s] = kInf;
            id[s] = 0x7fffffff;
        }
    }
    __device__ __forceinline__ bool full() const { return n >= K; }
    // Pruning test for a subtree or primitive whose lower bound is lb.
    __device__ __forceinline__ bool admits(float lb) const { return !full() || lb <= d[K - 1]; }
    __device__ __forceinline__ void offer(float nd, int nid) {
        if (full() && !closer(nd, nid, d[K - 1], id[K - 1])) return;
        float cd = nd;
        int cid = nid;
#pragma unroll
        for (int s = 0; s < K; ++s) {
            const bool sw = closer(cd, cid, d[s], id[s]);
            const float td = d[s];
            const int tid = id[s];
            d[s] = sw ? cd : td;
            id[s] = sw ? cid : tid;
            cd = sw ? td : cd;
            cid = sw ? tid : cid;
        }
        n = n < K ? n + 1 : K;
    }
};

// Stack entries of the closest / kNN walks carry the child's box distance above its id,
// truncated to the bits the id leaves free: the leading bits of a non-negative
// float are a lower bound of it.  A popped node whose bound already exceeds the
// k-th distance is dropped without being opened -- opening it would find every
// child beyond the k-th distance too (a child's box lies inside its parent's), so
// the walk and its results are unchanged.  idBits = 32 turns the keys off (trees
// whose wide ids need more than 23 bits).
// Bits of a stack entry taken by a node id below `idCount` (the rest hold the
// distance key); 32 = no key, when ids need more than 23 bits (fewer than 9 would
// be left, too few for the float's exponent and a mantissa bit).
__host__ __device__ __forceinline__ int stackIdBitsDev(int idCount) {
    int bits = 1;
    while (bits < 32 && (1LL << bits) < static_cast<long long>(idCount)) ++bits;
    return bits <= 23 ? bits : 32;
}

// The same by mask (the low idBits bits; all 32 when there is no key): the float's bits,
// shifted up over the sign, above the id.
__host__ __device__ __forceinline__ uint32_t stackIdMask(int idCount) {
    const int bits = idCount <= 2 ? 1 : 32 - __builtin_clz(static_cast<unsigned>(idCount - 1));
    return bits > 23 ? ~0u : (1u << bits) - 1u;
}
__device__ __forceinline__ uint32_t stackEntry(uint32_t id, uint32_t keyBits, uint32_t idMask) {
    return ((keyBits << 1) & ~idMask) | id;
}
__device__ __forceinline__ uint32_t stackKey(uint32_t v, uint32_t idMask) { return (v & ~idMask) >> 1; }

__device__ __forceinline__ int packEntry(int id, float key, int idBits) {
    if (idBits >= 32) return id;
    const uint32_t q = floatBits(key) >> (idBits - 1);
    return static_cast<int>((q << idBits) | static_cast<uint32_t>(id));
}
__device__ __forceinline__ int entryId(int v, int idBits) {
    return idBits >= 32 ? v : static_cast<int>(static_cast<uint32_t>(v) & ((1u << idBits) - 1u));
}
__device__ __forceinline__ float entryKey(int v, int idBits) {
    return idBits >= 32 ? 0.0f : bitsFloat((static_cast<uint32_t>(v) >> idBits) << (idBits - 1));
}

// ---- rays --------------------------------------------------------------------------
// Each iteration opens one interior node: its children are tested, leaves are
// intersected nearest first, and the nearest surviving interior child becomes the
// next node without a stack round trip; the other survivors are pushed far first.

// One ray-triangle leaf test.  With kSave the hit's scene index is kept too
// (equal t: the smaller scene index), for the differentiable mode; t is the same.
template <bool kSave>
__device__ __forceinline__ void rayLeaf(const Ray& ray, const Tri* __restrict__ tris,
                                        const int* __restrict__ primIds, int slot, float& best,
                                        bool& any, int& bestId) {
    float t;
    if (!rayTri(ray, tris[slot], t)) return;
    if (t < best) {
        best = t;
        any = true;
        if (kSave) bestId = primIds[slot];
    } else if (kSave && any && t == best) {
        const int sid = primIds[slot];
        if (sid < bestId) bestId = sid;
    }
}

template <bool kStats, bool kSave>
__global__ __launch_bounds__(kBlock) void rayBinaryKernel(const Node2* __restrict__ nodes,
                                                          const Tri* __restrict__ tris,
                                                          const Ray* __restrict__ rays,
                                                          const uint32_t* __restrict__ order,
                                                          int count, uint64_t* __restrict__ out,
                                                          unsigned long long* __restrict__ stats,
                                                          const int* __restrict__ primIds,
                                                          int* __restrict__ hitPrim) {
    __shared__ int lds[kLdsDepth * kBlock];
    const int i = xcdBlock() * kBlock + threadIdx.x;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    if (i < count) {
        const int q = order ? static_cast<int>(order[i]) : i;
        const Ray ray = rays[q];
        float best = ray.tMax;
        bool any = false;
        int bestId = -1;
        LaneStack st;
        SpillArea spill;
        st.init(lds);
        float tEnter;
        const Node2 root = nodes[0];
        int id = -1;
        if (rayBox(ray, nodeBox(root), best, tEnter)) {
            ++nodeTests;
            id = 0;
        }
        while (id >= 0) {
            if (kStats) ++opened;
            const Node2 nd = nodes[id];
            const int kid[2] = {nd.left, nd.right};
            float t[2];
            int c[2];
            bool leaf[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const Node2 cn = nodes[kid[s]];
                leaf[s] = cn.left < 0;
                c[s] = leaf[s] ? -cn.left - 1 : kid[s];
                t[s] = kInf;
                if (rayBox(ray, nodeBox(cn), best, t[s])) {
                    ++nodeTests;
                } else {
                    c[s] = kWideEmpty;
                    t[s] = kInf;
                }
            }
            const bool swap = t[1] < t[0];
            const int c0 = swap ? c[1] : c[0], c1 = swap ? c[0] : c[1];
            const bool l0 = swap ? leaf[1] : leaf[0], l1 = swap ? leaf[0] : leaf[1];
            if (c0 != kWideEmpty && l0) {
                ++leafTests;
                rayLeaf<kSave>(ray, tris, primIds, c0, best, any, bestId);
            }
            if (c1 != kWideEmpty && l1) {
                ++leafTests;
                rayLeaf<kSave>(ray, tris, primIds, c1, best, any, bestId);
            }
            const bool in0 = c0 != kWideEmpty && !l0;
            const bool in1 = c1 != kWideEmpty && !l1;
            if (in0) {
                if (in1) {
                    if (!st.room(1)) {
                        overflow = 1;
                        break;
                    }
                    QR_PUSH(st, spill, c1);
                }
                id = c0;
            } else if (in1) {
                id = c1;
            } else if (!st.empty()) {
                QR_POP(st, spill, id);
            } else {
                id = -1;
            }
        }
        out[q] = any ? ((uint64_t{1} << 32) | floatBits(best)) : 0ull;
        if (kSave) hitPrim[q] = any ? bestId : -1;
    }
    flushStats<kStats>(stats, nodeTests, leafTests, overflow, opened);
}

__device__ __forceinline__ void loadWide(const Wide4* __restrict__ wide, int id, WideEntry (&e)[4]) {
    const Wide4& wn = wide[id];
#pragma unroll
    for (int s = 0; s < 4; ++s) e[s] = wn.c[s];
}

// After the four children are sorted: the first interior survivor continues the
// descent, the rest are pushed far first.  Returns the next node, or pops one
// (-1 when the traversal is complete).  ok[s] says whether slot s survives.
__device__ __forceinline__ int descend(const int (&c)[4], const bool (&ok)[4], LaneStack& st,
                                       SpillArea& spill, int& overflow) {
    int next = -1;
    int first = -1;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (ok[s] && c[s] >= 0 && first < 0) first = s;
    }
    if (!st.room(3)) {
        overflow = 1;
        return -1;
    }
#pragma unroll
    for (int s = 3; s >= 0; --s) {
        if (ok[s] && c[s] >= 0 && s != first) QR_PUSH(st, spill, c[s]);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
        if (s == first) next = c[s];
    if (first < 0) {
        if (!st.empty()) {
            QR_POP(st, spill, next);
        }
    }
    return next;
}

// The same for entry distances as ray stacks keep them (not below zero): a negative best (a
// ray whose tMin is negative) drops nothing at zero.
__device__ __forceinline__ float stackReach(float best) { return fmaxf(rayReach(best), 0.0f); }

// One lane per ray over 4-wide nodes, for large ray sets.  The leaves of an opened node are
// tested one per lane and step, not slot by slot: the wave runs the triangle test (the
// longest piece of a step) as often as its busiest lane has leaves, not four times.  The
// children's box tests share the ray's reciprocals and have no branches; the nearest
// interior child is opened next and the others go on the stack farthest first by rank (no
// sort moves them), with their entry distance above their id: a popped entry that lies
// beyond the best hit is dropped unopened.  1M rays, kernel time before and after: city,
// cosine 682 -> 477 us, down 300 -> 242; 131k terrain, cosine 1009 -> 678, down 352 -> 298;
// icosphere 954 -> 705.  Opening nodes until some lane has a leaf before testing any was
// slower (icosphere 1097).
constexpr int kRayDepth = 16;  // stack entries per lane in LDS (8 workgroups a CU), the rest in scratch
template <bool kStats, bool kSave>
__global__ __launch_bounds__(kBlock) void rayWideKernel(const Wide4* __restrict__ wide,
                                                        const Tri* __restrict__ tris,
                                                        const Ray* __restrict__ rays,
                                                        const uint32_t* __restrict__ order,
                                                        int count, uint64_t* __restrict__ out,
                                                        unsigned long long* __restrict__ stats,
                                                        const int* __restrict__ primIds,
                                                        int* __restrict__ hitPrim, uint32_t idMask) {
    __shared__ int lds[kRayDepth * kBlock];
    const int i = xcdBlock() * kBlock + threadIdx.x;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    if (i < count) {
        const int q = order ? static_cast<int>(order[i]) : i;
        const Ray ray = rays[q];
        const RayPre pre = rayPrepare(ray);
        float best = ray.tMax;
        bool any = false;
        int bestId = -1;
        LaneStackT<kBlock, kRayDepth> st;
        SpillArea spill;
        st.init(lds);
        uint32_t next = 0;  // the entry to open (kDone: none left)
        constexpr uint32_t kDone = ~0u;
        while (next != kDone) {
            int leaf[4];
            uint32_t leaves = 0;
            if (kStats) ++opened;
            const Wide4& wn = wide[next & idMask];
            next = kDone;
            uint32_t key[4];
            int c[4];
            bool in[4];
            int m = 0;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const WideEntry e = wn.c[s];
                float t;
                c[s] = e.child;
                const bool adm = rayBoxPre(pre, entryBox(e), best, t) & (c[s] != kWideEmpty);
                if (kStats && adm) ++nodeTests;
                in[s] = adm & (c[s] >= 0);
                key[s] = in[s] ? (floatBits(fmaxf(t, 0.0f)) & ~3u) | s : 0xfffffffcu | s;
                m += in[s] ? 1 : 0;
                leaf[s] = -c[s] - 1;
                leaves |= adm & (c[s] < 0) ? 1u << s : 0u;
            }
            if (m > 0) {
                if (!st.room(3)) {
                    overflow = 1;
                    break;
                }
                const int a = key[1] < key[0], b = key[2] < key[0], d = key[3] < key[0];
                const int e = key[2] < key[1], f = key[3] < key[1], g = key[3] < key[2];
                const int rank[4] = {a + b + d, 1 - a + e + f, 2 - b - e + g, 3 - d - f - g};
                const int top = st.sp + m - 1;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const uint32_t v = stackEntry(static_cast<uint32_t>(c[s]), key[s], idMask);
                    if (rank[s] == 0) next = v;
                    if (in[s] & (rank[s] > 0)) {
                        const int at = top - rank[s];
                        if (at < kRayDepth) st.base[at * kBlock] = static_cast<int>(v);
                        else *spill.at(at - kRayDepth) = static_cast<int>(v);
                    }
                }
                st.sp = top;
            } else {
                const float reach = stackReach(best);
                while (!st.empty()) {
                    const uint32_t v = static_cast<uint32_t>(stackPop(st, spill));
                    if (bitsFloat(stackKey(v, idMask)) <= reach) {
                        next = v;
                        break;
                    }
                }
            }
            while (leaves != 0) {
                const int slot = (leaves & 1u) ? leaf[0] : ((leaves & 2u) ? leaf[1] : ((leaves & 4u) ? leaf[2] : leaf[3]));
                leaves &= leaves - 1u;
                if (kStats) ++leafTests;
                rayLeaf<kSave>(ray, tris, primIds, slot, best, any, bestId);
            }
        }
        out[q] = any ? ((uint64_t{1} << 32) | floatBits(best)) : 0ull;
        if (kSave) hitPrim[q] = any ? bestId : -1;
    }
    flushStats<kStats>(stats, nodeTests, leafTests, overflow, opened);
}

// ---- closest / kNN ------------------------------------------------------------------

template <typename L, int K>
__device__ __forceinline__ void writeList(const KnnList<K>& list, int k, ClosestResult* dst) {
#pragma unroll
    for (int s = 0; s < K; ++s) {
        if (s < k) {
            ClosestResult r{0u, -1};
            // (the fill's id: a NaN distance was counted, not kept)
            if (s < list.n && list.id[s] != 0x7fffffff) r = {floatBits(list.d[s]), list.id[s]};
            dst[s] = r;
        }
    }
}

// Closest / kNN walk of one query over a binary tree whose node ids, leaf slots
// and prim ids are local to `nodes`, `prims` and `primIds` (a plain tree, or one
// tree of a batch addressed through offset pointers).
template <typename L, int K, bool kStats, typename Stack>
__device__ __forceinline__ void nearestBinaryWalk(const Node2* __restrict__ nodes,
                                                  const typename L::Item* __restrict__ prims,
                                                  const int* __restrict__ primIds, V3 p,
                                                  KnnList<K>& list, Stack& st, SpillArea& spill,
                                                  int& nodeTests, int& leafTests, int& overflow,
                                                  int& opened, int idBits) {
    int id = hasNaN(p) ? -1 : 0;
    while (id >= 0) {
        if (kStats) ++opened;
        const Node2 nd = nodes[id];
        ++nodeTests;
        const int kid[2] = {nd.left, nd.right};
        float key[2];
        int c[2];
        bool leaf[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const Node2 cn = nodes[kid[s]];
            leaf[s] = cn.left < 0;
            c[s] = leaf[s] ? -cn.left - 1 : kid[s];
            key[s] = boxDist2(p, nodeBox(cn));
        }
        const bool swap = key[1] < key[0];
        const int c0 = swap ? c[1] : c[0], c1 = swap ? c[0] : c[1];
        const bool l0 = swap ? leaf[1] : leaf[0], l1 = swap ? leaf[0] : leaf[1];
        const float k0 = swap ? key[1] : key[0], k1 = swap ? key[0] : key[1];
        if (l0 && list.admits(k0)) {
            ++leafTests;
            list.offer(L::dist2(p, prims[c0]), primIds[c0]);
        }
        if (l1 && list.admits(k1)) {
            ++leafTests;
            list.offer(L::dist2(p, prims[c1]), primIds[c1]);
        }
        const bool in0 = !l0 && list.admits(k0);
        const bool in1 = !l1 && list.admits(k1);
        if (in0) {
            if (in1) {
                if (!st.room(1)) {
                    overflow = 1;
                    break;
                }
                stackPush(st, spill, packEntry(c1, k1, idBits));
            }
            id = c0;
        } else if (in1) {
            id = c1;
        } else {
            id = -1;
            while (!st.empty()) {
                const int v = stackPop(st, spill);
                if (list.admits(entryKey(v, idBits))) {
                    id = entryId(v, idBits);
                    break;
                }
            }
        }
    }
}

template <typename L, int K, bool kStats>
__global__ __launch_bounds__(kBlock) void nearestBinaryKernel(
    const Node2* __restrict__ nodes, const typename L::Item* __restrict__ prims,
    const int* __restrict__ primIds, const V3* __restrict__ points,
    const uint32_t* __restrict__ order, int count, int k, int outStride,
    ClosestResult* __restrict__ out, unsigned long long* __restrict__ stats, int idBits) {
    __shared__ int lds[kLdsDepth * kBlock];
    const int i = xcdBlock() * kBlock + threadIdx.x;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    if (i < count) {
        const int q = order ? static_cast<int>(order[i]) : i;
        KnnList<K> list;
        list.init();
        LaneStack st;
        SpillArea spill;
        st.init(lds);
        nearestBinaryWalk<L, K, kStats>(nodes, prims, primIds, points[q], list, st, spill, nodeTests,
                                        leafTests, overflow, opened, idBits);
        writeList<L, K>(list, k, out + static_cast<size_t>(q) * outStride);
    }
    flushStats<kStats>(stats, nodeTests, leafTests, overflow, opened);
}

// ---- batched scenes: persistent work-queue traversal ------------------------------------
// (The 4-wide variants with the stack in LDS are batchGroupKernel below.)
// Queries of all scenes form one queue (scene-major, optionally Morton-ordered inside
// each scene).  Each wave takes the next 64 queries with one atomic and walks, per
// lane, the tree of that query's scene (scene s: items from primOff[s]; binary nodes
// from 2 primOff[s] - s, or 4-wide nodes from wideRoot[s]); the grid is sized to the
// resident occupancy and every wave leaves when the queue is exhausted.  Stack
// placement: kD entries per lane in LDS with the rest in scratch (kD = 0: all in
// scratch), or, with kReg, the top kRegStack entries in registers.
template <typename L, int K, int kBT, int kD, bool kWide, bool kReg>
__global__ __launch_bounds__(kBT) void batchNearestKernel(
    const Node2* __restrict__ nodes, const Wide4* __restrict__ wide, const int* __restrict__ wideRoot,
    const typename L::Item* __restrict__ prims, const int* __restrict__ primIds, const int* __restrict__ primOff,
    const V3* __restrict__ points, const int* __restrict__ qScene, const uint32_t* __restrict__ order, int count,
    int k, int outStride, ClosestResult* __restrict__ out, int* __restrict__ counter) {
    __shared__ int lds[(kD > 0 && !kReg ? kD : 1) * kBT];
    const int lane = threadIdx.x & 63;
    while (true) {
        int base = 0;
        if (lane == 0) base = atomicAdd(counter, 64);
        base = __shfl(base, 0, 64);
        if (base >= count) break;
        const int i = base + lane;
        if (i < count) {
            const int q = order ? static_cast<int>(order[i]) : i;
            const int s = qScene[q];
            const int ps = primOff[s];
            KnnList<K> list;
            list.init();
            typename std::conditional<kReg, RegStack<kRegStack>, LaneStackT<kBT, kD>>::type st;
            SpillArea spill;
            st.init(lds);
            int a = 0, b = 0, c = 0, d = 0;
            if (kWide) {
                const int wr = wideRoot[s];
                // wide ids of the scene's tree stay below its wide-node count
                nearestWideWalk<L, K, false>(wide + wr, prims + ps, primIds + ps, points[q], list, st, spill, a, b,
                                             c, d, stackIdBitsDev(wideRoot[s + 1] - wr));
            } else {
                // node ids of the scene's tree stay below 2 n_s - 1
                nearestBinaryWalk<L, K, false>(nodes + (2 * ps - s), prims + ps, primIds + ps, points[q], list, st,
                                               spill, a, b, c, d, stackIdBitsDev(2 * (primOff[s + 1] - ps) - 1));
            }
            if (c) {
                int* w = gOverflowWord;
                if (w) __hip_atomic_store(w, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            writeList<L, K>(list, k, out + static_cast<size_t>(q) * outStride);
        }
    }
}

__global__ void batchResetKernel(int* __restrict__ counter) {
    if (threadIdx.x == 0 && blockIdx.x == 0) counter[0] = 0;
}

// Closest / kNN walk of one query over a 4-wide tree whose node ids, leaf slots and
// prim ids are local to `wide`, `prims` and `primIds` (root at wide[0]).
template <typename L, int K, bool kStats, typename Stack>
__device__ __forceinline__ void nearestWideWalk(const Wide4* __restrict__ wide,
                                                const typename L::Item* __restrict__ prims,
                                                const int* __restrict__ primIds, V3 p, KnnList<K>& list,
                                                Stack& st, SpillArea& spill, int& nodeTests, int& leafTests,
                                                int& overflow, int& opened, int idBits) {
    int id = hasNaN(p) ? -1 : 0;
    while (id >= 0) {
        if (kStats) ++opened;
        WideEntry e[4];
        loadWide(wide, id, e);
        float key[4];
        int c[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            c[s] = e[s].child;
            key[s] = kInf;
            if (c[s] != kWideEmpty) {
                const float d = boxDist2(p, entryBox(e[s]));
                if (list.admits(d)) {
                    key[s] = d;
                    ++nodeTests;
                } else {
                    c[s] = kWideEmpty;
                }
            }
        }
        sort4(key, c);
        // leaves now, nearest first, against the live bound
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (c[s] != kWideEmpty && c[s] < 0 && list.admits(key[s])) {
                const int slot = -c[s] - 1;
                ++leafTests;
                list.offer(L::dist2(p, prims[slot]), primIds[slot]);
            }
        }
        // nearest surviving interior child next; the others pushed far first with
        // their distance keys; pops skip entries the k-th distance has overtaken
        int first = -1;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (c[s] >= 0 && list.admits(key[s]) && first < 0) first = s;
        }
        if (!st.room(3)) {
            overflow = 1;
            break;
        }
#pragma unroll
        for (int s = 3; s >= 0; --s) {
            if (c[s] >= 0 && list.admits(key[s]) && s != first) stackPush(st, spill, packEntry(c[s], key[s], idBits));
        }
        id = -1;
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (s == first) id = c[s];
        if (first < 0) {
            while (!st.empty()) {
                const int v = stackPop(st, spill);
                if (list.admits(entryKey(v, idBits))) {
                    id = entryId(v, idBits);
                    break;
                }
            }
        }
    }
}

template <typename L, int K, bool kStats>
__global__ __launch_bounds__(kBlock) void nearestWideKernel(
    const Wide4* __restrict__ wide, const typename L::Item* __restrict__ prims,
    const int* __restrict__ primIds, const V3* __restrict__ points,
    const uint32_t* __restrict__ order, int count, int k, int outStride,
    ClosestResult* __restrict__ out, unsigned long long* __restrict__ stats, int idBits) {
    __shared__ int lds[kLdsDepth * kBlock];
    const int i = xcdBlock() * kBlock + threadIdx.x;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    if (i < count) {
        const int q = order ? static_cast<int>(order[i]) : i;
        KnnList<K> list;
        list.init();
        LaneStack st;
        SpillArea spill;
        st.init(lds);
        nearestWideWalk<L, K, kStats>(wide, prims, primIds, points[q], list, st, spill, nodeTests, leafTests,
                                      overflow, opened, idBits);
        writeList<L, K>(list, k, out + static_cast<size_t>(q) * outStride);
    }
    flushStats<kStats>(stats, nodeTests, leafTests, overflow, opened);
}

// ---- four lanes per query -------------------------------------------------------------
// For query sets too small to fill the GPU one lane per query, a quad of lanes
// walks one query: lane s takes entry s of each 4-wide node (one 128 B load per
// quad), tests its box and, if it is a leaf, its primitive -- in parallel.  Every
// quantity that steers the walk (the k-best list, the stack pointer, the next
// node) is kept identical in the four lanes: candidates are exchanged within the
// quad (DPP quad broadcasts) and offered in slot order by all four lanes.  The
// quad's stack is a private LDS column written by the pushing lanes.

template <int S>
__device__ __forceinline__ int quadGet(int v) {
    return __builtin_amdgcn_mov_dpp(v, S | (S << 2) | (S << 4) | (S << 6), 0xF, 0xF, false);
}
template <int S>
__device__ __forceinline__ float quadGetF(float v) {
    return __int_as_float(quadGet<S>(__float_as_int(v)));
}

constexpr int kQuadDepth = 96;  // 3 x the deepest 4-wide level a tree here can have (kMaxTreeDepth / 2)

// DPP quad permutation: lane s of each quad receives lane P[s] (2 bits per lane).
template <int P>
__device__ __forceinline__ int quadPerm(int v) {
    return __builtin_amdgcn_mov_dpp(v, P, 0xF, 0xF, false);
}
constexpr int kQuadXor1 = 1 | (0 << 2) | (3 << 4) | (2 << 6);
constexpr int kQuadXor2 = 2 | (3 << 2) | (0 << 4) | (1 << 6);
constexpr int kQuadPrev = 0 | (0 << 2) | (1 << 4) | (2 << 6);

// The k-best list of a quad, spread over its four lanes: lane s holds entries
// [s E, s E + E) of the sorted list (E = K / 4).  Same contents and order as
// KnnList<K> after the same offers: an offer (the same candidate in all four lanes)
// goes to position pos = number of entries not farther than it (a quad sum of the
// lanes' counts); entries at pos and after move one place down, the one crossing a
// lane boundary coming from the previous lane.  Every lane keeps the list's last
// entry (kd, kid) for pruning.  Per offer this is E compares and 2 E selects per
// lane instead of K of each in every lane.
template <int K>
struct QuadKnnList {
    static constexpr int E = K / 4;
    static_assert(K % 4 == 0, "K must be a multiple of 4");
    float d[E];
    int id[E];
    int n;
    float kd;
    int kid;
    __device__ __forceinline__ void init() {
        n = 0;
#pragma unroll
        for (int j = 0; j < E; ++j) {
            d[j] = kInf;
            id[j] = 0x7fffffff;
        }
        kd = kInf;
        kid = 0x7fffffff;
    }
    __device__ __forceinline__ bool admits(float lb) const { return n < K || lb <= kd; }
    __device__ __forceinline__ void offer(float nd, int nid, int slot) {
        if (n >= K && !closer(nd, nid, kd, kid)) return;
        int before = 0;
#pragma unroll
        for (int j = 0; j < E; ++j) before += closer(nd, nid, d[j], id[j]) ? 0 : 1;
        int pos = before + quadPerm<kQuadXor1>(before);
        pos += quadPerm<kQuadXor2>(pos);
        const float pd = __int_as_float(quadPerm<kQuadPrev>(__float_as_int(d[E - 1])));
        const int pi = quadPerm<kQuadPrev>(id[E - 1]);
#pragma unroll
        for (int j = E - 1; j >= 0; --j) {
            const int g = slot * E + j;
            const float od = j > 0 ? d[j - 1] : pd;
            const int oi = j > 0 ? id[j - 1] : pi;
            d[j] = g > pos ? od : (g == pos ? nd : d[j]);
            id[j] = g > pos ? oi : (g == pos ? nid : id[j]);
        }
        n = n < K ? n + 1 : K;
        kd = quadGetF<3>(d[E - 1]);
        kid = quadGet<3>(id[E - 1]);
    }
    __device__ __forceinline__ void store(ClosestResult* dst, int k, int slot) const {
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const int g = slot * E + j;
            if (g < k) {
                ClosestResult r{0u, -1};
                if (g < n && id[j] != 0x7fffffff) r = {floatBits(d[j]), id[j]};
                dst[g] = r;
            }
        }
    }
};

// k = 1: one entry, kept in every lane.
template <>
struct QuadKnnList<1> {
    float kd;
    int kid;
    int n;
    __device__ __forceinline__ void init() {
        kd = kInf;
        kid = 0x7fffffff;
        n = 0;
    }
    __device__ __forceinline__ bool admits(float lb) const { return n == 0 || lb <= kd; }
    __device__ __forceinline__ void offer(float nd, int nid, int) {
        if (n == 0 || closer(nd, nid, kd, kid)) {
            kd = nd;
            kid = nid;
        }
        n = 1;
    }
    __device__ __forceinline__ void store(ClosestResult* dst, int k, int slot) const {
        if (slot == 0 && k > 0) dst[0] = n ? ClosestResult{floatBits(kd), kid} : ClosestResult{0u, -1};
    }
};

template <typename L, int K, bool kStats>
__global__ __launch_bounds__(kBlock) void nearestQuadKernel(
    const Wide4* __restrict__ wide, const typename L::Item* __restrict__ prims,
    const int* __restrict__ primIds, const V3* __restrict__ points,
    const uint32_t* __restrict__ order, int count, int k, int outStride,
    ClosestResult* __restrict__ out, unsigned long long* __restrict__ stats, int idBits) {
    __shared__ int lds[kQuadDepth * (kBlock / 4)];
    const int t = xcdBlock() * kBlock + threadIdx.x;
    const int qi = t >> 2;
    const int slot = threadIdx.x & 3;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    if (qi < count) {  // the same for the four lanes of a quad
        const int q = order ? static_cast<int>(order[qi]) : qi;
        const V3 p = points[q];
        QuadKnnList<K> list;
        list.init();
        LdsInt* stk = (LdsInt*)(lds + (threadIdx.x >> 2) * kQuadDepth);
        int sp = 0;
        // The successor is requested before this node's leaves are tested: offers can
        // only shrink the k-th distance, so the walk continues either with the nearest
        // child that survives the box tests now or, if none survives the offers,
        // with the top of the stack -- that one is requested speculatively and the
        // entry is reloaded only when the offers pruned it.
        WideEntry e = wide[0].c[slot];
        const bool walk = !hasNaN(p);
        while (walk) {
            if (kStats && slot == 0) ++opened;
            const int ch = e.child;
            const bool leaf = ch < 0 && ch != kWideEmpty;
            typename L::Item it;
            int pid = 0;
            if (leaf) {
                it = prims[-ch - 1];
                pid = primIds[-ch - 1];
            }
            float d = kInf;
            bool adm = false;
            if (ch != kWideEmpty) {
                d = boxDist2(p, entryBox(e));
                adm = list.admits(d);
            }
            if (adm) ++nodeTests;
            int spec = -1;
            {
                const bool in0 = adm && !leaf;
                const float key0 = in0 ? d : kInf;
                const int child0 = in0 ? ch : -1;
                const float k0 = quadGetF<0>(key0), k1 = quadGetF<1>(key0), k2 = quadGetF<2>(key0), k3 = quadGetF<3>(key0);
                const int c0 = quadGet<0>(child0), c1 = quadGet<1>(child0), c2 = quadGet<2>(child0), c3 = quadGet<3>(child0);
                float bk = kInf;
                if (c3 >= 0) { spec = c3; bk = k3; }
                if (c2 >= 0 && !(bk < k2)) { spec = c2; bk = k2; }
                if (c1 >= 0 && !(bk < k1)) { spec = c1; bk = k1; }
                if (c0 >= 0 && !(bk < k0)) { spec = c0; bk = k0; }
                for (int j = sp - 1; spec < 0 && j >= 0; --j) {
                    const int v = stk[j];
                    if (list.admits(entryKey(v, idBits))) spec = entryId(v, idBits);
                }
            }
            // (the root when there is no successor: a cached, harmless read)
            const WideEntry se = wide[spec >= 0 ? spec : 0].c[slot];
            float cd = kInf;
            int cid = 0x7fffffff;
            int cand = 0;
            if (adm && leaf) {
                ++leafTests;
                cd = L::dist2(p, it);
                cid = pid;
                cand = 1;
            }
            {
                const float d0 = quadGetF<0>(cd), d1 = quadGetF<1>(cd), d2 = quadGetF<2>(cd), d3 = quadGetF<3>(cd);
                const int i0 = quadGet<0>(cid), i1 = quadGet<1>(cid), i2 = quadGet<2>(cid), i3 = quadGet<3>(cid);
                const int o0 = quadGet<0>(cand), o1 = quadGet<1>(cand), o2 = quadGet<2>(cand), o3 = quadGet<3>(cand);
                if (o0) list.offer(d0, i0, slot);
                if (o1) list.offer(d1, i1, slot);
                if (o2) list.offer(d2, i2, slot);
                if (o3) list.offer(d3, i3, slot);
            }
            const bool in = adm && !leaf && list.admits(d);
            const float key = in ? d : kInf;
            const int child = in ? ch : -1;
            const float k0 = quadGetF<0>(key), k1 = quadGetF<1>(key), k2 = quadGetF<2>(key), k3 = quadGetF<3>(key);
            const int c0 = quadGet<0>(child), c1 = quadGet<1>(child), c2 = quadGet<2>(child), c3 = quadGet<3>(child);
            // rank of this lane's child among the quad's surviving children (ties by slot)
            int rank = 0;
            rank += (slot != 0) && (k0 < key || (k0 == key && 0 < slot));
            rank += (slot != 1) && (k1 < key || (k1 == key && 1 < slot));
            rank += (slot != 2) && (k2 < key || (k2 == key && 2 < slot));
            rank += (slot != 3) && (k3 < key || (k3 == key && 3 < slot));
            const int m = (c0 >= 0) + (c1 >= 0) + (c2 >= 0) + (c3 >= 0);
            if (m > 0) {
                if (sp + m - 1 > kQuadDepth) {
                    if (slot == 0) overflow = 1;
                    break;
                }
                if (in && rank > 0) stk[sp + (m - 1 - rank)] = packEntry(ch, d, idBits);
                sp += m - 1;
                // the nearest survivor: smallest key, then smallest slot
                int next = -1;
                float bk = kInf;
                if (c3 >= 0) { next = c3; bk = k3; }
                if (c2 >= 0 && !(bk < k2)) { next = c2; bk = k2; }
                if (c1 >= 0 && !(bk < k1)) { next = c1; bk = k1; }
                if (c0 >= 0 && !(bk < k0)) { next = c0; bk = k0; }
                if (next == spec) e = se;
                else e = wide[next].c[slot];
            } else {
                while (sp > 0 && !list.admits(entryKey(stk[sp - 1], idBits))) --sp;
                if (sp == 0) break;
                --sp;
                const int next = entryId(stk[sp], idBits);
                if (next == spec) e = se;
                else e = wide[next].c[slot];
            }
        }
        list.store(out + static_cast<size_t>(q) * outStride, k, slot);
    }
    flushStats<kStats>(stats, nodeTests, leafTests, overflow, opened);
}

// Radius with four lanes per query: lane s tests entry s; hits of a node are
// counted, or written at the quad's cursor plus the number of hits in lower slots.
// kMode: kRadiusCount counts; kRadiusFill writes into the query's CSR segment
// (bounded by the next offset), skipping queries whose hits the capture pass already
// holds (counts[q] <= cap); kRadiusCaptureMode counts and writes the first `cap` hits
// into the query's fixed slot of `keys`, so that one walk serves every query with at
// most that many hits.
enum RadiusMode : int { kRadiusCount = 0, kRadiusFill = 1, kRadiusCaptureMode = 2 };
template <typename L, int kMode, bool kStats>
__global__ __launch_bounds__(kBlock) void radiusQuadKernel(
    const Wide4* __restrict__ wide, const typename L::Item* __restrict__ prims,
    const int* __restrict__ primIds, const V3* __restrict__ points, const uint32_t* __restrict__ order,
    int count, float r2, int* __restrict__ counts, const int* __restrict__ offsets,
    uint64_t* __restrict__ keys, unsigned long long* __restrict__ stats, int* __restrict__ maxCount, int cap) {
    __shared__ int lds[kQuadDepth * (kBlock / 4)];
    const int t = xcdBlock() * kBlock + threadIdx.x;
    const int qi = t >> 2;
    const int slot = threadIdx.x & 3;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    int queryHits = 0;
    constexpr bool kFill = kMode != kRadiusCount;  // hits are written somewhere
    bool live = qi < count;
    int q = 0;
    if (live) {
        q = order ? static_cast<int>(order[qi]) : qi;
        if (kMode == kRadiusFill && counts[q] <= cap) live = false;  // captured already
    }
    if (live) {
        const V3 p = points[q];
        int found = 0;
        const long long segBase = kMode == kRadiusCaptureMode ? static_cast<long long>(q) * cap : 0;
        int write = kMode == kRadiusFill ? offsets[q] : 0;
        const int end = kMode == kRadiusFill ? offsets[q + 1] : (kMode == kRadiusCaptureMode ? cap : 0);
        LdsInt* stk = (LdsInt*)(lds + (threadIdx.x >> 2) * kQuadDepth);
        int sp = 0;
        // The next node depends on the box tests only, so its entry is requested
        // before this node's leaves are tested: the leaf loads and tests overlap the
        // next node's load.
        WideEntry e = wide[0].c[slot];
        while (true) {
            if (kStats && slot == 0) ++opened;
            const int ch = e.child;
            const bool leaf = ch < 0 && ch != kWideEmpty;
            typename L::Item it;
            int pid = 0;
            if (leaf) {
                it = prims[-ch - 1];
                if (kFill) pid = primIds[-ch - 1];
            }
            const bool adm = ch != kWideEmpty && boxDist2(p, entryBox(e)) <= r2;
            if (adm) ++nodeTests;
            const int child = (adm && !leaf) ? ch : -1;
            const int c0 = quadGet<0>(child), c1 = quadGet<1>(child), c2 = quadGet<2>(child), c3 = quadGet<3>(child);
            const int m = (c0 >= 0) + (c1 >= 0) + (c2 >= 0) + (c3 >= 0);
            int next = -1;
            if (m > 0) {
                if (sp + m - 1 > kQuadDepth) {
                    if (slot == 0) overflow = 1;
                    break;
                }
                // the lowest surviving slot continues; the others are pushed in slot order
                const int first = c0 >= 0 ? 0 : (c1 >= 0 ? 1 : (c2 >= 0 ? 2 : 3));
                const int below = (slot > 0 && c0 >= 0) + (slot > 1 && c1 >= 0) + (slot > 2 && c2 >= 0);
                if (child >= 0 && slot != first) stk[sp + below - 1] = child;
                sp += m - 1;
                next = first == 0 ? c0 : (first == 1 ? c1 : (first == 2 ? c2 : c3));
            } else if (sp > 0) {
                --sp;
                next = stk[sp];
            }
            WideEntry ne;
            if (next >= 0) ne = wide[next].c[slot];
            int hit = 0;
            float d2 = 0.0f;
            if (adm && leaf) {
                ++leafTests;
                d2 = L::dist2(p, it);
                hit = d2 <= r2 ? 1 : 0;
            }
            const int h0 = quadGet<0>(hit), h1 = quadGet<1>(hit), h2 = quadGet<2>(hit), h3 = quadGet<3>(hit);
            if (kFill) {
                const int before = (slot > 0 ? h0 : 0) + (slot > 1 ? h1 : 0) + (slot > 2 ? h2 : 0);
                const int at = write + before;
                if (hit && at < end)
                    keys[segBase + at] = (static_cast<uint64_t>(floatBits(d2)) << 32) | static_cast<uint32_t>(pid);
                write += h0 + h1 + h2 + h3;
            } else {
                found += hit;
            }
            if (next < 0) break;
            e = ne;
        }
        if (kMode == kRadiusCount) {
            const int total = quadGet<0>(found) + quadGet<1>(found) + quadGet<2>(found) + quadGet<3>(found);
            if (slot == 0) counts[q] = total;
            queryHits = total;
        } else if (kMode == kRadiusCaptureMode) {
            if (slot == 0) counts[q] = write;
            queryHits = write;
        }
    }
    if (kMode != kRadiusFill) waveMaxAtomic(maxCount, queryHits);
    flushStats<kStats>(stats, nodeTests, leafTests, overflow, opened);
}

template <typename V>
__device__ __forceinline__ V waveXor(V v, int m) {
    return __shfl_xor(v, m, 64);
}

// Bitonic sort of one (key, value) pair per lane, ascending by (key, value), over
// aligned groups of `width` lanes (a power of two, at most 64; the default sorts
// the whole wave).
__device__ __forceinline__ void waveSortPairs(float& k, int& v, int lane, int width = 64) {
    for (int size = 2; size <= width; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            const float ok = waveXor(k, stride);
            const int ov = waveXor(v, stride);
            const bool up = (lane & size) == 0 || size == width;
            const bool low = (lane & stride) == 0;
            const bool otherFirst = closer(ok, ov, k, v);
            // the lower lane of an ascending pair keeps the smaller, the upper the larger
            const bool take = (low == up) ? otherFirst : !otherFirst;
            if (take) {
                k = ok;
                v = ov;
            }
        }
    }
}

// LDS stack of the walks that give a query a group of lanes: entries per wave, split among
// its queries.  A round pops w entries and pushes at most 4w, and w is held to
// (stack - kWaveHeadroom - sp) / 3 (at least 1), so sp stays below stack - kWaveHeadroom
// except while popping one entry per round, which adds at most 3 per 4-wide level -- within
// the headroom for 32 levels, half of kMaxTreeDepth (the quad kernels' stack assumes the same).
constexpr int kWaveStack = 1024;
constexpr int kWaveHeadroom = 3 * 32 + 4;

// ---- steps of a group of G lanes (16, 32 or 64, aligned within the wave) ----------------
// A group works on one query; the groups of a wave run the same instructions, so the
// steps below keep to vector operations and wave-uniform branches.

// The group's own bits of a ballot.  G <= 32: the half-wave word, masked to the group
// and left in place (32-bit counts and shifts instead of 64-bit ones); G = 64: all.
template <int G>
struct GroupBits {
    using Word = uint32_t;
    Word mask;       // the group's lanes
    Word lower;      // those below this lane
    Word lowerQuad;  // those in lower quads than this lane's
    bool high;       // the group lies in lanes 32..63
    int base;        // lane of bit 0
    __device__ __forceinline__ void init(int lane) {
        const int at = lane & 31;
        high = lane >= 32;
        base = lane & 32;
        mask = G == 32 ? ~0u : ((1u << (G & 31)) - 1u) << (at & ~(G - 1));
        lower = mask & ((1u << at) - 1u);
        lowerQuad = mask & ((1u << (at & ~3)) - 1u);
    }
    __device__ __forceinline__ Word of(unsigned long long ballot) const {
        return (high ? static_cast<uint32_t>(ballot >> 32) : static_cast<uint32_t>(ballot)) & mask;
    }
    __device__ __forceinline__ static int count(Word w) { return __popc(w); }
    __device__ __forceinline__ static int first(Word w) { return __ffs(static_cast<int>(w)) - 1; }
};
template <>
struct GroupBits<64> {
    using Word = unsigned long long;
    Word lower, lowerQuad;
    static constexpr int base = 0;
    __device__ __forceinline__ void init(int lane) {
        lower = (1ull << lane) - 1ull;
        lowerQuad = (1ull << (lane & ~3)) - 1ull;
    }
    __device__ __forceinline__ Word of(unsigned long long ballot) const { return ballot; }
    __device__ __forceinline__ static int count(Word w) { return __popcll(w); }
    __device__ __forceinline__ static int first(Word w) { return __ffsll(static_cast<long long>(w)) - 1; }
};

__device__ __forceinline__ uint32_t minU(uint32_t a, uint32_t b) { return a < b ? a : b; }
template <int kCtrl>
__device__ __forceinline__ uint32_t dppU(uint32_t x) {
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), kCtrl, 0xF, 0xF, true));
}
// Smallest x over the group, in every lane: within rows of 16 by DPP (one instruction a
// step, no LDS permute), across rows by the row and half swaps.
template <int G>
__device__ __forceinline__ uint32_t groupMin(uint32_t x) {
    x = minU(x, dppU<0xB1>(x));   // quad_perm [1,0,3,2]
    x = minU(x, dppU<0x4E>(x));   // quad_perm [2,3,0,1]
    if constexpr (G >= 8) x = minU(x, dppU<0x141>(x));   // row_half_mirror
    if constexpr (G >= 16) x = minU(x, dppU<0x140>(x));  // row_mirror
    if constexpr (G >= 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        x = minU(r[0], r[1]);
    }
    if constexpr (G == 64) {
        const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        x = minU(r[0], r[1]);
    }
    return x;
}
// The group's lane i receives lane i - 1's x, its first lane 0.
template <int G>
__device__ __forceinline__ uint32_t groupShiftUp(uint32_t x, int gl) {
    if constexpr (G <= 16) {
        const int v = __builtin_amdgcn_update_dpp(0, static_cast<int>(x), 0x111, 0xF, 0xF, false);
        return static_cast<uint32_t>(G < 16 && gl == 0 ? 0 : v);
    } else {
        const int v = __builtin_amdgcn_update_dpp(0, static_cast<int>(x), 0x138, 0xF, 0xF, false);
        return static_cast<uint32_t>(G == 32 && gl == 0 ? 0 : v);
    }
}
__device__ __forceinline__ uint32_t permuteU(int lane, uint32_t x) {
    return static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(lane << 2, static_cast<int>(x)));
}

// A (dist2, index) pair as one ordered integer: dist2 is non-negative, so its bits order
// as it does, and equal distances order by index.  (inf, INT_MAX) is an empty place; a
// NaN distance lies behind it and is never taken.
constexpr uint32_t kInfBits = 0x7f800000u;
constexpr uint32_t kNoPrim = 0x7fffffffu;
__device__ __forceinline__ unsigned long long pairKey(uint32_t d, uint32_t id) {
    return (static_cast<unsigned long long>(d) << 32) | id;
}

// Rank of a lane's child among its quad's four by box distance (no child: rank 3, or
// what is left).  The slot takes the key's two low bits, so no two keys are equal; the
// order only steers the walk.
__device__ __forceinline__ int quadRank(bool child, uint32_t dBits, int slot) {
    const uint32_t key = child ? (dBits & ~3u) | static_cast<uint32_t>(slot) : 0xfffffffcu | static_cast<uint32_t>(slot);
    int rank = dppU<0xB1>(key) < key ? 1 : 0;
    rank += dppU<0x4E>(key) < key ? 1 : 0;
    rank += dppU<0x1B>(key) < key ? 1 : 0;  // quad_perm [3,2,1,0]
    return rank;
}

// Entry `slot` of 4-wide node `id`: its box and child code (>= 0 a node, < 0 a leaf
// reference -(leaf slot + 1), kWideEmpty nothing).
struct WideNodes {
    const Wide4* __restrict__ wide;
    __device__ __forceinline__ int entry(int id, int slot, Box& box) const {
        const WideEntry e = wide[id].c[slot];
        box = entryBox(e);
        return e.child;
    }
};

// The same over binary nodes: entry `slot` of the up to four grandchildren of interior
// node `id` (a leaf child stands for itself in its first slot).
struct BinaryNodes {
    const Node2* __restrict__ nodes;
    __device__ __forceinline__ int entry(int id, int slot, Box& box) const {
        const int c = (slot & 2) != 0 ? nodes[id].right : nodes[id].left;
        Node2 cn = nodes[c];
        int code = c;
        if (cn.left < 0) {
            code = (slot & 1) != 0 ? kWideEmpty : cn.left;
        } else {
            code = (slot & 1) != 0 ? cn.right : cn.left;
            cn = nodes[code];
            code = cn.left < 0 ? cn.left : code;
        }
        box = nodeBox(cn);
        return code;
    }
};

// Closest / kNN walk of one query by a group of G lanes.  The group's quads expand up to
// G / 4 nodes of the walk per round from a stack in LDS, lane s of a quad testing entry s
// of its node.  The k-best list is spread one entry per lane, sorted by (dist2, index),
// for any k up to G (the group's lanes beyond k keep the entries that fell off the k
// best: they cost nothing and are never read).  A round's leaf candidates closer than the
// k-th go in one by one: each is broadcast to its group, and the entries behind its place
// move up one lane (a DPP shift; no ballot or place count).  kOne (k = 1): the group's
// smallest candidate by DPP.  Interior children are pushed nearest parent first and, within a parent,
// nearest on top; for Gaussians, whose leaf test costs the most, in box-distance order
// over the whole group.  A subtree or primitive is passed over only when its bound lies
// beyond the k-th distance, so the list ends as the k best by (dist2, index) whatever the
// walk order.
//
// Bound by VALU issue: the round is kept to as few instructions as possible.  The k-th
// key stands for the list's fill (an empty list's is infinite), masks and counts are
// 32-bit words of the group, the box test has no branches, reductions and shifts are DPP,
// and a leaf's primitive is loaded once its box is admitted (a quarter of them are).
// Against 64-bit masks, LDS permutes and short-circuit tests, kernel time on a
// 2M-triangle terrain with 100k queries: closest 277 -> 205 us, kNN16 443 -> 308 us; one
// path through all regions of the triangle distance instead of its exits: no faster here,
// 15 % slower around an icosphere (1.01 -> 1.16 ms).
template <typename L, bool kOne, int G, bool kStats, typename Nodes>
struct GroupNearest {
    static_assert(G == 16 || G == 32 || G == 64, "lanes per query");
    static constexpr bool kSortPushes = L::kKind == 2;
    static constexpr int kQuads = G / 4;                 // nodes a query expands per round
    static constexpr int kStack = kWaveStack / (64 / G);  // stack entries per query
    int k;             // list length, at most G (kOne: 1)
    uint32_t ld, lid;  // this lane's list entry (k > 1)
    uint32_t kd, kid;  // the list's k-th (the same in every lane)

    __device__ __forceinline__ void walk(const Nodes& nodes, const typename L::Item* __restrict__ prims,
                                         const int* __restrict__ primIds, V3 p, LdsInt* stk, int lane,
                                         uint32_t idMask, int& nodeTests, int& leafTests, int& overflow,
                                         int& opened) {
        const int gl = lane & (G - 1);  // lane within the group
        const int quad = gl >> 2;
        const int slot = lane & 3;
        GroupBits<G> gb;
        gb.init(lane);
        ld = kd = kInfBits;
        lid = kid = kNoPrim;
        if (gl == 0) stk[0] = 0;
        // A NaN query ends at the root, however many children wait.  (A check before the walk
        // holds the root's read until the query's: closest, 100k queries, 1 % more.)
        const int done = hasNaN(p) ? INT_MAX : 0;
        int sp = 1;
        do {
            int take = takeOf(sp);
            int node = -1;
            bool cut = false;
            if (quad < take) {
                const uint32_t v = static_cast<uint32_t>(stk[sp - 1 - quad]);
                cut = stackKey(v, idMask) > kd;
                node = cut ? -1 : static_cast<int>(v & idMask);
            }
            const unsigned long long cuts = __ballot(cut);
            if (cuts != 0 && gb.of(cuts) != 0) {
                // the bound has overtaken entries the quads would take: drop those of
                // the top G (order kept) and take again, so no quad idles on them
                const int look = sp < G ? sp : G;
                uint32_t v = 0;
                bool keep = false;
                if (gl < look) {
                    v = static_cast<uint32_t>(stk[sp - look + gl]);
                    keep = stackKey(v, idMask) <= kd;
                }
                const typename GroupBits<G>::Word kept = gb.of(__ballot(keep));
                if (keep) stk[sp - look + gb.count(kept & gb.lower)] = static_cast<int>(v);
                sp = sp - look + gb.count(kept);
                take = takeOf(sp);
                node = -1;
                if (quad < take) node = static_cast<int>(static_cast<uint32_t>(stk[sp - 1 - quad]) & idMask);
            }
            sp -= take;
            if (kStats && slot == 0 && node >= 0) ++opened;
            Box box{{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
            int ch = kWideEmpty;
            if (node >= 0) ch = nodes.entry(node, slot, box);
            const bool leaf = static_cast<uint32_t>(ch) > static_cast<uint32_t>(kWideEmpty);
            const uint32_t d = floatBits(boxDist2(p, box));
            const bool adm = (ch != kWideEmpty) & (d <= kd);
            if (kStats && adm) ++nodeTests;
            uint32_t cd = ~0u, cid = ~0u;
            bool better = false;
            if (adm & leaf) {
                if (kStats) ++leafTests;
                const uint32_t pid = static_cast<uint32_t>(primIds[-ch - 1]);
                const uint32_t dd = floatBits(L::dist2(p, prims[-ch - 1]));
                better = pairKey(dd, pid) < pairKey(kd, kid);
                cd = better ? dd : ~0u;
                cid = better ? pid : ~0u;
            }
            const unsigned long long bm = __ballot(better);
            if (bm != 0) {
                if constexpr (kOne) {
                    const uint32_t m = groupMin<G>(cd);
                    const uint32_t mi = groupMin<G>(cd == m ? cid : ~0u);
                    const bool got = m != ~0u;  // (a candidate is closer than the entry)
                    kd = got ? m : kd;
                    kid = got ? mi : kid;
                } else {
                    insertAll(gb, gb.of(bm), cd, cid, lane, gl);
                }
            }
            // interior children that survive the updated bound: quad j popped the j-th
            // nearest entry, so its children go above those of quads j+1..
            const bool push = adm & !leaf & (d <= kd);
            const unsigned long long pb = __ballot(push);
            if (pb != 0) {
                const typename GroupBits<G>::Word pm = gb.of(pb);
                const int pushes = gb.count(pm);
                const int top = sp + pushes;
                if (top > kStack) {  // deeper than the stack bound allows
                    if (gl == 0) overflow = 1;
                    sp = 0;
                } else {
                    if constexpr (kSortPushes) {  // all of the round's children in box-distance order
                        float pk = push ? bitsFloat(d) : kInf;
                        int pv = push ? ch : 0x7fffffff;
                        waveSortPairs(pk, pv, lane, G);
                        if (gl < pushes) stk[top - 1 - gl] = static_cast<int>(stackEntry(static_cast<uint32_t>(pv), floatBits(pk), idMask));
                    } else {
                        const int rank = quadRank(push, d, slot);
                        if (push) stk[top - 1 - gb.count(pm & gb.lowerQuad) - rank] = static_cast<int>(stackEntry(static_cast<uint32_t>(ch), d, idMask));
                    }
                    sp = top;
                }
            }
        } while (sp > done);
    }

    // Nodes to take from a stack of sp entries: one per quad, fewer when the stack could
    // otherwise outgrow its room (see kWaveStack).
    __device__ __forceinline__ static int takeOf(int sp) {
        const int room = kStack - kWaveHeadroom - sp;
        int width = kQuads;
        if (room < 3 * kQuads) width = room < 3 ? 1 : room / 3;
        return width < sp ? width : sp;
    }

    __device__ __forceinline__ void insertAll(const GroupBits<G>& gb, typename GroupBits<G>::Word rest, uint32_t cd,
                                              uint32_t cid, int lane, int gl) {
        while (__ballot(rest != 0) != 0) {
            // a group that has none left broadcasts the key behind all others
            const int src = rest != 0 ? gb.base + gb.first(rest) : lane;
            uint32_t c = permuteU(src, cd), ci = permuteU(src, cid);
            c = rest != 0 ? c : ~0u;
            rest &= rest - 1;
            const unsigned long long ck = pairKey(c, ci);
            const uint32_t pd = groupShiftUp<G>(ld, gl), pi = groupShiftUp<G>(lid, gl);
            const bool stays = pairKey(ld, lid) < ck;
            const bool here = pairKey(pd, pi) < ck;  // the entry below is closer: the candidate's place
            const uint32_t nd = here ? c : pd, ni = here ? ci : pi;
            ld = stays ? ld : nd;
            lid = stays ? lid : ni;
        }
        const int last = (lane & ~(G - 1)) + k - 1;
        kd = permuteU(last, ld);
        kid = permuteU(last, lid);
    }

    __device__ __forceinline__ void store(ClosestResult* __restrict__ dst, int gl) const {
        const uint32_t d = kOne ? kd : ld, i = kOne ? kid : lid;
        if (gl < (kOne ? 1 : k)) dst[gl] = i == kNoPrim ? ClosestResult{0u, -1} : ClosestResult{d, static_cast<int>(i)};
    }
};

// The walk over a plain tree: 64 / G queries per wave.
template <typename L, bool kOne, int G, bool kStats, typename Nodes>
__global__ __launch_bounds__(kBlock) void nearestWaveKernel(
    Nodes nodes, const typename L::Item* __restrict__ prims,
    const int* __restrict__ primIds, const V3* __restrict__ points, const uint32_t* __restrict__ order,
    int count, int k, int outStride, ClosestResult* __restrict__ out, unsigned long long* __restrict__ stats,
    uint32_t idMask) {
    __shared__ int lds[kWaveStack * (kBlock / 64)];
    const int lane = threadIdx.x & 63;
    const int qi = (xcdBlock() * (kBlock / 64) + (threadIdx.x >> 6)) * (64 / G) + lane / G;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    if (qi < count) {  // the same in the whole group
        const int q = order ? static_cast<int>(order[qi]) : qi;
        GroupNearest<L, kOne, G, kStats, Nodes> g;
        g.k = k;
        LdsInt* stk = (LdsInt*)(lds + (threadIdx.x >> 6) * kWaveStack + (lane / G) * g.kStack);
        g.walk(nodes, prims, primIds, points[q], stk, lane, idMask, nodeTests, leafTests, overflow, opened);
        g.store(out + static_cast<size_t>(q) * outStride, lane & (G - 1));
    }
    flushStats<kStats>(stats, nodeTests, leafTests, overflow, opened);
}

// Radius capture of one query by a group of G lanes (the layout above): every admitted
// interior child goes on the stack in lane order, hits are counted and the first `cap` of
// them kept in the query's slot of `capture`, in no particular order (radiusCompactKernel
// sorts each segment as it moves it).
template <typename L, bool kStats, int G, typename Nodes>
__global__ __launch_bounds__(kBlock) void radiusGroupKernel(
    Nodes nodes, const typename L::Item* __restrict__ prims, const int* __restrict__ primIds,
    const V3* __restrict__ points, const uint32_t* __restrict__ order, int count, float r2,
    int* __restrict__ counts, uint64_t* __restrict__ capture, unsigned long long* __restrict__ stats,
    int* __restrict__ maxCount, int cap) {
    constexpr int kQuads = G / 4;
    constexpr int kStack = kWaveStack / (64 / G);
    __shared__ int lds[kWaveStack * (kBlock / 64)];
    const int lane = threadIdx.x & 63;
    const int gl = lane & (G - 1);
    const int quad = gl >> 2;
    const int slot = lane & 3;
    const int qi = (xcdBlock() * (kBlock / 64) + (threadIdx.x >> 6)) * (64 / G) + lane / G;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    int found = 0;
    if (qi < count) {  // the same in the whole group
        const int q = order ? static_cast<int>(order[qi]) : qi;
        const V3 p = points[q];
        GroupBits<G> gb;
        gb.init(lane);
        LdsInt* stk = (LdsInt*)(lds + (threadIdx.x / G) * kStack);
        uint64_t* seg = capture + static_cast<long long>(q) * cap;
        if (gl == 0) stk[0] = 0;
        int sp = 1;
        while (sp > 0) {
            const int room = kStack - kWaveHeadroom - sp;
            int take = kQuads;
            if (room < 3 * kQuads) take = room < 3 ? 1 : room / 3;
            take = take < sp ? take : sp;
            int node = -1;
            if (quad < take) node = stk[sp - 1 - quad];
            sp -= take;
            if (kStats && slot == 0 && node >= 0) ++opened;
            Box box{{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
            int ch = kWideEmpty;
            if (node >= 0) ch = nodes.entry(node, slot, box);
            const bool leaf = static_cast<uint32_t>(ch) > static_cast<uint32_t>(kWideEmpty);
            const bool adm = (ch != kWideEmpty) & (boxDist2(p, box) <= r2);
            if (kStats && adm) ++nodeTests;
            const bool push = adm & !leaf;
            const unsigned long long pb = __ballot(push);
            if (pb != 0) {
                const typename GroupBits<G>::Word pm = gb.of(pb);
                const int pushes = gb.count(pm);
                if (sp + pushes > kStack) {  // deeper than the stack bound allows
                    if (gl == 0) overflow = 1;
                    break;
                }
                if (push) stk[sp + gb.count(pm & gb.lower)] = ch;
                sp += pushes;
            }
            bool hit = false;
            float d2 = 0.0f;
            uint32_t pid = 0;
            if (adm & leaf) {
                if (kStats) ++leafTests;
                pid = static_cast<uint32_t>(primIds[-ch - 1]);
                d2 = L::dist2(p, prims[-ch - 1]);
                hit = d2 <= r2;
            }
            const unsigned long long hb = __ballot(hit);
            if (hb != 0) {
                const typename GroupBits<G>::Word hm = gb.of(hb);
                if (hit) {
                    const int at = found + gb.count(hm & gb.lower);
                    if (at < cap) seg[at] = (static_cast<uint64_t>(floatBits(d2)) << 32) | pid;
                }
                found += gb.count(hm);
            }
        }
        if (gl == 0) counts[q] = found;
    }
    waveMaxAtomic(maxCount, found);
    flushStats<kStats>(stats, nodeTests, leafTests, overflow, opened);
}

// Batched scenes by groups: G lanes walk one query of the batch's queue on its own
// scene's 4-wide tree (scene s: items from primOff[s], nodes from wideRoot[s]).  Queries
// lie scene by scene, so an XCD's contiguous range stays on a few scenes' nodes.
template <typename L, bool kOne, int G, int kBT>
__global__ __launch_bounds__(kBT) void batchGroupKernel(
    const Wide4* __restrict__ wide, const int* __restrict__ wideRoot, const typename L::Item* __restrict__ prims,
    const int* __restrict__ primIds, const int* __restrict__ primOff, const V3* __restrict__ points,
    const int* __restrict__ qScene, const uint32_t* __restrict__ order, int count, int k, int outStride,
    ClosestResult* __restrict__ out) {
    __shared__ int lds[kWaveStack * (kBT / 64)];
    const int lane = threadIdx.x & 63;
    const int qi = (xcdBlock() * (kBT / 64) + (threadIdx.x >> 6)) * (64 / G) + lane / G;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    if (qi < count) {  // the same in the whole group
        const int q = order ? static_cast<int>(order[qi]) : qi;
        const int s = qScene[q];
        const int ps = primOff[s], wr = wideRoot[s];
        GroupNearest<L, kOne, G, false, WideNodes> g;
        g.k = k;
        LdsInt* stk = (LdsInt*)(lds + (threadIdx.x >> 6) * kWaveStack + (lane / G) * g.kStack);
        g.walk(WideNodes{wide + wr}, prims + ps, primIds + ps, points[q], stk, lane, stackIdMask(wideRoot[s + 1] - wr),
               nodeTests, leafTests, overflow, opened);
        g.store(out + static_cast<size_t>(q) * outStride, lane & (G - 1));
    }
    flushStats<false>(nullptr, nodeTests, leafTests, overflow, opened);
}

// Closest-hit walk of one ray by a group of G lanes (the layout of the query walks above).
// A round's hits reduce to the group's smallest (t, then, when saved, primitive index --
// the lane kernels' rule for equal t), boxes are tested against the best t so far with
// the lane kernels' slack, and popped entries whose entry distance (kept in the stack
// entry, truncated: a lower bound; not below zero there) is beyond it are dropped.
// Interior children go on the stack nearest parent first, each parent's nearest on top.
template <int G, bool kStats, bool kSave, typename Nodes>
__global__ __launch_bounds__(kBlock) void rayWaveKernel(Nodes nodes, const Tri* __restrict__ tris,
                                                        const Ray* __restrict__ rays,
                                                        const uint32_t* __restrict__ order, int count,
                                                        uint64_t* __restrict__ out,
                                                        unsigned long long* __restrict__ stats,
                                                        const int* __restrict__ primIds,
                                                        int* __restrict__ hitPrim, uint32_t idMask) {
    constexpr int kQuads = G / 4;
    constexpr int kStack = kWaveStack / (64 / G);
    __shared__ int lds[kStack * (kBlock / G)];
    const int lane = threadIdx.x & 63;
    const int gl = lane & (G - 1);
    const int quad = gl >> 2;
    const int slot = lane & 3;
    const int qi = (xcdBlock() * (kBlock / 64) + (threadIdx.x >> 6)) * (64 / G) + lane / G;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    if (qi < count) {  // the same in the whole group
        const int q = order ? static_cast<int>(order[qi]) : qi;
        const Ray ray = rays[q];
        const RayPre pre = rayPrepare(ray);
        GroupBits<G> gb;
        gb.init(lane);
        float best = ray.tMax;
        bool any = false;
        uint32_t bestId = kNoPrim;
        LdsInt* stk = (LdsInt*)(lds + (threadIdx.x / G) * kStack);
        if (gl == 0) stk[0] = 0;
        int sp = 1;
        while (sp > 0) {
            int take = kQuads;
            const int room = kStack - kWaveHeadroom - sp;
            if (room < 3 * kQuads) take = room < 3 ? 1 : room / 3;
            take = take < sp ? take : sp;
            int node = -1;
            if (quad < take) {
                const uint32_t v = static_cast<uint32_t>(stk[sp - 1 - quad]);
                if (bitsFloat(stackKey(v, idMask)) <= stackReach(best)) node = static_cast<int>(v & idMask);
            }
            sp -= take;
            if (kStats && slot == 0 && node >= 0) ++opened;
            Box box{{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
            int ch = kWideEmpty;
            if (node >= 0) ch = nodes.entry(node, slot, box);
            const bool leaf = static_cast<uint32_t>(ch) > static_cast<uint32_t>(kWideEmpty);
            float tEnter;
            const bool adm = rayBoxPre(pre, box, best, tEnter) & (ch != kWideEmpty);
            if (kStats && adm) ++nodeTests;
            float ht = kInf;
            uint32_t hid = ~0u;
            bool hit = false;
            if (adm & leaf) {
                if (kStats) ++leafTests;
                float t;
                // the lane kernels' rule: a nearer hit, or an equal one once there is a hit
                if (rayTri(ray, tris[-ch - 1], t) && (t < best || (any && t == best))) {
                    ht = t;
                    hit = true;
                    if (kSave) hid = static_cast<uint32_t>(primIds[-ch - 1]);
                }
            }
            const unsigned long long hb = __ballot(hit);
            if (hb != 0) {
                const uint32_t mine = hit ? orderedBits(ht) : ~0u;
                const uint32_t m = groupMin<G>(mine);
                const bool got = m != ~0u;
                const float t = got ? fromOrderedBits(m) : best;
                if (kSave) {
                    const uint32_t mi = groupMin<G>(mine == m ? hid : ~0u);
                    bestId = !got ? bestId : (t < best || mi < bestId ? mi : bestId);
                }
                best = t;
                any |= got;
            }
            const bool push = adm & !leaf & (tEnter <= rayReach(best));
            const unsigned long long pb = __ballot(push);
            if (pb != 0) {
                const typename GroupBits<G>::Word pm = gb.of(pb);
                const int top = sp + gb.count(pm);
                if (top > kStack) {  // deeper than the stack bound allows
                    if (gl == 0) overflow = 1;
                    sp = 0;
                } else {
                    const uint32_t key = floatBits(fmaxf(tEnter, 0.0f));
                    const int rank = quadRank(push, key, slot);
                    if (push) stk[top - 1 - gb.count(pm & gb.lowerQuad) - rank] = static_cast<int>(stackEntry(static_cast<uint32_t>(ch), key, idMask));
                    sp = top;
                }
            }
        }
        if (gl == 0) {
            out[q] = any ? ((uint64_t{1} << 32) | floatBits(best)) : 0ull;
            if (kSave) hitPrim[q] = any ? static_cast<int>(bestId) : -1;
        }
    }
    flushStats<kStats>(stats, nodeTests, leafTests, overflow, opened);
}

// ---- radius: count and fill passes ---------------------------------------------------
// kFill = false counts matches per query; kFill = true writes the 64-bit keys
// (dist2 bits << 32 | index) into the query's CSR segment (bounded by the next
// offset, so a fill can never write past its segment).
template <typename L, bool kWide, bool kFill, bool kStats>
__global__ __launch_bounds__(kBlock) void radiusKernel(
    const Node2* __restrict__ nodes, const Wide4* __restrict__ wide,
    const typename L::Item* __restrict__ prims, const int* __restrict__ primIds,
    const V3* __restrict__ points, const uint32_t* __restrict__ order, int count, float r2,
    int* __restrict__ counts, const int* __restrict__ offsets, uint64_t* __restrict__ keys,
    unsigned long long* __restrict__ stats, int* __restrict__ maxCount) {
    __shared__ int lds[kLdsDepth * kBlock];
    int queryHits = 0;
    const int i = xcdBlock() * kBlock + threadIdx.x;
    int nodeTests = 0, leafTests = 0, overflow = 0, opened = 0;
    if (i < count) {
        const int q = order ? static_cast<int>(order[i]) : i;
        const V3 p = points[q];
        int found = 0;
        int write = kFill ? offsets[q] : 0;
        const int end = kFill ? offsets[q + 1] : 0;
        auto leafTest = [&](int slot) {
            ++leafTests;
            const float d2 = L::dist2(p, prims[slot]);
            if (d2 <= r2) {
                if (kFill) {
                    if (write < end)
                        keys[write++] = (static_cast<uint64_t>(floatBits(d2)) << 32) |
                                        static_cast<uint32_t>(primIds[slot]);
                } else {
                    ++found;
                }
            }
        };
        LaneStack st;
        SpillArea spill;
        st.init(lds);
        int id = -1;
        if (!kWide) {
            const Node2 root = nodes[0];
            if (boxDist2(p, nodeBox(root)) <= r2) {
                ++nodeTests;
                id = 0;
            }
        } else {
            id = 0;
        }
        while (id >= 0) {
            if (kStats) ++opened;
            int c[4] = {kWideEmpty, kWideEmpty, kWideEmpty, kWideEmpty};
            bool ok[4] = {false, false, false, false};
            if (!kWide) {
                const Node2 nd = nodes[id];
                const int kid[2] = {nd.left, nd.right};
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const Node2 cn = nodes[kid[s]];
                    if (boxDist2(p, nodeBox(cn)) > r2) continue;
                    ++nodeTests;
                    if (cn.left < 0) {
                        leafTest(-cn.left - 1);
                    } else {
                        c[s] = kid[s];
                        ok[s] = true;
                    }
                }
            } else {
                WideEntry e[4];
                loadWide(wide, id, e);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int ch = e[s].child;
                    if (ch == kWideEmpty || boxDist2(p, entryBox(e[s])) > r2) continue;
                    ++nodeTests;
                    if (ch < 0) {
                        leafTest(-ch - 1);
                    } else {
                        c[s] = ch;
                        ok[s] = true;
                    }
                }
            }
            id = descend(c, ok, st, spill, overflow);
        }
        if (!kFill) counts[q] = found;
        queryHits = found;
    }
    if (!kFill) waveMaxAtomic(maxCount, queryHits);
    flushStats<kStats>(stats, nodeTests, leafTests, overflow, opened);
}

// ---- segment sort ----------------------------------------------------------------
// Sorts each CSR segment ascending.  One wave per segment of up to kWaveCap keys
// (bitonic network in LDS); longer segments are handled by one workgroup each
// with a bitonic network over up to kBlockCap keys.
constexpr int kWaveCap = 256;
constexpr int kBlockCap = 8192;

// Bitonic sort of cap (a power of two, at least 4) keys in LDS by `lanes` threads (a wave,
// or a whole workgroup), ascending.  A chain of LDS round trips: a round therefore does two
// steps, strides 2 h and h, on four keys in registers (the last stride alone when their
// number is odd), and a thread's four loads are in flight together -- about 30 rounds for
// 1,024 keys instead of 55.  A wave's 64 consecutive quads lie in 256 consecutive keys
// while h <= 64, so only rounds of longer strides and the round after them need the
// workgroup's barrier; within a wave LDS accesses run in order (the fence keeps the
// compiler to it).
__device__ __forceinline__ void orderKeys(uint64_t& a, uint64_t& b, bool up) {
    const bool swap = (a > b) == up;  // (equal keys: either way)
    const uint64_t x = swap ? b : a, y = swap ? a : b;
    a = x;
    b = y;
}
__device__ __forceinline__ void bitonicLds(uint64_t* buf, int cap, int lane, int lanes) {
    bool far = false;  // the round before reached across waves
    for (int size = 2; size <= cap; size <<= 1) {
        int stride = size >> 1;
        while (stride > 0) {
            const bool two = stride > 1;
            const int h = two ? stride >> 1 : 1;
            const bool reach = h > 64;
            if (lanes > 64 && (reach || far)) __syncthreads();
            else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            far = reach;
            for (int p = lane; p < cap >> 2; p += lanes) {
                const int i = ((p & ~(h - 1)) << 2) | (p & (h - 1));
                uint64_t k0 = buf[i], k1 = buf[i + h], k2 = buf[i + 2 * h], k3 = buf[i + 3 * h];
                const bool up = (i & size) == 0 || size == cap;
                const bool up2 = ((i + 2 * h) & size) == 0 || size == cap;  // (differs at size 2 only)
                if (two) {
                    orderKeys(k0, k2, up);
                    orderKeys(k1, k3, up);
                }
                orderKeys(k0, k1, up);
                orderKeys(k2, k3, up2);
                buf[i] = k0;
                buf[i + h] = k1;
                buf[i + 2 * h] = k2;
                buf[i + 3 * h] = k3;
            }
            stride >>= two ? 2 : 1;
        }
    }
    if (lanes > 64) __syncthreads();
    else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

__global__ __launch_bounds__(kBlock) void segSortWaveKernel(const int* __restrict__ offsets,
                                                            uint64_t* __restrict__ keys,
                                                            int count) {
    __shared__ uint64_t smem[kBlock / 64][kWaveCap];
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int seg = blockIdx.x * (kBlock / 64) + w;
    if (seg >= count) return;
    const int begin = offsets[seg];
    const int m = offsets[seg + 1] - begin;
    if (m <= 1 || m > kWaveCap) return;
    int cap = 4;
    while (cap < m) cap <<= 1;
    uint64_t* buf = smem[w];
    for (int i = lane; i < cap; i += 64) buf[i] = i < m ? keys[begin + i] : ~0ull;
    __builtin_amdgcn_wave_barrier();
    bitonicLds(buf, cap, lane, 64);
    for (int i = lane; i < m; i += 64) keys[begin + i] = buf[i];
}

// Segments of kWaveCap+1 .. kBlockCap keys, listed by segClassifyKernel (info[0] of
// them); each workgroup takes list entries blockIdx.x, blockIdx.x + gridDim.x, ...
__global__ __launch_bounds__(kBlock) void segSortBlockKernel(const int* __restrict__ offsets,
                                                             const int* __restrict__ segList,
                                                             const int* __restrict__ info,
                                                             uint64_t* __restrict__ keys) {
    extern __shared__ uint64_t dyn[];
    const int listed = info[0];
    for (int e = blockIdx.x; e < listed; e += gridDim.x) {
        const int seg = segList[e];
        const int begin = offsets[seg];
        const int m = offsets[seg + 1] - begin;
        int cap = 2;
        while (cap < m) cap <<= 1;
        for (int i = threadIdx.x; i < cap; i += kBlock) dyn[i] = i < m ? keys[begin + i] : ~0ull;
        __syncthreads();
        bitonicLds(dyn, cap, threadIdx.x, kBlock);
        for (int i = threadIdx.x; i < m; i += kBlock) keys[begin + i] = dyn[i];
        __syncthreads();
    }
}

// Collects segments longer than the wave cap; info[0] = count of block-sized ones,
// info[1] = count of segments beyond the block cap, info[2] = max segment length.
__global__ void segClassifyKernel(const int* __restrict__ offsets, int count,
                                  int* __restrict__ blockList, int* __restrict__ hugeList,
                                  int* __restrict__ info) {
    const int s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= count) return;
    const int m = offsets[s + 1] - offsets[s];
    if (m > kWaveCap && m <= kBlockCap) blockList[atomicAdd(&info[0], 1)] = s;
    if (m > kBlockCap) hugeList[atomicAdd(&info[1], 1)] = s;
}

__global__ void zeroIntsKernel(int* __restrict__ p, int n) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void splitKeysKernel(const uint64_t* __restrict__ keys, int m, uint32_t* __restrict__ lo,
                                uint32_t* __restrict__ hi) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= m) return;
    const uint64_t k = keys[i];
    lo[i] = static_cast<uint32_t>(k);
    hi[i] = static_cast<uint32_t>(k >> 32);
}

__global__ void gatherU32Kernel(const uint32_t* __restrict__ src, const uint32_t* __restrict__ idx, int m,
                                uint32_t* __restrict__ dst) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < m) dst[i] = src[idx[i]];
}

// keys[i] = hiSorted[i] << 32 | lo[ord[i]]
__global__ void joinKeysKernel(const uint32_t* __restrict__ hiSorted, const uint32_t* __restrict__ lo,
                               const uint32_t* __restrict__ ord, int m, uint64_t* __restrict__ keys) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < m) keys[i] = (static_cast<uint64_t>(hiSorted[i]) << 32) | lo[ord[i]];
}

// ---- Morton reordering of queries / rays ------------------------------------------------
// quantize10 over the query (or ray-origin) bounds (src/gpu/morton.h:8-29).
__device__ __forceinline__ uint32_t quant10(float v, float lo, float hi) {
    if (!(hi > lo)) return 0u;
    float f = (v - lo) / (hi - lo);
    f = fminf(fmaxf(f, 0.0f), 1.0f);
    return static_cast<uint32_t>(f * 1023.0f + 0.5f);
}
__device__ __forceinline__ uint32_t spread10b(uint32_t v) {
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__global__ void pointBoundsInitKernel(uint32_t* __restrict__ bb) {
    if (threadIdx.x < 3) bb[threadIdx.x] = orderedBits(kInf);
    if (threadIdx.x >= 3 && threadIdx.x < 6) bb[threadIdx.x] = orderedBits(-kInf);
}

// Bounds of points laid out with `stride` floats per element (3 for points, 8 for
// rays: origin first, 8 + 3 for ray directions).  Every workgroup's six atomics meet at
// the same six words, so there is one set per workgroup and at most kBoundsGrid of them
// (one per wave of up to 1,024 workgroups: 262k points 73 us).
constexpr int kBoundsGrid = 256;
__global__ void pointBoundsKernel(const float* __restrict__ base, int stride, int count,
                                  uint32_t* __restrict__ bb) {
    __shared__ uint32_t part[6][kBlock / 64];
    float lo0 = kInf, lo1 = kInf, lo2 = kInf, hi0 = -kInf, hi1 = -kInf, hi2 = -kInf;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < count; i += kBlock * gridDim.x) {
        const float* p = base + static_cast<size_t>(i) * stride;
        lo0 = fminf(lo0, p[0]);
        lo1 = fminf(lo1, p[1]);
        lo2 = fminf(lo2, p[2]);
        hi0 = fmaxf(hi0, p[0]);
        hi1 = fmaxf(hi1, p[1]);
        hi2 = fmaxf(hi2, p[2]);
    }
    const uint32_t v[6] = {reduce64<MinU>(orderedBits(lo0)), reduce64<MinU>(orderedBits(lo1)),
                           reduce64<MinU>(orderedBits(lo2)), reduce64<MaxU>(orderedBits(hi0)),
                           reduce64<MaxU>(orderedBits(hi1)), reduce64<MaxU>(orderedBits(hi2))};
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < 6; ++k) part[k][threadIdx.x >> 6] = v[k];
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int k = static_cast<int>(threadIdx.x);
        uint32_t x = part[k][0];
        for (int w = 1; w < kBlock / 64; ++w) x = k < 3 ? MinU::op(x, part[k][w]) : MaxU::op(x, part[k][w]);
        if (k < 3) atomicMin(&bb[k], x);
        else atomicMax(&bb[k], x);
    }
}

// fixedBox: use [-1,1]^3 (ray directions) instead of the measured bounds.
__global__ void mortonKeysKernel(const float* __restrict__ base, int stride, int count,
                                 const uint32_t* __restrict__ bb, int fixedBox, int drop,
                                 uint32_t* __restrict__ keys, uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[4][256];
    for (int i = threadIdx.x; i < 4 * 256; i += kBlock) (&h[0][0])[i] = 0u;
    float lo[3], hi[3];
    for (int a = 0; a < 3; ++a) {
        lo[a] = fixedBox ? -1.0f : fromOrderedBits(bb[a]);
        hi[a] = fixedBox ? 1.0f : fromOrderedBits(bb[3 + a]);
    }
    __syncthreads();
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < count; i += kBlock * gridDim.x) {
        const float* p = base + static_cast<size_t>(i) * stride;
        const uint32_t code = (spread10b(quant10(p[0], lo[0], hi[0])) |
                              (spread10b(quant10(p[1], lo[1], hi[1])) << 1) |
                              (spread10b(quant10(p[2], lo[2], hi[2])) << 2)) >> drop;
        keys[i] = code;
        atomicAdd(&h[0][code & 255u], 1u);
        atomicAdd(&h[1][(code >> 8) & 255u], 1u);
        atomicAdd(&h[2][(code >> 16) & 255u], 1u);
        atomicAdd(&h[3][code >> 24], 1u);
    }
    __syncthreads();
    flushHistogram(&h[0][0], 4 * 256, hist);
}

// Sort keys of a batch's queries, one workgroup per scene: the bounds of the scene's points,
// then (scene, Morton code within those bounds) per point, and the digit counts.  Queries
// lie scene by scene, so no pass has to look a point's scene up and the bounds need no
// atomics.
constexpr int kBatchKeysBlock = 1024;
__global__ __launch_bounds__(kBatchKeysBlock) void batchQueryKeysKernel(const V3* __restrict__ points,
                                                                        const int* __restrict__ qOff, int codeBits,
                                                                        uint32_t* __restrict__ keys,
                                                                        uint32_t* __restrict__ hist) {
    __shared__ uint32_t part[6][kBatchKeysBlock / 64];
    __shared__ uint32_t h[4][256];
    const int sc = static_cast<int>(blockIdx.x);
    const int begin = qOff[sc], end = qOff[sc + 1];
    if (begin == end) return;  // the same for the whole workgroup
    for (int i = threadIdx.x; i < 4 * 256; i += kBatchKeysBlock) (&h[0][0])[i] = 0u;
    uint32_t v[6] = {~0u, ~0u, ~0u, 0u, 0u, 0u};
    for (int i = begin + static_cast<int>(threadIdx.x); i < end; i += kBatchKeysBlock) {
        const V3 p = points[i];
        const uint32_t o[3] = {orderedBits(p.x), orderedBits(p.y), orderedBits(p.z)};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            v[a] = MinU::op(v[a], o[a]);
            v[3 + a] = MaxU::op(v[3 + a], o[a]);
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        v[a] = reduce64<MinU>(v[a]);
        v[3 + a] = reduce64<MaxU>(v[3 + a]);
    }
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < 6; ++k) part[k][wave] = v[k];
    }
    __syncthreads();
    float lo[3], hi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        uint32_t l = ~0u, u = 0u;
        for (int w = 0; w < kBatchKeysBlock / 64; ++w) {
            l = MinU::op(l, part[a][w]);
            u = MaxU::op(u, part[3 + a][w]);
        }
        lo[a] = fromOrderedBits(l);
        hi[a] = fromOrderedBits(u);
    }
    for (int i = begin + static_cast<int>(threadIdx.x); i < end; i += kBatchKeysBlock) {
        const V3 p = points[i];
        const uint32_t code = (spread10b(quant10(p.x, lo[0], hi[0])) | (spread10b(quant10(p.y, lo[1], hi[1])) << 1) |
                               (spread10b(quant10(p.z, lo[2], hi[2])) << 2)) >> (30 - codeBits);
        const uint32_t key = (static_cast<uint32_t>(sc) << codeBits) | code;
        keys[i] = key;
        atomicAdd(&h[0][key & 255u], 1u);
        atomicAdd(&h[1][(key >> 8) & 255u], 1u);
        atomicAdd(&h[2][(key >> 16) & 255u], 1u);
        atomicAdd(&h[3][key >> 24], 1u);
    }
    __syncthreads();
    flushHistogram(&h[0][0], 4 * 256, hist);
}

__global__ void zeroU64Kernel(unsigned long long* __restrict__ p, int n) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

}  // namespace

// ---------------------------------------------------------------------------------------
// Host launchers.

void zeroInts(int* p, int n, hipStream_t s) {
    zeroIntsKernel<<<blocksFor(n, kBlock), kBlock, 0, s>>>(p, n);
}

void zeroStats(unsigned long long* stats, hipStream_t s) {
    zeroU64Kernel<<<blocksFor(kStatWords, kBlock), kBlock, 0, s>>>(stats, kStatWords);
}

void mortonOrder(const float* base, int stride, int count, int boxMode, SortWorkspace& ws,
                 uint32_t* keys, uint32_t* keysSorted, uint32_t* orderOut, uint32_t* bb,
                 hipStream_t s) {
    // The order only steers locality (results do not depend on it), so the code is
    // cut to whole 8-bit digits: the top 16 bits up to 262,144 elements (at most four
    // per cell; the 100k-query terrain walks measured no slower than on the full
    // code), 24 up to 16M, all 30 above -- one or two sort passes fewer.
    int passes = 4, drop = 0;
    if (count <= (1 << 18)) {
        passes = 2;
        drop = 14;
    } else if (count <= (1 << 24)) {
        passes = 3;
        drop = 6;
    }
    ws.reserve(static_cast<size_t>(count));
    sortClear(ws, static_cast<size_t>(count), passes, s);
    int grid = blocksFor(count, kBlock * 4);
    if (grid < 1) grid = 1;
    if (grid > 1024) grid = 1024;
    if (boxMode == kBoxMeasure) {
        pointBoundsInitKernel<<<1, 64, 0, s>>>(bb);
        pointBoundsKernel<<<grid < kBoundsGrid ? grid : kBoundsGrid, kBlock, 0, s>>>(base, stride, count, bb);
    }
    mortonKeysKernel<<<grid, kBlock, 0, s>>>(base, stride, count, bb, boxMode == kBoxUnit ? 1 : 0, drop,
                                             keys, ws.hist.p);
    hipCheck(hipGetLastError(), "morton keys");
    sortPairs(ws, keys, nullptr, keysSorted, orderOut, static_cast<size_t>(count), passes, s);
}

bool batchQueryOrder(const V3* points, const int* qOff, int n, int scenes, int maxPerScene, SortWorkspace& ws,
                     uint32_t* keys, uint32_t* keysSorted, uint32_t* order, hipStream_t s) {
    if (maxPerScene > kBatchOrderMax) return false;
    if (n <= 0) return true;
    // the scene's bits and as much of the Morton code as whole digits leave room for: the
    // order steers locality only
    int sceneBits = 1;
    while ((1LL << sceneBits) < scenes) ++sceneBits;
    const int passes = sceneBits <= 12 ? 3 : 4;
    const int codeBits = 8 * passes - sceneBits;
    ws.reserve(static_cast<size_t>(n));
    sortClear(ws, static_cast<size_t>(n), passes, s);
    batchQueryKeysKernel<<<scenes, kBatchKeysBlock, 0, s>>>(points, qOff, codeBits, keys, ws.hist.p);
    hipCheck(hipGetLastError(), "batch query keys");
    sortPairs(ws, keys, nullptr, keysSorted, order, static_cast<size_t>(n), passes, s);
    return true;
}

// 0 automatic, 1 one lane per query, 2 four lanes per query, 3 one wave per query,
// 4 closest / kNN and rays tuned whatever the query count, 5 / 6 16 / 32 lanes per query
int gTraversalMode = 0;

// Shapes of a walk over 4-wide nodes.
// (Group8 / 16 / 32: that many lanes per query; Group8 serves rays only.)
enum NearestShape : int {
    kShapeLane = 0, kShapeQuad = 1, kShapeWave = 2, kShapeGroup16 = 3, kShapeGroup32 = 4, kShapeGroup8 = 5
};

// Tuned shapes.  The best shape depends on how long and how uneven the walks are, which
// the query count alone does not tell: 262,144 closest queries on the terrain run fastest
// 16 lanes per query (410 us, one wave per query 597), as many in and around an icosphere
// -- long walks of very different lengths -- one wave per query (970 us against 1312).
// From kTuneFrom queries on a call for a (tree, k class, query count octave) times the
// three group shapes on its own queries and keeps the fastest (tunedShape): the second such
// call, or the first when no like call -- a tree of that leaf kind and size octave, that k
// class and count octave -- has been timed yet.  The first call else takes the shape of the
// last like call that was: a mesh that moves is a new tree every step, walked once (262,144
// queries around a 328k-triangle icosphere rebuilt each step: 2780 us a step with the
// timing in it, 1600 without).
constexpr int kTuneFrom = 65536;

struct TuneKey {
    uint64_t tree;  // the topology's serial number: the next tree in the same memory is another one
    int kind, K, octave;
    bool operator<(const TuneKey& o) const {
        return std::tie(tree, kind, K, octave) < std::tie(o.tree, o.kind, o.K, o.octave);
    }
};
static std::mutex gTuneMutex;
static std::map<TuneKey, int> gTuned;  // by tree: the shape, or kCalledOnce (not timed yet)
static std::map<TuneKey, int> gLike;   // by the tree's size octave: the last shape timed
constexpr int kCalledOnce = -1;
constexpr size_t kKeptMax = 4096;  // entries of gTuned; more are of trees in their thousands, all forgotten

static int octaveOf(int count) {
    int octave = 0;
    while ((2LL << octave) <= count) ++octave;
    return octave;
}

// The shape kept for this call (gTuneMutex held), or that of the last like call, or kCalledOnce.
static int keptShape(const TuneKey& key, int wideCount) {
    const auto own = gTuned.find(key);
    if (own != gTuned.end() && own->second != kCalledOnce) return own->second;
    TuneKey like = key;
    like.tree = static_cast<uint64_t>(octaveOf(wideCount));
    const auto it = gLike.find(like);
    return it != gLike.end() ? it->second : kCalledOnce;
}

static void keepShape(const TuneKey& key, int wideCount, int shape) {
    std::lock_guard<std::mutex> lock(gTuneMutex);
    if (gTuned.size() >= kKeptMax) gTuned.clear();
    gTuned[key] = shape;
    TuneKey like = key;
    like.tree = static_cast<uint64_t>(octaveOf(wideCount));
    gLike[like] = shape;
}

void forgetShapes(uint64_t serial) {
    std::lock_guard<std::mutex> lock(gTuneMutex);
    gTuned.erase(gTuned.lower_bound({serial, 0, 0, 0}), gTuned.lower_bound({serial + 1, 0, 0, 0}));
}

int keptShapes() {
    std::lock_guard<std::mutex> lock(gTuneMutex);
    int kept = 0;
    for (const auto& e : gTuned) kept += e.second != kCalledOnce ? 1 : 0;
    return kept;
}

// G lanes per ray, over the 4-wide nodes or, with a.wide false, the binary ones.
template <int G, bool kSave, typename Nodes>
static void launchRayGroupOn(Nodes nodes, int idCount, const TraverseArgs& a, const Ray* rays, int count,
                             uint64_t* out, int* hitPrim, unsigned long long* stats, hipStream_t s) {
    const Tri* tris = static_cast<const Tri*>(a.items);
    const uint32_t idMask = stackIdMask(idCount);
    const int grid = blocksFor(count, (kBlock / 64) * (64 / G));
    if (stats)
        rayWaveKernel<G, true, kSave><<<grid, kBlock, 0, s>>>(nodes, tris, rays, a.order, count, out, stats, a.primIds, hitPrim, idMask);
    else
        rayWaveKernel<G, false, kSave><<<grid, kBlock, 0, s>>>(nodes, tris, rays, a.order, count, out, nullptr, a.primIds, hitPrim, idMask);
}
template <int G, bool kSave>
static void launchRayGroup(const TraverseArgs& a, const Ray* rays, int count, uint64_t* out, int* hitPrim,
                           unsigned long long* stats, hipStream_t s) {
    if (a.wide)
        launchRayGroupOn<G, kSave>(WideNodes{a.wideNodes}, a.wideCount, a, rays, count, out, hitPrim, stats, s);
    else
        launchRayGroupOn<G, kSave>(BinaryNodes{a.nodes}, a.nodeCount, a, rays, count, out, hitPrim, stats, s);
}

template <bool kSave>
static void launchRayShape(int shape, const TraverseArgs& a, const Ray* rays, int count, uint64_t* out,
                           int* hitPrim, unsigned long long* stats, hipStream_t s) {
    const Tri* tris = static_cast<const Tri*>(a.items);
    if (shape == kShapeWave) {
        launchRayGroup<64, kSave>(a, rays, count, out, hitPrim, stats, s);
    } else if (shape == kShapeGroup32) {
        launchRayGroup<32, kSave>(a, rays, count, out, hitPrim, stats, s);
    } else if (shape == kShapeGroup16) {
        launchRayGroup<16, kSave>(a, rays, count, out, hitPrim, stats, s);
    } else if (shape == kShapeGroup8) {
        launchRayGroup<8, kSave>(a, rays, count, out, hitPrim, stats, s);
    } else {
        const int grid = blocksFor(count, kBlock);
        if (stats)
            rayWideKernel<true, kSave><<<grid, kBlock, 0, s>>>(a.wideNodes, tris, rays, a.order, count, out, stats,
                                                              a.primIds, hitPrim, stackIdMask(a.wideCount));
        else
            rayWideKernel<false, kSave><<<grid, kBlock, 0, s>>>(a.wideNodes, tris, rays, a.order, count, out,
                                                               nullptr, a.primIds, hitPrim, stackIdMask(a.wideCount));
    }
}

// Lanes per ray by the number of rays (same bits).  Small sets are latency chains that
// more lanes shorten; at a million the lane kernel needs the fewest instructions on
// coherent rays.  Measured (kernel us, city SAH tree, cosine rays, 4-wide: 1 / 8 / 16 / 32 /
// 64 lanes): 1k 140 / - / 16 / 14 / 13, 4k 117 / 25 / 18 / 14 / 15, 16k - / - / 24 / 25 /
// 35, 64k 168 / 51 / 51 / 71 / 111, 262k 187 / 128 / 155 / 250 / 409, 1M 477 / 430 / 561 /
// 939 / 1511; straight down, 262k 107 / 101 / 151, 1M 242 / 326 / 534; around an
// icosphere 64k 186 / 61 / 68, 262k 245 / 191 / 220.  Binary nodes cross over alike.  Mode
// 1 forces one lane, mode 3 one wave; mode 4 times one lane against one wave on the first
// call for a 4-wide tree, save flag and ray-count octave.
constexpr int kRayLaneFrom = 393216;
template <bool kSave>
static int rayShape(const TraverseArgs& a, const Ray* rays, int count, uint64_t* out, int* hitPrim,
                    hipStream_t s) {
    if (gTraversalMode == 1) return kShapeLane;
    if (gTraversalMode == 3) return a.wide ? kShapeWave : kShapeLane;
    if (gTraversalMode != 4 || !a.wide) {
        if (count < 3072) return kShapeWave;
        if (count < 12288) return kShapeGroup32;
        if (count < 49152) return kShapeGroup16;
        return count < kRayLaneFrom ? kShapeGroup8 : kShapeLane;
    }
    const TuneKey key{a.serial, 100 + (kSave ? 1 : 0), 0, octaveOf(count)};
    {
        std::lock_guard<std::mutex> lock(gTuneMutex);
        const auto it = gTuned.find(key);
        if (it != gTuned.end()) return it->second;
    }
    EventSet<4> ev;
    ev.record(0, s);
    launchRayShape<kSave>(kShapeLane, a, rays, count, out, hitPrim, nullptr, s);
    ev.record(1, s);
    ev.record(2, s);
    launchRayShape<kSave>(kShapeWave, a, rays, count, out, hitPrim, nullptr, s);
    ev.record(3, s);
    hipCheck(hipGetLastError(), "ray tuning");
    ev.sync(3);
    const int best = ev.ms(2, 3) < ev.ms(0, 1) ? kShapeWave : kShapeLane;
    std::lock_guard<std::mutex> lock(gTuneMutex);
    if (gTuned.size() >= kKeptMax) gTuned.clear();
    gTuned[key] = best;
    return best;
}

template <bool kSave>
static void launchRaysT(const TraverseArgs& a, const Ray* rays, int count, uint64_t* out, int* hitPrim,
                        hipStream_t s) {
    const int grid = blocksFor(count, kBlock);
    if (grid == 0) return;
    const Tri* tris = static_cast<const Tri*>(a.items);
    const int shape = rayShape<kSave>(a, rays, count, out, hitPrim, s);
    if (a.wide || shape != kShapeLane) {
        launchRayShape<kSave>(shape, a, rays, count, out, hitPrim, a.stats, s);
    } else {
        if (a.stats)
            rayBinaryKernel<true, kSave><<<grid, kBlock, 0, s>>>(a.nodes, tris, rays, a.order, count, out, a.stats,
                                                                a.primIds, hitPrim);
        else
            rayBinaryKernel<false, kSave><<<grid, kBlock, 0, s>>>(a.nodes, tris, rays, a.order, count, out,
                                                                 nullptr, a.primIds, hitPrim);
    }
    hipCheck(hipGetLastError(), "raycast");
}

void launchRays(const TraverseArgs& a, const Ray* rays, int count, uint64_t* out, hipStream_t s) {
    launchRaysT<false>(a, rays, count, out, nullptr, s);
}

void launchRaysSave(const TraverseArgs& a, const Ray* rays, int count, uint64_t* out, int* hitPrim,
                    hipStream_t s) {
    launchRaysT<true>(a, rays, count, out, hitPrim, s);
}

void setTraversalMode(int mode) { gTraversalMode = mode; }

namespace {
constexpr int kOverflowDevices = 64;
std::mutex gOverflowMutex;
int* gOverflowHost[kOverflowDevices] = {};

int* overflowHost() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kOverflowDevices) return nullptr;
    std::lock_guard<std::mutex> lock(gOverflowMutex);
    return gOverflowHost[dev];
}
}  // namespace

void armOverflowWord() {
    int dev = 0;
    hipCheck(hipGetDevice(&dev), "get device");
    if (dev < 0 || dev >= kOverflowDevices) return;
    std::lock_guard<std::mutex> lock(gOverflowMutex);
    if (gOverflowHost[dev]) return;
    int* h = nullptr;
    hipCheck(hipHostMalloc(reinterpret_cast<void**>(&h), 256, hipHostMallocDefault), "overflow word");
    *h = 0;
    int* d = nullptr;
    hipCheck(hipHostGetDevicePointer(reinterpret_cast<void**>(&d), h, 0), "overflow word address");
    hipCheck(hipMemcpyToSymbol(HIP_SYMBOL(gOverflowWord), &d, sizeof(d)), "overflow word symbol");
    gOverflowHost[dev] = h;
}

void checkOverflow() {
    int* h = overflowHost();
    if (!h || __atomic_load_n(h, __ATOMIC_ACQUIRE) == 0) return;
    __atomic_store_n(h, 0, __ATOMIC_RELEASE);
    throw DeviceError("traversal stack overflow: the tree is deeper than the traversal stack holds, "
                      "so some results are incomplete");
}


// Lanes per closest / kNN query (64, 32 or 16) by the number of queries.  A small set
// fills the device only with more lanes per query; a large one is served with the fewest
// instructions by 16.  Measured (kernel us at 64 / 32 / 16 lanes): the 2M-triangle terrain,
// SAH tree, closest 8k 43 / 52 / 78, 16k 64 / 62 / 88, 60k 165 / 140 / 145, kNN16 32k
// 160 / 143 / 159; around an icosphere, where walks are long and uneven, closest 16k
// 155 / 284 / 473, 60k 264 / 364 / 561 -- so triangles change late, and from kTuneFrom
// queries on the call times the three; 1M points kNN8 4k 33 / 32 / 41, 16k 69 / 52 / 53,
// 60k 196 / 125 / 88; 1M Gaussians closest 4k 64 / 47 / 58, 32k 253 / 152 / 126.  One lane
// and four lanes per query are behind at every count up to 1M (terrain closest 1M: 3253
// and 2900 against 1361; points kNN8 1M: 1135 and 1338 against 810).
template <typename L>
static int lanesPerQuery(int count, int k) {
    constexpr int kBelow64 = L::kKind == 0 ? 16384 : 3072;
    constexpr int kBelow32 = L::kKind == 0 ? kTuneFrom : (L::kKind == 1 ? 12288 : 28672);
    const int lanes = count < kBelow64 ? 64 : (count < kBelow32 ? 32 : 16);
    return k > 16 && lanes < 32 ? 32 : lanes;  // the list takes a lane per entry
}

// G lanes per query (64: one wave per query), k at most G; over the 4-wide nodes or, with
// a.wide false, the binary ones.
template <typename L, bool kOne, int G, typename Nodes>
static void launchGroupOn(Nodes nodes, int idCount, const TraverseArgs& a, const V3* pts, int count, int k,
                          int outStride, ClosestResult* out, unsigned long long* stats, hipStream_t s) {
    const auto* prims = static_cast<const typename L::Item*>(a.items);
    const uint32_t idMask = stackIdMask(idCount);
    const int grid = blocksFor(count, (kBlock / 64) * (64 / G));
    if (stats)
        nearestWaveKernel<L, kOne, G, true><<<grid, kBlock, 0, s>>>(nodes, prims, a.primIds, pts, a.order, count, k, outStride, out, stats, idMask);
    else
        nearestWaveKernel<L, kOne, G, false><<<grid, kBlock, 0, s>>>(nodes, prims, a.primIds, pts, a.order, count, k, outStride, out, nullptr, idMask);
}
template <typename L, bool kOne, int G>
static void launchGroup(const TraverseArgs& a, const V3* pts, int count, int k, int outStride, ClosestResult* out,
                        unsigned long long* stats, hipStream_t s) {
    if (a.wide)
        launchGroupOn<L, kOne, G>(WideNodes{a.wideNodes}, a.wideCount, a, pts, count, k, outStride, out, stats, s);
    else
        launchGroupOn<L, kOne, G>(BinaryNodes{a.nodes}, a.nodeCount, a, pts, count, k, outStride, out, stats, s);
}

template <typename L, int K>
static void launchShape(int shape, const TraverseArgs& a, const V3* pts, int count, int k, int outStride,
                        ClosestResult* out, unsigned long long* stats, hipStream_t s) {
    const auto* prims = static_cast<const typename L::Item*>(a.items);
    const int idBits = stackIdBitsDev(a.wideCount);
    if (shape == kShapeWave) {
        launchGroup<L, K == 1, 64>(a, pts, count, k, outStride, out, stats, s);
    } else if (shape == kShapeGroup16 || shape == kShapeGroup32) {
        if (shape == kShapeGroup16 && K <= 16)
            launchGroup<L, K == 1, 16>(a, pts, count, k, outStride, out, stats, s);
        else  // (more than 16 entries need 32 lanes)
            launchGroup<L, K == 1, 32>(a, pts, count, k, outStride, out, stats, s);
    } else if (shape == kShapeQuad) {
        const int grid = blocksFor(4LL * count, kBlock);
        if (stats)
            nearestQuadKernel<L, K, true><<<grid, kBlock, 0, s>>>(a.wideNodes, prims, a.primIds, pts, a.order, count, k, outStride, out, stats, idBits);
        else
            nearestQuadKernel<L, K, false><<<grid, kBlock, 0, s>>>(a.wideNodes, prims, a.primIds, pts, a.order, count, k, outStride, out, nullptr, idBits);
    } else {
        const int grid = blocksFor(count, kBlock);
        if (stats)
            nearestWideKernel<L, K, true><<<grid, kBlock, 0, s>>>(a.wideNodes, prims, a.primIds, pts, a.order, count, k, outStride, out, stats, idBits);
        else
            nearestWideKernel<L, K, false><<<grid, kBlock, 0, s>>>(a.wideNodes, prims, a.primIds, pts, a.order, count, k, outStride, out, nullptr, idBits);
    }
}

// Binary nodes: the group walk tests a node's grandchildren as if it were 4-wide.  One lane
// per query is behind at every count measured for triangles and Gaussians (8,192-triangle
// terrain closest 257 queries 675 us against 22, 100k 937 against 221, 400k 1150 against
// 656; 262k Gaussians kNN8 100k 1527 against 480) and ahead for points, whose leaf test is
// the cheapest, from about 131,072 queries (1M points closest 100k 215 us against 171, 400k
// 344 against 591).  Mode 1 forces one lane here too.
template <typename L>
static int binaryLaneFrom() {
    return L::kKind == 1 ? 131072 : INT_MAX;
}

// The shape for a set of `count` queries by the measured crossovers (above).
template <typename L, int K>
static int defaultShape(int count) {
    const int lanes = lanesPerQuery<L>(count, K);
    return lanes == 64 ? kShapeWave : (lanes == 32 ? kShapeGroup32 : kShapeGroup16);
}

// The shape for this tree and size class (see kTuneFrom); a call that times has its results
// written already (done), every shape writing the same.  From kTuneSplitFrom queries on
// each shape walks a part of its own, so that such a call costs about what a later one does.
// A part is every fourth run of 256 visits: contiguous parts of ordered queries are regions
// of the scene, and the emptiest one's shape would win.  The first part is walked untimed,
// since it finds the tree outside the caches.  With fewer queries a part would not fill the
// device and say little: each shape walks all, after the first part.  (The parts are an
// order made for this call: as a mapping inside the walks they cost every other call 1 %.)
constexpr int kTuneSplitFrom = 3 * 65536;
constexpr int kPartRun = 256;
struct Parts {
    int n;
    int first[5];  // where each part begins in the order, and the end
};
static Parts partsOf(int count, int n) {
    Parts p{n, {0}};
    for (int i = 0; i < n; ++i) {  // whole rounds of n runs, then what is left
        const int round = n * kPartRun, rest = count % round - i * kPartRun;
        p.first[i + 1] = p.first[i] + count / round * kPartRun + std::min(std::max(rest, 0), kPartRun);
    }
    return p;
}
// The visits part by part.
static __global__ void partOrderKernel(const uint32_t* __restrict__ order, int count, Parts parts,
                                       uint32_t* __restrict__ out) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= count) return;
    const int run = i / kPartRun, part = run % parts.n;
    int first = 0;
#pragma unroll
    for (int p = 1; p < 4; ++p) first = part == p ? parts.first[p] : first;
    out[first + run / parts.n * kPartRun + i % kPartRun] = order ? order[i] : static_cast<uint32_t>(i);
}

struct TunedShape {
    int shape;
    bool done;
};
template <typename L, int K>
static TunedShape tunedShape(const TraverseArgs& a, const V3* pts, int count, int k, int outStride,
                             ClosestResult* out, hipStream_t s) {
    const TuneKey key{a.serial, L::kKind, K, octaveOf(count)};
    {
        std::lock_guard<std::mutex> lock(gTuneMutex);
        const bool again = gTuned.count(key) != 0 && gTuned[key] == kCalledOnce;
        const int shape = keptShape(key, a.wideCount);
        if (shape != kCalledOnce && !again) {
            if (gTuned.size() >= kKeptMax) gTuned.clear();
            gTuned.emplace(key, kCalledOnce);
            return {shape, false};
        }
    }
    constexpr int kShapes = K <= 16 ? 3 : 2;
    const int shapes[3] = {kShapeGroup32, kShapeWave, kShapeGroup16};
    QuietFree quiet;
    DevBuf<uint32_t> visits;
    try {
        visits.alloc(static_cast<size_t>(count));
    } catch (const OomError&) {  // the call itself needs no memory
        return {defaultShape<L, K>(count), false};
    }
    const Parts parts = partsOf(count, kShapes + 1);
    partOrderKernel<<<blocksFor(count, kBlock), kBlock, 0, s>>>(a.order, count, parts, visits.p);
    const bool split = count >= kTuneSplitFrom;
    TraverseArgs part = a;
    part.order = visits.p;
    launchShape<L, K>(shapes[0], part, pts, parts.first[1], k, outStride, out, nullptr, s);
    EventSet<kShapes + 1> ev;
    ev.record(0, s);
    for (int i = 0; i < kShapes; ++i) {
        part.order = visits.p + parts.first[i + 1];
        if (split) launchShape<L, K>(shapes[i], part, pts, parts.first[i + 2] - parts.first[i + 1], k, outStride, out, nullptr, s);
        else launchShape<L, K>(shapes[i], a, pts, count, k, outStride, out, nullptr, s);
        ev.record(i + 1, s);
    }
    hipCheck(hipGetLastError(), "nearest tuning");
    ev.sync(kShapes);
    quiet.begin();
    int best = shapes[0];
    float bestMs = 0.0f;
    for (int i = 0; i < kShapes; ++i) {
        const float ms = ev.ms(i, i + 1);
        if (i == 0 || ms < bestMs) {
            best = shapes[i];
            bestMs = ms;
        }
    }
    keepShape(key, a.wideCount, best);
    return {best, true};
}

// The shape an earlier tuning chose for this tree or a like call, else the measured
// crossovers' (no timing trials).
template <typename L, int K>
static int cachedShape(const TraverseArgs& a, int count) {
    std::lock_guard<std::mutex> lock(gTuneMutex);
    const int shape = keptShape({a.serial, L::kKind, K, octaveOf(count)}, a.wideCount);
    return shape != kCalledOnce ? shape : defaultShape<L, K>(count);
}

template <typename L, int K>
static void launchNearestTK(const TraverseArgs& a, const V3* pts, int count, int k, int outStride,
                            ClosestResult* out, hipStream_t s) {
    const auto* prims = static_cast<const typename L::Item*>(a.items);
    if (!a.wide && gTraversalMode != 1 && count < binaryLaneFrom<L>()) {
        launchShape<L, K>(defaultShape<L, K>(count), a, pts, count, k, outStride, out, a.stats, s);
        return;
    }
    if (!a.wide) {
        const int grid = blocksFor(count, kBlock);
        if (a.stats)
            nearestBinaryKernel<L, K, true><<<grid, kBlock, 0, s>>>(a.nodes, prims, a.primIds, pts, a.order, count, k, outStride, out, a.stats, stackIdBitsDev(a.nodeCount));
        else
            nearestBinaryKernel<L, K, false><<<grid, kBlock, 0, s>>>(a.nodes, prims, a.primIds, pts, a.order, count, k, outStride, out, nullptr, stackIdBitsDev(a.nodeCount));
        return;
    }
    int shape;
    bool tune = false;
    switch (gTraversalMode) {
        case 1: shape = kShapeLane; break;
        case 2: shape = kShapeQuad; break;
        case 3: shape = kShapeWave; break;
        case 5: shape = kShapeGroup16; break;
        case 6: shape = kShapeGroup32; break;
        case 4:
            tune = a.tune;
            shape = cachedShape<L, K>(a, count);
            break;
        default:
            tune = a.tune && count >= kTuneFrom;
            shape = count < kTuneFrom ? defaultShape<L, K>(count) : cachedShape<L, K>(a, count);
    }
    if (tune) {
        const TunedShape t = tunedShape<L, K>(a, pts, count, k, outStride, out, s);
        if (t.done && !a.stats) return;
        shape = t.shape;
    }
    launchShape<L, K>(shape, a, pts, count, k, outStride, out, a.stats, s);
}

template <typename L>
static void launchNearestT(const TraverseArgs& a, const V3* pts, int count, int k, int outStride,
                           ClosestResult* out, hipStream_t s) {
    if (k == 1) {
        launchNearestTK<L, 1>(a, pts, count, k, outStride, out, s);
    } else if (k <= 4) {
        launchNearestTK<L, 4>(a, pts, count, k, outStride, out, s);
    } else if (k <= 8) {
        launchNearestTK<L, 8>(a, pts, count, k, outStride, out, s);
    } else if (k <= 16) {
        launchNearestTK<L, 16>(a, pts, count, k, outStride, out, s);
    } else {
        launchNearestTK<L, 32>(a, pts, count, k, outStride, out, s);
    }
}

// Ordering is four to six launches, 25-30 us up to 262,144 elements and 80 us at a million.
// With a group of lanes on each query neighbouring queries share little that input order
// does not find in the caches too.  Measured on queries and rays in random order (call in
// us, input order / ordered):
//   4-wide nodes: closest, 2M-triangle terrain 60k 163 / 184, 100k 230 / 246, 200k 391 /
//   378; 131k terrain 60k 202 / 209, 131k 364 / 350; 1M points 100k 92 / 116; icosphere 60k
//   405 / 400, 100k 449 / 429.  kNN16, 131k terrain 60k 415 / 405, 100k 562 / 513;
//   icosphere 60k 774 / 771, 80k 880 / 734; 2M terrain 100k 328 / 343.  Radius, 1M points 60k
//   659 / 678, 131k 1061 / 918; 2M terrain 131k 160 / 184.
//   Binary nodes: terrain closest 8k 146 / 153, 16k 251 / 234; points kNN16 16k 121 / 140,
//   32k 184 / 165.
//   Rays, 4-wide: city, cosine 131k 99 / 127, 380k 195 / 242, down 380k 163 / 205; one lane
//   per ray (larger sets) profits: 1M down 370 / 341, 131k terrain 629 / 386.  Binary:
//   terrain cosine 131k 227 / 216, 33k 87 / 102.
bool orderingPays(const TraverseArgs& a, WalkKind walk, int count) {
    if (gTraversalMode != 0) return true;  // forced shapes keep their order
    if (walk == kWalkRays) return count >= (a.wide ? kRayLaneFrom : 98304);
    if (!a.wide) return count >= (a.kind == 0 ? 12288 : 24576);
    return count >= (walk == kWalkClosest ? 131072 : 65536);
}

static void launchNearest(const TraverseArgs& a, const V3* pts, int count, int k, int outStride,
                          ClosestResult* out, hipStream_t s) {
    if (count <= 0) return;
    switch (a.kind) {
        case 0: launchNearestT<TriLeaf>(a, pts, count, k, outStride, out, s); break;
        case 1: launchNearestT<PointLeaf>(a, pts, count, k, outStride, out, s); break;
        default: launchNearestT<GaussLeaf>(a, pts, count, k, outStride, out, s); break;
    }
    hipCheck(hipGetLastError(), k == 1 ? "closest" : "knn");
}

void launchClosest(const TraverseArgs& a, const V3* pts, int count, ClosestResult* out,
                   hipStream_t s) {
    launchNearest(a, pts, count, 1, 1, out, s);
}

void launchKnn(const TraverseArgs& a, const V3* pts, int count, int k, int outStride,
               ClosestResult* out, hipStream_t s) {
    launchNearest(a, pts, count, k, outStride, out, s);
}

// Whether a radius call captures its hits in one walk (by groups of lanes, or on quads):
// unless one lane per query is forced.
static bool radiusCaptures() { return gTraversalMode != 1; }

// cap > 0: a fill on quads after a capture (only the queries the capture could not
// hold are walked); cap == 0: the per-lane count / fill kernels.
template <typename L, bool kFill>
static void launchRadiusT(const TraverseArgs& a, const V3* pts, int count, float r2, int* counts,
                          const int* offsets, uint64_t* keys, int* maxCount, int cap, hipStream_t s) {
    const int grid = blocksFor(count, kBlock);
    const auto* prims = static_cast<const typename L::Item*>(a.items);
    unsigned long long* st = kFill ? nullptr : a.stats;
    if (kFill && cap > 0) {
        const int qgrid = blocksFor(4LL * count, kBlock);
        radiusQuadKernel<L, kRadiusFill, false><<<qgrid, kBlock, 0, s>>>(a.wideNodes, prims, a.primIds, pts, a.order, count, r2, counts, offsets, keys, nullptr, maxCount, cap);
    } else if (a.wide) {
        if (st)
            radiusKernel<L, true, kFill, true><<<grid, kBlock, 0, s>>>(a.nodes, a.wideNodes, prims, a.primIds, pts, a.order, count, r2, counts, offsets, keys, st, maxCount);
        else
            radiusKernel<L, true, kFill, false><<<grid, kBlock, 0, s>>>(a.nodes, a.wideNodes, prims, a.primIds, pts, a.order, count, r2, counts, offsets, keys, nullptr, maxCount);
    } else {
        if (st)
            radiusKernel<L, false, kFill, true><<<grid, kBlock, 0, s>>>(a.nodes, a.wideNodes, prims, a.primIds, pts, a.order, count, r2, counts, offsets, keys, st, maxCount);
        else
            radiusKernel<L, false, kFill, false><<<grid, kBlock, 0, s>>>(a.nodes, a.wideNodes, prims, a.primIds, pts, a.order, count, r2, counts, offsets, keys, nullptr, maxCount);
    }
}

// Lanes per radius query (4: the quad kernel, when mode 2 forces it).  Measured (kernel us at
// 64 / 32 / 16 / 4 lanes): 1M points r = 1, 5k 29 / 44 / 76 / 333, 20k 56 / 66 / 100 / 398,
// 60k 586 / 466 / 440 / 686, 400k 2326 / 1389 / 966 / 950; the 2M-triangle terrain r = 2,
// 20k 31 / 28 / 29 / 74, 100k 131 / 98 / 75 / 86, 400k 453 / 324 / 222 / 214; 262k
// Gaussians 20k 117 / 108 / 121 / 290, 131k 707 / 471 / 504 / 788.
static int radiusLanes(int count) {
    if (gTraversalMode == 2) return 4;
    if (gTraversalMode == 3) return 64;
    if (gTraversalMode == 6) return 32;
    return count < 16384 ? 64 : (count < 40960 ? 32 : 16);
}

template <typename L, int G, typename Nodes>
static void launchCaptureGroup(Nodes nodes, const TraverseArgs& a, const V3* pts, int count, float r2, int* counts,
                               uint64_t* capture, int cap, int* maxCount, hipStream_t s) {
    const auto* prims = static_cast<const typename L::Item*>(a.items);
    const int grid = blocksFor(count, (kBlock / 64) * (64 / G));
    if (a.stats)
        radiusGroupKernel<L, true, G><<<grid, kBlock, 0, s>>>(nodes, prims, a.primIds, pts, a.order, count, r2, counts, capture, a.stats, maxCount, cap);
    else
        radiusGroupKernel<L, false, G><<<grid, kBlock, 0, s>>>(nodes, prims, a.primIds, pts, a.order, count, r2, counts, capture, nullptr, maxCount, cap);
}

template <typename L, int G>
static void launchCaptureOn(const TraverseArgs& a, const V3* pts, int count, float r2, int* counts,
                            uint64_t* capture, int cap, int* maxCount, hipStream_t s) {
    if (a.wide)
        launchCaptureGroup<L, G>(WideNodes{a.wideNodes}, a, pts, count, r2, counts, capture, cap, maxCount, s);
    else
        launchCaptureGroup<L, G>(BinaryNodes{a.nodes}, a, pts, count, r2, counts, capture, cap, maxCount, s);
}

template <typename L>
static void launchCaptureT(const TraverseArgs& a, const V3* pts, int count, float r2, int* counts,
                           uint64_t* capture, int cap, int* maxCount, hipStream_t s) {
    const int lanes = radiusLanes(count);
    if (lanes == 64) {
        launchCaptureOn<L, 64>(a, pts, count, r2, counts, capture, cap, maxCount, s);
        return;
    }
    if (lanes == 32) {
        launchCaptureOn<L, 32>(a, pts, count, r2, counts, capture, cap, maxCount, s);
        return;
    }
    if (lanes == 16 || !a.wide) {
        launchCaptureOn<L, 16>(a, pts, count, r2, counts, capture, cap, maxCount, s);
        return;
    }
    const int qgrid = blocksFor(4LL * count, kBlock);
    const auto* prims = static_cast<const typename L::Item*>(a.items);
    if (a.stats)
        radiusQuadKernel<L, kRadiusCaptureMode, true><<<qgrid, kBlock, 0, s>>>(a.wideNodes, prims, a.primIds, pts, a.order, count, r2, counts, nullptr, capture, a.stats, maxCount, cap);
    else
        radiusQuadKernel<L, kRadiusCaptureMode, false><<<qgrid, kBlock, 0, s>>>(a.wideNodes, prims, a.primIds, pts, a.order, count, r2, counts, nullptr, capture, nullptr, maxCount, cap);
}

// Hits captured per query by the single walk; a second walk serves only the queries
// with more.  Up to 2,048 per query while the buffer stays within 256 MB (20k queries:
// 1,638, which holds every segment of the 1M-point cloud at r = 1, at most 572), at
// least 64 while 512 MB hold them (the 2M-triangle terrain at r = 2 has at most 43);
// fewer than 8 turns the capture off.
int radiusCaptureCap(int count) {
    if (count <= 0) return 64;
    const long long roomy = (256LL << 20) / static_cast<long long>(sizeof(uint64_t)) / count;
    if (roomy >= 64) return roomy > 2048 ? 2048 : static_cast<int>(roomy);
    const long long tight = (512LL << 20) / static_cast<long long>(sizeof(uint64_t)) / count;
    if (tight >= 64) return 64;
    return tight < 8 ? 0 : static_cast<int>(tight);
}

bool launchRadiusCapture(const TraverseArgs& a, const V3* pts, int count, float r2, int* counts,
                         uint64_t* capture, int cap, int* maxCount, hipStream_t s) {
    if (count <= 0) return false;
    if (!radiusCaptures() || cap <= 0) {
        switch (a.kind) {
            case 0: launchRadiusT<TriLeaf, false>(a, pts, count, r2, counts, nullptr, nullptr, maxCount, 0, s); break;
            case 1: launchRadiusT<PointLeaf, false>(a, pts, count, r2, counts, nullptr, nullptr, maxCount, 0, s); break;
            default: launchRadiusT<GaussLeaf, false>(a, pts, count, r2, counts, nullptr, nullptr, maxCount, 0, s); break;
        }
        hipCheck(hipGetLastError(), "radius count");
        return false;
    }
    switch (a.kind) {
        case 0: launchCaptureT<TriLeaf>(a, pts, count, r2, counts, capture, cap, maxCount, s); break;
        case 1: launchCaptureT<PointLeaf>(a, pts, count, r2, counts, capture, cap, maxCount, s); break;
        default: launchCaptureT<GaussLeaf>(a, pts, count, r2, counts, capture, cap, maxCount, s); break;
    }
    hipCheck(hipGetLastError(), "radius capture");
    return true;
}

void launchRadiusFill(const TraverseArgs& a, const V3* pts, int count, float r2, const int* counts,
                      int cap, const int* offsets, uint64_t* keys, hipStream_t s) {
    if (count <= 0) return;
    int* c = const_cast<int*>(counts);  // read only by the fill pass
    switch (a.kind) {
        case 0: launchRadiusT<TriLeaf, true>(a, pts, count, r2, c, offsets, keys, nullptr, cap, s); break;
        case 1: launchRadiusT<PointLeaf, true>(a, pts, count, r2, c, offsets, keys, nullptr, cap, s); break;
        default: launchRadiusT<GaussLeaf, true>(a, pts, count, r2, c, offsets, keys, nullptr, cap, s); break;
    }
    hipCheck(hipGetLastError(), "radius fill");
}

namespace {
// Moves the captured hits into the result, each segment sorted by (dist2, index) -- the
// order of the 64-bit keys, dist2 being non-negative.  A workgroup serves four queries:
// segments of up to 64 hits in one wave's registers (a hit per lane), then the longer ones
// one after another by the whole workgroup through a bitonic network in LDS (one wave
// alone took 100 us over the longest of them); beyond kCompactSort they move as they are.
// Queries with more than `cap` hits are left to the fill walk; a segment that would end
// past `capacity` keys is skipped (the caller moves again into a buffer of the exact size).
// Sorting here takes the place of a pass over all segments and of three launches for the
// long ones: 20k segments of 16 hits on average, 2 % above 64 and up to 566 long, took
// 84 us in those launches and take 31 here.
constexpr int kCompactSort = 2048;
__global__ __launch_bounds__(kBlock) void radiusCompactKernel(const int* __restrict__ counts,
                                                              const int* __restrict__ offsets,
                                                              const uint64_t* __restrict__ capture, int count,
                                                              int cap, uint64_t* __restrict__ keys,
                                                              long long capacity) {
    constexpr int kWaves = kBlock / 64;
    __shared__ uint64_t buf[kCompactSort];
    __shared__ int longCount[kWaves];  // the wave's segment, when the workgroup is to sort it
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long first = static_cast<long long>(blockIdx.x) * kWaves;
    const long long q = first + wave;
    int c = q < count ? counts[q] : 0;
    const long long off = c > 0 ? offsets[q] : 0;
    if (c > cap || off + c > capacity) c = 0;
    if (lane == 0) longCount[wave] = c > 64 && c <= kCompactSort ? c : 0;
    const uint64_t* src = capture + q * cap;
    uint64_t* dst = keys + off;
    if (c <= 64) {
        float d = kInf;
        int id = 0x7fffffff;
        if (lane < c) {
            const uint64_t k = src[lane];
            d = bitsFloat(static_cast<uint32_t>(k >> 32));
            id = static_cast<int>(static_cast<uint32_t>(k));
        }
        int w = 2;
        while (w < c) w <<= 1;
        if (c > 1) waveSortPairs(d, id, lane, w);
        if (lane < c) dst[lane] = (static_cast<uint64_t>(floatBits(d)) << 32) | static_cast<uint32_t>(id);
    } else if (c > kCompactSort) {
        for (int j = lane; j < c; j += 64) dst[j] = src[j];
    }
    __syncthreads();
    for (int s = 0; s < kWaves; ++s) {
        const int m = longCount[s];  // the same in every thread
        if (m == 0) continue;
        const uint64_t* from = capture + (first + s) * cap;
        uint64_t* to = keys + offsets[first + s];
        int w = 128;
        while (w < m) w <<= 1;
        for (int j = threadIdx.x; j < w; j += kBlock) buf[j] = j < m ? from[j] : ~0ull;
        __syncthreads();
        bitonicLds(buf, w, threadIdx.x, kBlock);
        for (int j = threadIdx.x; j < m; j += kBlock) to[j] = buf[j];
        __syncthreads();
    }
}

// The radius call's two host-side figures in one step: the total hit count and the
// largest per-query count (the maximum of the kMaxCopies words), stored straight into
// the caller's pinned host words.
__global__ void radiusSummaryKernel(const int* __restrict__ total, const int* __restrict__ maxCopies,
                                    int* __restrict__ host) {
    const int lane = threadIdx.x;
    int m = lane < kMaxCopies ? maxCopies[lane] : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(m, off, 64);
        m = o > m ? o : m;
    }
    if (lane == 0) {
        __hip_atomic_store(&host[0], *total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(&host[1], m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
}  // namespace

void radiusCompact(const int* counts, const int* offsets, const uint64_t* capture, int count, int cap,
                   uint64_t* keys, long long capacity, hipStream_t s) {
    if (count <= 0 || cap <= 0) return;
    radiusCompactKernel<<<blocksFor(count, kBlock / 64), kBlock, 0, s>>>(counts, offsets, capture, count, cap,
                                                                        keys, capacity);
    hipCheck(hipGetLastError(), "radius compact");
}

bool radiusCompactSorts(int maxSeg, int cap) { return maxSeg <= cap && maxSeg <= kCompactSort; }

// Offsets, total and largest count of a small query set in one workgroup: thread t takes
// a run of up to kOffsetsRun counts (a multiple of four: 16-byte loads, all in flight at
// once, kept in registers for the second use), the workgroup scans the runs' sums.
namespace {
constexpr int kOffsetsBlock = 1024, kOffsetsRun = kRadiusOffsetsMax / kOffsetsBlock;
static_assert(kOffsetsRun % 4 == 0, "runs of int4");
__global__ __launch_bounds__(kOffsetsBlock) void radiusOffsetsKernel(const int* __restrict__ counts, int n, int run,
                                                                     int* __restrict__ offsets,
                                                                     int* __restrict__ host) {
    __shared__ int sums[kOffsetsBlock / 64], most[kOffsetsBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int begin = static_cast<int>(threadIdx.x) * run;
    int4 c[kOffsetsRun / 4];
    int sum = 0, big = 0;
#pragma unroll
    for (int k = 0; k < kOffsetsRun / 4; ++k) {
        const int i = begin + 4 * k;
        c[k] = {0, 0, 0, 0};
        if (4 * k < run) {
            if (i + 3 < n) {
                c[k] = *reinterpret_cast<const int4*>(counts + i);
            } else {
                if (i < n) c[k].x = counts[i];
                if (i + 1 < n) c[k].y = counts[i + 1];
                if (i + 2 < n) c[k].z = counts[i + 2];
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kOffsetsRun / 4; ++k) {
        sum += c[k].x + c[k].y + c[k].z + c[k].w;
        const int a = c[k].x > c[k].y ? c[k].x : c[k].y, b = c[k].z > c[k].w ? c[k].z : c[k].w;
        big = a > big ? a : big;
        big = b > big ? b : big;
    }
    int x = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
        const int o = __shfl_xor(big, off, 64);
        big = o > big ? o : big;
    }
    if (lane == 63) {
        sums[wave] = x;
        most[wave] = big;
    }
    __syncthreads();
    int at = x - sum, total = 0;
    for (int w = 0; w < kOffsetsBlock / 64; ++w) {
        at += w < wave ? sums[w] : 0;
        total += sums[w];
        big = most[w] > big ? most[w] : big;
    }
#pragma unroll
    for (int k = 0; k < kOffsetsRun / 4; ++k) {
        const int i = begin + 4 * k;
        const int4 o = {at, at + c[k].x, at + c[k].x + c[k].y, at + c[k].x + c[k].y + c[k].z};
        if (4 * k < run) {
            if (i + 3 < n) {
                *reinterpret_cast<int4*>(offsets + i) = o;
            } else {
                if (i < n) offsets[i] = o.x;
                if (i + 1 < n) offsets[i + 1] = o.y;
                if (i + 2 < n) offsets[i + 2] = o.z;
            }
        }
        at = o.w + c[k].w;
    }
    if (threadIdx.x == 0) {
        offsets[n] = total;
        __hip_atomic_store(&host[0], total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(&host[1], big, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
}  // namespace

bool radiusOffsets(const int* counts, int n, int* offsets, int* hostDev, hipStream_t s) {
    if (n > kRadiusOffsetsMax) return false;
    const int run = (blocksFor(n, kOffsetsBlock) + 3) & ~3;
    radiusOffsetsKernel<<<1, kOffsetsBlock, 0, s>>>(counts, n, run, offsets, hostDev);
    hipCheck(hipGetLastError(), "radius offsets");
    return true;
}

void radiusSummary(const int* total, const int* maxCopies, int* hostDev, hipStream_t s) {
    static_assert(kMaxCopies <= 64, "one lane per copy");
    radiusSummaryKernel<<<1, 64, 0, s>>>(total, maxCopies, hostDev);
    hipCheck(hipGetLastError(), "radius summary");
}

void segmentSort(const int* offsets, uint64_t* keys, int count, int maxSeg, int* scratchInts,
                 hipStream_t s) {
    if (count <= 0 || maxSeg <= 1) return;
    const int wavesPerBlock = kBlock / 64;
    segSortWaveKernel<<<blocksFor(count, wavesPerBlock), kBlock, 0, s>>>(offsets, keys, count);
    hipCheck(hipGetLastError(), "segment sort (wave)");
    if (maxSeg <= kWaveCap) return;
    // scratchInts: [info 4][blockList count][hugeList count]
    int* info = scratchInts;
    int* blockList = scratchInts + 4;
    int* hugeList = blockList + count;
    zeroU64Kernel<<<1, kBlock, 0, s>>>(reinterpret_cast<unsigned long long*>(info), 2);
    segClassifyKernel<<<blocksFor(count, kBlock), kBlock, 0, s>>>(offsets, count, blockList,
                                                                  hugeList, info);
    // the block-sized segments: a fixed grid walks the device-side list (no host round trip)
    const int grid = count < 1024 ? count : 1024;
    segSortBlockKernel<<<grid, kBlock, kBlockCap * sizeof(uint64_t), s>>>(offsets, blockList, info, keys);
    hipCheck(hipGetLastError(), "segment sort (block)");
    if (maxSeg <= kBlockCap) return;
    int h[2] = {0, 0};
    hipCheck(hipMemcpyAsync(h, info, sizeof(h), hipMemcpyDeviceToHost, s), "seg info");
    hipCheck(hipStreamSynchronize(s), "seg info sync");
    if (h[1] > 0) {
        // Segments above the workgroup network's capacity: each is sorted by the
        // device radix sort as two stable 32-bit passes (index half, then distance
        // half), which orders the 64-bit keys exactly.
        std::vector<int> huge(static_cast<size_t>(h[1]));
        hipCheck(hipMemcpyAsync(huge.data(), hugeList, sizeof(int) * huge.size(), hipMemcpyDeviceToHost, s),
                 "huge list");
        std::vector<int> offs(static_cast<size_t>(count) + 1);
        hipCheck(hipMemcpyAsync(offs.data(), offsets, sizeof(int) * offs.size(), hipMemcpyDeviceToHost, s),
                 "huge offsets");
        hipCheck(hipStreamSynchronize(s), "huge sync");
        int maxM = 0;
        for (int sg : huge) maxM = std::max(maxM, offs[static_cast<size_t>(sg) + 1] - offs[static_cast<size_t>(sg)]);
        SortWorkspace ws;
        ws.reserve(static_cast<size_t>(maxM));
        DevBuf<uint32_t> lo(maxM), hi(maxM), tmp(maxM), ord1(maxM), ord2(maxM);
        for (int sg : huge) {
            const int off = offs[static_cast<size_t>(sg)];
            const int m = offs[static_cast<size_t>(sg) + 1] - off;
            splitKeysKernel<<<blocksFor(m, kBlock), kBlock, 0, s>>>(keys + off, m, lo.p, hi.p);
            sortClear(ws, static_cast<size_t>(m), 4, s);
            sortHistogram(ws, lo.p, static_cast<size_t>(m), 4, s);
            sortPairs(ws, lo.p, nullptr, tmp.p, ord1.p, static_cast<size_t>(m), 4, s);
            gatherU32Kernel<<<blocksFor(m, kBlock), kBlock, 0, s>>>(hi.p, ord1.p, m, tmp.p);
            sortClear(ws, static_cast<size_t>(m), 4, s);
            sortHistogram(ws, tmp.p, static_cast<size_t>(m), 4, s);
            sortPairs(ws, tmp.p, ord1.p, hi.p, ord2.p, static_cast<size_t>(m), 4, s);
            joinKeysKernel<<<blocksFor(m, kBlock), kBlock, 0, s>>>(hi.p, lo.p, ord2.p, m, keys + off);
            hipCheck(hipGetLastError(), "segment sort (huge)");
        }
        hipCheck(hipStreamSynchronize(s), "huge sort sync");
    }
}


// ---- batched traversal launchers ---------------------------------------------------------

namespace {

int residentCus() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0;
        hipCheck(hipGetDevice(&dev), "get device");
        hipDeviceProp_t prop{};
        hipCheck(hipGetDeviceProperties(&prop, dev), "device properties");
        cus = prop.multiProcessorCount;
    }
    return cus;
}

template <typename L, int K, int kBT, int kD, bool kWide, bool kReg>
void launchBatchTKV(const BatchQueryArgs& a, hipStream_t s) {
    auto kern = batchNearestKernel<L, K, kBT, kD, kWide, kReg>;
    static int perCu = 0;
    if (perCu == 0) {
        hipCheck(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, reinterpret_cast<const void*>(kern), kBT, 0),
                 "occupancy");
        if (perCu < 1) perCu = 1;
    }
    const int waves = (a.count + 63) / 64;
    int grid = perCu * residentCus();
    const int need = (waves * 64 + kBT - 1) / kBT;
    if (grid > need) grid = need;
    if (grid < 1) grid = 1;
    kern<<<grid, kBT, 0, s>>>(a.nodes, a.wide, a.wideRoot, static_cast<const typename L::Item*>(a.items), a.primIds,
                              a.primOff, a.points, a.qScene, a.order, a.count, a.k, a.outStride, a.out, a.counter);
}

template <typename L, int G, int kBT>
void launchBatchGroup(const BatchQueryArgs& a, hipStream_t s) {
    const int grid = blocksFor(a.count, (kBT / 64) * (64 / G));
    const auto kern = a.k <= 1 ? batchGroupKernel<L, true, G, kBT> : batchGroupKernel<L, false, G, kBT>;
    kern<<<grid, kBT, 0, s>>>(a.wide, a.wideRoot, static_cast<const typename L::Item*>(a.items), a.primIds, a.primOff,
                              a.points, a.qScene, a.order, a.count, a.k, a.outStride, a.out);
}

// The 4-wide LDS-stack variants: as many lanes per query as a plain call of that many
// queries takes.  One lane per query on a work queue, which these replaced, left the
// device waiting for the longest walks: 51k closest / kNN8 queries over 64 scenes 646 /
// 1012 us against 109 / 190, 1.73M over 2,048 scenes 1986 / 3329 against 1389 / 2563.
template <typename L, int kBT>
void launchBatchGroups(const BatchQueryArgs& a, hipStream_t s) {
    switch (lanesPerQuery<L>(a.count, a.k)) {
        case 64: launchBatchGroup<L, 64, kBT>(a, s); break;
        case 32: launchBatchGroup<L, 32, kBT>(a, s); break;
        default: launchBatchGroup<L, 16, kBT>(a, s); break;
    }
}

template <typename L, int K>
void launchBatchTK(const BatchQueryArgs& a, int variant, hipStream_t s) {
    switch (variant) {
        case kBatchLds256: launchBatchTKV<L, K, 256, kLdsDepth, false, false>(a, s); break;
        case kBatchLds64: launchBatchTKV<L, K, 64, kLdsDepth, false, false>(a, s); break;
        case kBatchScratch64: launchBatchTKV<L, K, 64, 0, false, false>(a, s); break;
        case kBatchReg64: launchBatchTKV<L, K, 64, 0, false, true>(a, s); break;
        case kBatchWideLds256: launchBatchGroups<L, 256>(a, s); break;
        case kBatchWideLds64: launchBatchGroups<L, 64>(a, s); break;
        case kBatchWideScratch64: launchBatchTKV<L, K, 64, 0, true, false>(a, s); break;
        default: launchBatchTKV<L, K, 64, 0, true, true>(a, s); break;
    }
}

template <typename L>
void launchBatchT(const BatchQueryArgs& a, int variant, hipStream_t s) {
    if (a.k <= 1) {
        launchBatchTK<L, 1>(a, variant, s);
    } else if (a.k <= 8) {
        launchBatchTK<L, 8>(a, variant, s);
    } else {
        launchBatchTK<L, 32>(a, variant, s);
    }
}

}  // namespace

void launchBatchNearest(const BatchQueryArgs& a, int variant, hipStream_t s) {
    if (a.count <= 0) return;
    if (a.k > 32) throw ArgError("k must be in [1, 32]");
    switch (a.kind) {
        case 0: launchBatchT<TriLeaf>(a, variant, s); break;
        case 1: launchBatchT<PointLeaf>(a, variant, s); break;
        default: launchBatchT<GaussLeaf>(a, variant, s); break;
    }
    hipCheck(hipGetLastError(), "batch traversal");
}

void launchBatchReset(int* counter, hipStream_t s) {
    batchResetKernel<<<1, 64, 0, s>>>(counter);
    hipCheck(hipGetLastError(), "batch reset");
}

}  // namespace qr
