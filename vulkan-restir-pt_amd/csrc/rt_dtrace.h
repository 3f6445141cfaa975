// Software ray traversal (replaces the driver traversal behind
// rayQueryProceedEXT, src/shader/ray_query.glsl:6-70; CDNA4 has no ray
// tracing units).
//
// The traversed tree is the 4-wide collapse of the binary LBVH: one 128-B node
// (8 x float4: lo.x/lo.y/lo.z/hi.x/hi.y/hi.z of the four children as float4s,
// the four child references, padding) per visit. The hit children are ordered
// by entry distance (slot order on ties): the node's leaves are tested first, the
// nearest internal child is visited next and the others wait on the stack.
//
// What bounds it is the number of instructions a wave issues (the kernels built
// on it run at 65-80 % of the SIMDs' VALU issue slots with 13-40 of 64 lanes
// active), then the latency of the dependent node fetches. Hence:
//  - the near and far plane of each axis are loaded from the address that the
//    direction's sign gives, instead of a min and a max per slab;
//  - all four children go through one sorting network on integer keys (leaves
//    above the internal children) and are written to the stack without
//    branches: missed children sort last and land above the top;
//  - a lane that holds a leaf waits until a third of the wave's busy lanes do
//    (RT_LEAF_SHARE), so a triangle test is issued for many lanes at once. Each
//    lane's own order of node visits and triangle tests does not change.
// Against the version with a branch per slot, which tested a node's leaves before
// going on: 1920x1080 terrain frame (1.1M triangles) 5.12 -> 4.08 ms, 1M random
// closest-hit rays 387 -> 317 us, 64x64 frame 968 -> 691 us. Waiting for half of
// the lanes or for a fifth: 4.16 and 4.10 ms.
//
// Per lane: a short stack in LDS (strided by the block size so a wave's pushes
// and pops hit distinct banks) that spills to a private array for deep trees.
// Closest-hit traversal keeps each entry's distance beside it (spilled entries: its
// top 16 bits, i.e. rounded toward zero; a negative one as -inf) and drops a popped
// node that lies beyond the closest hit found since it was pushed. That changes no
// result: a node's box contains its children's boxes, and the slab distances are
// monotone in the bounds under IEEE rounding, so every child of such a node would
// fail its own box test against the same closest hit. The counting builds count the
// visits of the order that the oracle specifies, which keeps 16 bits of every
// distance and never drops a node's nearest internal child; the plain builds visit
// at most those nodes.
// Leaves hold one triangle, tested with the watertight algorithm of Woop,
// Benthin and Wald (JCGT 2013) including its double-precision fallback. Box
// tests use (bound - o) * (1 / d) with IEEE minNum/maxNum so that 0 * inf slabs
// are dropped. Closest hit accepts tmin <= t < tBest.
#pragma once
#include "rt_dscene.h"

#ifndef RT_LDS_STACK
#define RT_LDS_STACK 11
#endif
#define RT_SPILL_STACK 244
#define RT_MAX_STACK (RT_LDS_STACK + RT_SPILL_STACK)
// Leaf tests are issued once RT_LEAF_SHARE x the lanes holding a leaf reach the lanes at a node.
#ifndef RT_LEAF_SHARE
#define RT_LEAF_SHARE 2
#endif
#define RT_LEAF 0x80000000u
#define RT_EMPTY 0xffffffffu

namespace rtd {

// Work counters of the counting kernel builds (nodes, triangles, rays).
struct TraceCounters { unsigned long long nodes, tris, rays; };

// Pixel queue of a persistent pass. The work items (pixels in tile order) are
// split into kQueueParts contiguous bands of tiles, each with its own counter
// of claimed items in its own 128-B line, so that the waves' claims spread over
// kQueueParts atomics instead of one; `done` counts finished workgroups. All are
// zero between launches (the last workgroup of a launch clears them).
constexpr uint32_t kQueueParts = 8;
struct WorkQueue {
    struct Part { uint32_t next, pad[31]; } part[kQueueParts];
    uint32_t done, pad[31];
};

struct RayT {
    f3 o, d, invd;
    float tmin, tmax;
    int kx, ky, kz;
    float Sx, Sy, Sz;
    uint32_t nx, ny, nz;  // byte offsets of the near planes in a node: lo, or hi where the direction is negative
    bool flat;            // a reciprocal is infinite: the ray's slabs can hold 0 * inf
};

RT_DEV float comp(f3 v, int k) { return k == 0 ? v.x : (k == 1 ? v.y : v.z); }

RT_DEV RayT makeRay(f3 o, f3 d, float tmin, float tmax) {
    RayT r;
    r.o = o; r.d = d; r.tmin = tmin; r.tmax = tmax;
    r.invd = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    int kz = (ax > ay) ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    int kx = kz + 1; if (kx == 3) kx = 0;
    int ky = kx + 1; if (ky == 3) ky = 0;
    float dz = comp(d, kz);
    if (dz < 0.0f) { int t = kx; kx = ky; ky = t; }
    r.kx = kx; r.ky = ky; r.kz = kz;
    r.Sx = comp(d, kx) / dz; r.Sy = comp(d, ky) / dz; r.Sz = 1.0f / dz;
    r.nx = r.invd.x < 0.0f ? 48u : 0u;
    r.ny = r.invd.y < 0.0f ? 64u : 16u;
    r.nz = r.invd.z < 0.0f ? 80u : 32u;
    r.flat = isinf(r.invd.x) || isinf(r.invd.y) || isinf(r.invd.z);
    return r;
}

// Slab test of one child from its near and far planes; an empty slot's planes (lo = inf, hi = -inf)
// never pass it.
RT_DEV bool slabHit(const RayT& r, float nx, float ny, float nz, float fx, float fy, float fz, float tBest,
                    float& tEnter) {
    float a = (nx - r.o.x) * r.invd.x, A = (fx - r.o.x) * r.invd.x;
    float b = (ny - r.o.y) * r.invd.y, B = (fy - r.o.y) * r.invd.y;
    float c = (nz - r.o.z) * r.invd.z, C = (fz - r.o.z) * r.invd.z;
    tEnter = fmaxf(fmaxf(fmaxf(a, b), c), r.tmin);
    return tEnter <= fminf(fminf(fminf(A, B), C), tBest);
}
// The same for a ray with an infinite reciprocal: 0 * inf is dropped by minNum/maxNum.
RT_DEV bool slabHitFlat(const RayT& r, float nx, float ny, float nz, float fx, float fy, float fz, float tBest,
                        float& tEnter) {
    float a = (nx - r.o.x) * r.invd.x, A = (fx - r.o.x) * r.invd.x;
    float b = (ny - r.o.y) * r.invd.y, B = (fy - r.o.y) * r.invd.y;
    float c = (nz - r.o.z) * r.invd.z, C = (fz - r.o.z) * r.invd.z;
    tEnter = fmaxf(fmaxf(fmaxf(fminf(a, A), fminf(b, B)), fminf(c, C)), r.tmin);
    return tEnter <= fminf(fminf(fminf(fmaxf(a, A), fmaxf(b, B)), fmaxf(c, C)), tBest);
}

RT_DEV bool triHit(const RayT& r, f3 v0, f3 v1, f3 v2, float tBest, float& tOut, float& b1, float& b2) {
    f3 A = v0 - r.o, B = v1 - r.o, C = v2 - r.o;
    float Akz = comp(A, r.kz), Bkz = comp(B, r.kz), Ckz = comp(C, r.kz);
    float Ax = comp(A, r.kx) - r.Sx * Akz, Ay = comp(A, r.ky) - r.Sy * Akz;
    float Bx = comp(B, r.kx) - r.Sx * Bkz, By = comp(B, r.ky) - r.Sy * Bkz;
    float Cx = comp(C, r.kx) - r.Sx * Ckz, Cy = comp(C, r.ky) - r.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {
        U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    // one sign throughout, else the ray passes outside; no branches, so a wave's lanes leave together
    const bool inside = fminf(fminf(U, V), W) >= 0.0f || fmaxf(fmaxf(U, V), W) <= 0.0f;
    float det = U + V + W;
    float Az = r.Sz * Akz, Bz = r.Sz * Bkz, Cz = r.Sz * Ckz;
    float T = U * Az + V * Bz + W * Cz;
    const bool neg = det < 0.0f;
    T = neg ? -T : T; V = neg ? -V : V; W = neg ? -W : W;
    float rcp = 1.0f / fabsf(det);
    float t = T * rcp;
    tOut = t; b1 = V * rcp; b2 = W * rcp;
    return inside & (det != 0.0f) & (t >= r.tmin) & (t < tBest);
}

// LDS stack slice of this lane: words lane, lane + stride, lane + 2 stride, ...
// (a typed LDS pointer, so that an access is never merged with one to the spilled entries).
typedef __attribute__((address_space(3))) uint32_t LdsWord;
struct TStack {
    LdsWord* lds;
    uint32_t stride;
};

// The LDS of a block's traversal stacks, kWords words per lane: RT_LDS_STACK entries of two words (a child
// reference and its key), or twice as many of one word where no keys are kept.
template <int kThreads, int kWords = 2 * RT_LDS_STACK>
struct StackLDS {
    uint32_t word[kWords * kThreads];
};

template <int kThreads, int kWords>
RT_DEV TStack laneStack(StackLDS<kThreads, kWords>& s) {
    return TStack{(LdsWord*)s.word + threadIdx.x, (uint32_t)kThreads};
}

// Push order of a node's children as signed integers, missed children last: the hit internal
// children from the farthest to the nearest, then the hit leaves from the farthest to the nearest.
// For a ray with tmin > 0, whose entry distances are positive: the bits of t order as t does, a leaf
// carries bit 31 in its reference, and no hit has the missed children's key. ~key is what the stack
// keeps: the entry distance as a float, negative for a leaf.
RT_DEV int pushKey(bool h, float t, uint32_t ref) {
    return h ? (int)~(__float_as_uint(t) | (ref & RT_LEAF)) : 0x7fffffff;
}
// The same order for any other ray. Its entry distances can be zero of either sign, which order alike, or
// negative, so a leaf cannot be told by the distance's sign and takes a bit above it.
RT_DEV unsigned long long pushKeySigned(bool h, float t, uint32_t ref) {
    const uint32_t b = __float_as_uint(t + 0.0f);
    const uint32_t rank = (b >> 31) ? ~b : b | 0x80000000u;
    return h ? (unsigned long long)(ref >> 31) << 32 | (uint32_t)~rank : ~0ull;
}
// What the stack keeps of such a key: the distance, or -inf, never beyond a hit, for a leaf or a negative one (which
// would be a greater one once cut to its top 16 bits).
RT_DEV uint32_t storedKey(unsigned long long k) {
    const uint32_t rank = ~(uint32_t)k;
    return (k >> 32) == 0u && rank >= 0x80000000u ? rank & 0x7fffffffu : 0xff800000u;
}
template <class Key>
RT_DEV void order2(Key& ka, uint32_t& ra, Key& kb, uint32_t& rb) {
    const bool sw = kb < ka;
    const Key k = min(ka, kb);
    kb = max(ka, kb);
    ka = k;
    const uint32_t t = sw ? rb : ra;
    rb = sw ? ra : rb;
    ra = t;
}
// Slots 3, 2, 1, 0 through a stable network of adjacent comparators: on equal keys the lower slot ends
// nearer the top.
template <class Key>
RT_DEV void order4(Key& k3, uint32_t& c3, Key& k2, uint32_t& c2, Key& k1, uint32_t& c1, Key& k0, uint32_t& c0) {
    order2(k3, c3, k2, c2);
    order2(k2, c2, k1, c1); order2(k3, c3, k2, c2);
    order2(k1, c1, k0, c0); order2(k2, c2, k1, c1); order2(k3, c3, k2, c2);
}

// One lane's ray under way: idle when cur is RT_EMPTY, else at node or leaf cur with sp stack entries.
struct Walk {
    RayT r;
    float tBest;
    uint32_t cur;
    int sp;
};
// The part of a lane's stack beyond its LDS entries (it must outlive the calls of walk() that a ray takes).
struct StackSpill {
    uint32_t ref[RT_SPILL_STACK];
    uint16_t key[RT_SPILL_STACK];
};
struct WalkWork { unsigned long long nodes, tris; };

RT_DEV void startWalk(const DevScene& S, Walk& w, f3 o, f3 d, float tmin, float tmax) {
    w.r = makeRay(o, d, tmin, tmax);
    w.tBest = tmax;
    w.sp = 0;
    // A non-finite ray hits nothing; reject it here, because the slab test
    // (fminf/fmaxf drop NaN operands) would accept every box and the ray would
    // walk the whole tree.
    w.cur = isfinite(o.x) && isfinite(o.y) && isfinite(o.z) && isfinite(d.x) && isfinite(d.y) && isfinite(d.z) &&
                    S.numPrims != 0u ? 0u : RT_EMPTY;
}

// Walks the lanes' rays until fewer than minBusy of the wave's (converged) lanes are busy. kAny: a lane stops at
// its first hit. hit.inst is set on a hit and is the caller's to initialise. kCull: closest-hit queries drop
// popped nodes beyond the closest hit (the result is the same either way; the reuse passes' replays, which rarely
// pop such nodes, leave it off to save registers). kAnyTmin: the rays' tmin may be zero or negative; without it they
// must be positive.
template <bool kAny, bool kCount, bool kCull, int kStackWords = 2 * RT_LDS_STACK, bool kAnyTmin = false>
RT_DEV void walk(const DevScene& S, Walk& w, bool skipLights, TStack st, StackSpill& spill, int minBusy, Isec& hit,
                 WalkWork& work) {
    constexpr bool kKeep = kCull && !kAny;  // keys kept on the stack
    constexpr int kWords = kKeep ? 2 : 1;
    constexpr int kCap = kStackWords / kWords;
    static_assert(kCap + RT_SPILL_STACK >= RT_MAX_STACK, "the build bounds the stack depth by RT_MAX_STACK");
    const int entry = kWords * (int)st.stride;
    const RayT& r = w.r;
    float tBest = w.tBest;
    uint32_t cur = w.cur;
    int sp = w.sp;
    auto popOne = [&]() {
        sp--;
        uint32_t ref;
        float t = 0.0f;
        if (sp < kCap) {
            const LdsWord* e = st.lds + sp * entry;
            ref = e[0];
            if (kKeep) t = __uint_as_float(e[st.stride]);
        } else {
            ref = spill.ref[sp - kCap];
            if (kKeep) t = __uint_as_float((uint32_t)spill.key[sp - kCap] << 16);
        }
        if (kCount) t = __uint_as_float(__float_as_uint(t) & 0xffff0000u);
        cur = kKeep && t > tBest ? RT_EMPTY : ref;
    };
    // the next node or leaf; closest-hit rays drop nodes beyond the hit (a shadow ray's tBest is fixed)
    auto pop = [&]() {
        if (kKeep) {
            while (cur == RT_EMPTY && sp > 0) popOne();
        } else if (sp > 0) {
            popOne();
        }
    };
    unsigned long long nodeLanes = __ballot((int)cur >= 0), leafLanes = __ballot((int)cur < -1);
    while (__popcll(nodeLanes | leafLanes) >= minBusy) {
        if (RT_LEAF_SHARE * __popcll(leafLanes) >= __popcll(nodeLanes)) {
            if ((int)cur < -1) {
                const float4* tp = S.leafTris + 3 * (size_t)(cur & ~RT_LEAF);
                const float4 a = tp[0], b = tp[1], c = tp[2];
                const uint32_t inst = __float_as_uint(a.w);
                const bool skip = skipLights & (inst == 0u);
                if (kCount) work.tris += skip ? 0 : 1;
                float t, b1, b2;
                const bool h = triHit(r, mk3(a.x, a.y, a.z), mk3(b.x, b.y, b.z), mk3(c.x, c.y, c.z), tBest, t, b1, b2);
                cur = RT_EMPTY;
                if (h & !skip) {
                    hit.inst = inst;
                    if (kAny) {
                        sp = 0;
                    } else {
                        tBest = t;
                        hit.b1 = b1; hit.b2 = b2; hit.prim = __float_as_uint(b.w);
                    }
                }
                pop();
            }
        }
        if ((int)cur >= 0) {
            const char* np = reinterpret_cast<const char*>(S.nodes) + 128 * (size_t)cur;
            const float4 nx = *reinterpret_cast<const float4*>(np + r.nx), fx = *reinterpret_cast<const float4*>(np + (r.nx ^ 48u));
            const float4 ny = *reinterpret_cast<const float4*>(np + r.ny), fy = *reinterpret_cast<const float4*>(np + (r.ny ^ 80u));
            const float4 nz = *reinterpret_cast<const float4*>(np + r.nz), fz = *reinterpret_cast<const float4*>(np + (r.nz ^ 112u));
            const float4 cr = *reinterpret_cast<const float4*>(np + 96);
            if (kCount) work.nodes++;
            uint32_t c0 = __float_as_uint(cr.x), c1 = __float_as_uint(cr.y), c2 = __float_as_uint(cr.z),
                     c3 = __float_as_uint(cr.w);
            float t0, t1, t2, t3;
            bool h0 = slabHit(r, nx.x, ny.x, nz.x, fx.x, fy.x, fz.x, tBest, t0);
            bool h1 = slabHit(r, nx.y, ny.y, nz.y, fx.y, fy.y, fz.y, tBest, t1);
            bool h2 = slabHit(r, nx.z, ny.z, nz.z, fx.z, fy.z, fz.z, tBest, t2);
            bool h3 = slabHit(r, nx.w, ny.w, nz.w, fx.w, fy.w, fz.w, tBest, t3);
            // (counted visits are those of min and max, also for the box of the unused child of a one-leaf tree)
            if (kCount || r.flat) {
                h0 = slabHitFlat(r, nx.x, ny.x, nz.x, fx.x, fy.x, fz.x, tBest, t0) & (c0 != RT_EMPTY);
                h1 = slabHitFlat(r, nx.y, ny.y, nz.y, fx.y, fy.y, fz.y, tBest, t1) & (c1 != RT_EMPTY);
                h2 = slabHitFlat(r, nx.z, ny.z, nz.z, fx.z, fy.z, fz.z, tBest, t2) & (c2 != RT_EMPTY);
                h3 = slabHitFlat(r, nx.w, ny.w, nz.w, fx.w, fy.w, fz.w, tBest, t3) & (c3 != RT_EMPTY);
            }
            const int n = (int)h0 + (int)h1 + (int)h2 + (int)h3;
            uint32_t key[4];  // of c3, c2, c1, c0 once ordered
            if (!kAnyTmin || r.tmin > 0.0f) {
                int k0 = pushKey(h0, t0, c0), k1 = pushKey(h1, t1, c1), k2 = pushKey(h2, t2, c2), k3 = pushKey(h3, t3, c3);
                order4(k3, c3, k2, c2, k1, c1, k0, c0);
                key[0] = ~(uint32_t)k3; key[1] = ~(uint32_t)k2; key[2] = ~(uint32_t)k1; key[3] = ~(uint32_t)k0;
            } else {
                unsigned long long k0 = pushKeySigned(h0, t0, c0), k1 = pushKeySigned(h1, t1, c1),
                                   k2 = pushKeySigned(h2, t2, c2), k3 = pushKeySigned(h3, t3, c3);
                order4(k3, c3, k2, c2, k1, c1, k0, c0);
                key[0] = storedKey(k3); key[1] = storedKey(k2); key[2] = storedKey(k1); key[3] = storedKey(k0);
            }
            const uint32_t cs[4] = {c3, c2, c1, c0};
            if (kCount && kKeep) {
                // the counted order visits a node's nearest internal child without a distance check: the
                // last entry that is not a leaf
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (q < n && !(cs[q] >> 31) && (q + 1 == n || (cs[q + 1 < 4 ? q + 1 : 3] >> 31))) { key[q] = 0xff800000u; break; }
            }
            if (sp + 4 <= kCap) {  // the missed children land above the top
                LdsWord* e = st.lds + sp * entry;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    e[q * entry] = cs[q];
                    if (kKeep) e[q * entry + (int)st.stride] = key[q];
                }
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (q >= n) continue;
                    const int pos = sp + q;
                    if (pos < kCap) {
                        st.lds[pos * entry] = cs[q];
                        if (kKeep) st.lds[pos * entry + (int)st.stride] = key[q];
                    } else if (pos - kCap < RT_SPILL_STACK) {  // the build bounds the stack depth
                        spill.ref[pos - kCap] = cs[q];
                        if (kKeep) spill.key[pos - kCap] = (uint16_t)(key[q] >> 16);
                    }
                }
            }
            sp += n;
            cur = RT_EMPTY;
            pop();
        }
        nodeLanes = __ballot((int)cur >= 0);
        leafLanes = __ballot((int)cur < -1);
    }
    w.tBest = tBest;
    w.cur = cur;
    w.sp = sp;
}

RT_DEV void countWork(TraceCounters* ctr, const WalkWork& work, unsigned long long rays) {
    atomicAdd(&ctr->nodes, work.nodes); atomicAdd(&ctr->tris, work.tris); atomicAdd(&ctr->rays, rays);
}

// One ray per lane, to the end.
template <bool kAny, bool kCount, bool kCull = true, bool kAnyTmin = false>
RT_DEV bool traverse(const DevScene& S, f3 o, f3 d, float tmin, bool skipLights, TStack st, float& tBest, Isec& hit,
                     TraceCounters* ctr) {
    StackSpill spill;
    WalkWork work{0, 0};
    Walk w;
    startWalk(S, w, o, d, tmin, tBest);
    hit.inst = RT_EMPTY;
    walk<kAny, kCount, kCull, 2 * RT_LDS_STACK, kAnyTmin>(S, w, skipLights, st, spill, 1, hit, work);
    tBest = w.tBest;
    if (kCount && S.numPrims != 0u) countWork(ctr, work, 1ull);
    return hit.inst != RT_EMPTY;
}

}  // namespace rtd
