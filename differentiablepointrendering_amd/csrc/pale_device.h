// pale_device.h -- device functions of the gfx950 renderer: closest-hit
// traversal, surfel and triangle tests, sampling, Russian roulette, light
// sampling and the photon-grid irradiance gather.
//
// Traversal keeps the reference's visiting order exactly (near-far child
// push with ties to the left child, IntersectionKernels.h:21-32 and
// :585-675), so the closest hit -- including which surfel wins an exact tie
// in t -- is the reference's.  The stack lives in LDS: entry k of a lane is
// at stk[k * kStackStride] (bank-conflict free per row).  A
// stack entry is (node reference, entry distance); re-testing a popped box
// against the current best distance is done with the stored entry distance,
// which equals the reference's full slab re-test because the other two
// rejection conditions do not depend on the best distance.
#pragma once

#include "pale_common.h"

namespace pale {

struct DevScene {
    const SurfelGeo* geo;
    const SurfelShade* shade;
    const WideNode* nodes;
    const QuadNode* quads;  // of the cloud's nodes
    const TriGeo* tris;
    const DevInstance* inst;
    const TlasNode* tlas;
    const DevMaterial* mats;
    const DevLight* lights;
    const DevEmTri* emTris;
    uint32_t nInst;
    uint32_t nTlas;
    uint32_t nLights;
    uint32_t stackDepth;
    uint32_t cloudInst;  // instance of the point cloud (kInvalid if none)
};

struct DevGrid {
    const float4* posPow;  // sorted photons: position, power.x / (pi radius^2)
    const float4* dirPow;  // incoming direction, power.y / (pi radius^2)
    const float* powZ;     // power.z / (pi radius^2)
    const uint32_t* cellStart;  // exclusive prefix over cells, total+1 entries
    float ox, oy, oz;
    float cx, cy, cz;
    float inv;  // 1 / the cell size
    int rx, ry, rz;
    float radius;
    const uint32_t* attempted;  // deposits attempted (T), device memory
    uint32_t capacity;          // photon capacity
    uint32_t valid;      // a photon map exists
};

struct Hit {
    F3 pos;
    uint32_t inst, prim;  // inst kInvalid: miss
};

// Per-thread work counters of the counting mode (the per-query units of the
// algorithmic byte count: popped nodes, AABB slab tests, primitive tests,
// gather cells / non-empty cells / photons).
struct Work {
    uint32_t pops, aabb, prims, cells, cellsNE, photons, gathers;
};

__device__ __forceinline__ F3 ld3(const float4& v) { return mk3(v.x, v.y, v.z); }

// safeInvDir (KernelHelpers.h:140-147)
__device__ __forceinline__ F3 safeInvDir(F3 d) {
    return mk3(fabsf(d.x) < 1e-6f ? 1e30f : 1.0f / d.x, fabsf(d.y) < 1e-6f ? 1e30f : 1.0f / d.y,
               fabsf(d.z) < 1e-6f ? 1e30f : 1.0f / d.z);
}

// slabIntersectAABB (KernelHelpers.h:149-214); clampLo is 0 for TLAS nodes
// and 1e-6 for BVH nodes.
__device__ __forceinline__ bool slab(F3 o, F3 inv, float mnx, float mny, float mnz, float mxx, float mxy,
                                     float mxz, float limit, float clampLo, float& tEntry) {
    const float t0x = (mnx - o.x) * inv.x, t0y = (mny - o.y) * inv.y, t0z = (mnz - o.z) * inv.z;
    const float t1x = (mxx - o.x) * inv.x, t1y = (mxy - o.y) * inv.y, t1z = (mxz - o.z) * inv.z;
    const float tmin = fmaxf(fmaxf(fminf(t0x, t1x), fminf(t0y, t1y)), fminf(t0z, t1z));
    const float tmax = fminf(fminf(fmaxf(t0x, t1x), fmaxf(t0y, t1y)), fmaxf(t0z, t1z));
    if (tmin > tmax) return false;
    if (tmax < 0.0f) return false;
    if (tmin > limit) return false;
    tEntry = fmaxf(tmin, clampLo);
    return true;
}

// An LDS word pair.  The device pass types it as LDS memory so that stack
// accesses compile to LDS instructions; the host pass only parses the code.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) uint2 LdsUint2;
typedef __attribute__((address_space(3))) uint64_t LdsU64;
#else
typedef uint2 LdsUint2;
typedef uint64_t LdsU64;
#endif

// Threads of a traversal workgroup: the distance between a lane's stack
// entries in LDS, as a constant (a shift; a variable one is a multiplication
// at a quarter of the rate on every push and pop).
constexpr uint32_t kStackStride = 128;

struct LaneStack {
    LdsUint2* base;
    uint32_t cap;
    uint2* spill;  // the lane's spilled entries, entry k at spill[k - inLds]
    uint32_t inLds;
    // SmallStack::push (GPUDataTypes.h:398-402): a push beyond capacity is
    // dropped, so sp never exceeds cap and every pop reads a written slot.
    __device__ __forceinline__ void push(uint32_t& sp, uint32_t ref, float t) const {
        if (sp < cap) {
            const uint2 v = make_uint2(ref, __float_as_uint(t));
            if (sp < inLds)
                base[sp * kStackStride] = v;
            else
                spill[sp - inLds] = v;
            ++sp;
        }
    }
    // The cloud traversal holds at most three entries per two levels of the
    // tree, which the stack is made for.
    __device__ __forceinline__ void pushBounded(uint32_t& sp, uint32_t ref, float t) const {
        const uint2 v = make_uint2(ref, __float_as_uint(t));
        if (sp < inLds)
            base[sp * kStackStride] = v;
        else
            spill[sp - inLds] = v;
        ++sp;
    }
    // The LDS read is unconditional and a relaxed atomic load, so that it
    // stays an LDS instruction: two plain loads would be merged into one
    // generic (flat) load of a selected address, which goes through the
    // vector-memory path even when it reads LDS.  A spilled entry is then
    // read again from the spill area.
    __device__ __forceinline__ uint2 get(uint32_t k) const {
        const LdsU64* p = reinterpret_cast<const LdsU64*>(base + min(k, inLds - 1u) * kStackStride);
        const uint64_t bits = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        uint2 v = make_uint2((uint32_t)bits, (uint32_t)(bits >> 32));
        if (k >= inLds) v = spill[k - inLds];
        return v;
    }
};

struct LocalHit {
    F3 pos;
    uint32_t prim;
};

// intersectBLASPointCloudFirstHit (IntersectionKernels.h:585-675) with
// intersectSurfel (KernelHelpers.h:637-669), its work counted; alpha_geom is
// left to who needs it (a pure function of the hit, surfelAlpha).
__device__ bool traverseCloud(const DevScene& S, const DevInstance& I, F3 o, F3 d, const LaneStack& st,
                              uint32_t base, LocalHit& out, Work& w) {
    const F3 inv = safeInvDir(d);
    float best = __builtin_huge_valf();
    float te;
    w.aabb++;  // the reference slab-tests the root when it pops it
    if (!slab(o, inv, I.rmnx, I.rmny, I.rmnz, I.rmxx, I.rmxy, I.rmxz, best, 1e-6f, te)) {
        w.pops++;
        return false;
    }
    bool firstPop = true;
    uint32_t sp = base;
    st.push(sp, I.rootRef, te);
    uint32_t bestIdx = 0;
    F3 bestX = mk3(0, 0, 0);
    bool any = false;
    while (sp > base) {
        const uint2 e = st.get(--sp);
        w.pops++;
        if (!firstPop) w.aabb++;  // re-test of a popped box (root already counted)
        firstPop = false;
        if (__uint_as_float(e.y) > best) continue;
        const uint32_t ref = e.x;
        if (ref & kLeafBit) {
            const uint32_t first = leafFirst(ref), cnt = leafCount(ref);
            w.prims += cnt;
            for (uint32_t k = 0; k < cnt; ++k) {
                const uint32_t si = first + k;
                const float4* g = reinterpret_cast<const float4*>(S.geo + si);
                const float4 g0 = g[0], g1 = g[1];
                const F3 n = mk3(g1.x, g1.y, g1.z);
                const float nd = dot(n, d);
                if (fabsf(nd) < 1e-6f) continue;
                const F3 p = mk3(g0.x, g0.y, g0.z);
                const float t = dot(n, p - o) / nd;
                if (t <= 1e-5f || t >= best) continue;
                const float4 g2 = g[2], g3 = g[3];
                const F3 x = o + d * t;
                const F3 r = x - p;
                const float uu = dot(mk3(g2.x, g2.y, g2.z), r) / g0.w;
                const float vv = dot(mk3(g3.x, g3.y, g3.z), r) / g1.w;
                const float r2 = uu * uu + vv * vv;
                if (r2 >= 1.0f) continue;
                any = true;
                best = t;
                bestIdx = si;
                bestX = x;
            }
            continue;
        }
        const float4* nd4 = reinterpret_cast<const float4*>(S.nodes + ref);
        const float4 a = nd4[0], b = nd4[1], c = nd4[2];
        const uint2 refs = reinterpret_cast<const uint2*>(S.nodes + ref)[6];  // left, right (not the padding)
        w.aabb += 2;
        float tl = __builtin_huge_valf(), tr = __builtin_huge_valf();
        const bool hl = slab(o, inv, a.x, a.y, a.z, a.w, b.x, b.y, best, 1e-6f, tl);
        const bool hr = slab(o, inv, b.z, b.w, c.x, c.y, c.z, c.w, best, 1e-6f, tr);
        if (hl && hr) {
            if (tl <= tr) {
                st.push(sp, refs.y, tr);
                st.push(sp, refs.x, tl);
            } else {
                st.push(sp, refs.x, tl);
                st.push(sp, refs.y, tr);
            }
        } else if (hl) {
            st.push(sp, refs.x, tl);
        } else if (hr) {
            st.push(sp, refs.y, tr);
        }
    }
    if (!any) return false;
    out.prim = bestIdx;
    out.pos = bestX;
    return true;
}

// The closest hit's alpha, (1 - r^2)^(4 e^beta) in binary64, as a call: its
// 64-bit constants then stay inside the call instead of being hoisted into
// registers that live across the traversal loop (inlined, they pushed the
// camera walk into scratch spills; as a call the walk has none, and the
// walk, photon and adjoint traces run 2-10 % faster).
__device__ __attribute__((noinline)) float hitAlpha(float oneMinusR2, float e4b) { return pow_r(oneMinusR2, e4b); }

// Squared radius of the point x of a surfel's plane in its support, as the
// surfel test forms it.
__device__ __forceinline__ float surfelR2(const SurfelGeo& g, F3 x) {
    const F3 r = x - mk3(g.px, g.py, g.pz);
    const float uu = dot(mk3(g.tux, g.tuy, g.tuz), r) / g.su;
    const float vv = dot(mk3(g.tvx, g.tvy, g.tvz), r) / g.sv;
    return uu * uu + vv * vv;
}

// alpha of a surfel at its hit point (object space): a function of the two, so
// the traversal carries neither alpha nor radius.
__device__ __forceinline__ float surfelAlpha(const SurfelGeo& g, F3 x) {
    return hitAlpha(1.0f - surfelR2(g, x), g.e4b);
}

// Traversal of the cloud without the counters and without a stack round trip
// for the nearer child: the reference pushes the farther child, then the
// nearer, and pops the nearer at once with an unchanged best, so descending
// into the nearer child directly visits the same nodes in the same order.
// It is written as single steps on a lane's state, so that a wave can choose
// which lanes step (traceWave); a lane's own sequence of steps, and with it
// every result, does not depend on that choice.
constexpr uint32_t kRefDone = kInvalid;  // the traversal has ended (no leaf reference: first < 2^29 - 4)

struct CloudLane {
    F3 o, d, inv;                    // object-space ray
    float best;                      // closest hit so far
    uint32_t bestIdx;                // its surfel (kInvalid: none)
    uint32_t ref;                    // node or leaf to visit, kRefDone at the end
    uint32_t sp, base;               // stack height; the height below this traversal
};

// Starts a traversal above the stack entries the lane holds; false if the ray
// misses the root box.
__device__ __forceinline__ bool cloudBegin(const DevInstance& I, F3 o, F3 d, uint32_t sp, CloudLane& c) {
    c.o = o;
    c.d = d;
    c.inv = safeInvDir(d);
    c.best = __builtin_huge_valf();
    c.bestIdx = kInvalid;
    c.sp = c.base = sp;
    c.ref = I.rootRef;
    float te;
    return slab(o, c.inv, I.rmnx, I.rmny, I.rmnz, I.rmxx, I.rmxy, I.rmxz, c.best, 1e-6f, te);
}

// The next entry that does not start beyond the current best.
__device__ __forceinline__ void cloudPop(const LaneStack& st, CloudLane& c) {
    c.ref = kRefDone;
    while (c.sp > c.base) {
        const uint2 e = st.get(--c.sp);
        if (__uint_as_float(e.y) > c.best) continue;
        c.ref = e.x;
        break;
    }
}

// One step: the two levels below a node at once.
//
// The binary tree's step tests the children's boxes, goes on to the nearer (ties
// to the left) and later, if it is still in range, to the farther, each of which
// tests its own children then.  A grandchild's box lies in its parent's, and
// every operation of the slab test is monotone, also as rounded, so a
// grandchild that passes implies that its parent passes, with an entry not
// after its own; and a test passed earlier is only undone by a closer hit, which
// the stored entry shows at the pop.  Testing the four grandchildren now and
// keeping them in the order (nearer child's nearer, its farther, farther child's
// nearer, its farther) therefore visits the same leaves in the same order.  The
// children's entries, which that order needs, come from the grandchildren's
// planes (a child's box is their union; k_quad_nodes checks it).
//
// slab() with clampLo 1e-6; its three rejections are one comparison: max(tmin,
// 0) > min(tmax, limit) holds exactly when one of them does, also with NaN in
// tmin, tmax or limit (the limit is positive, fmin and fmax pass a NaN over).
__device__ __forceinline__ void cloudNode(const DevScene& S, const LaneStack& st, CloudLane& c) {
    const float4* q = reinterpret_cast<const float4*>(S.quads + c.ref);
    const float4 nx = q[0], xx = q[1], ny = q[2], xy = q[3], nz = q[4], xz = q[5];
    const uint4 refs = reinterpret_cast<const uint4*>(S.quads + c.ref)[6];
    const float mn[3][4] = {{nx.x, nx.y, nx.z, nx.w}, {ny.x, ny.y, ny.z, ny.w}, {nz.x, nz.y, nz.z, nz.w}};
    const float mx[3][4] = {{xx.x, xx.y, xx.z, xx.w}, {xy.x, xy.y, xy.z, xy.w}, {xz.x, xz.y, xz.z, xz.w}};
    const float o[3] = {c.o.x, c.o.y, c.o.z}, inv[3] = {c.inv.x, c.inv.y, c.inv.z};
    float lo[3][4], hi[3][4];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float t0 = (mn[a][k] - o[a]) * inv[a], t1 = (mx[a][k] - o[a]) * inv[a];
            lo[a][k] = fminf(t0, t1);
            hi[a][k] = fmaxf(t0, t1);
        }
    }
    float t[4];
    bool h[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float tmin = fmaxf(fmaxf(lo[0][k], lo[1][k]), lo[2][k]);
        const float tmax = fminf(fminf(hi[0][k], hi[1][k]), hi[2][k]);
        t[k] = fmaxf(tmin, 1e-6f);
        h[k] = !(fmaxf(tmin, 0.0f) > fminf(tmax, c.best));
    }
    h[1] = h[1] && refs.y != kInvalid;
    h[3] = h[3] && refs.w != kInvalid;
    const float tl = fmaxf(fmaxf(fmaxf(fminf(lo[0][0], lo[0][1]), fminf(lo[1][0], lo[1][1])), fminf(lo[2][0], lo[2][1])), 1e-6f);
    const float tr = fmaxf(fmaxf(fmaxf(fminf(lo[0][2], lo[0][3]), fminf(lo[1][2], lo[1][3])), fminf(lo[2][2], lo[2][3])), 1e-6f);
    // Order: within the pairs, then the pairs.
    const bool sl = !(t[0] <= t[1]), sr = !(t[2] <= t[3]), sp = !(tl <= tr);
    const uint32_t la = sl ? refs.y : refs.x, lb = sl ? refs.x : refs.y, ra = sr ? refs.w : refs.z, rb = sr ? refs.z : refs.w;
    const float lta = sl ? t[1] : t[0], ltb = sl ? t[0] : t[1], rta = sr ? t[3] : t[2], rtb = sr ? t[2] : t[3];
    const bool hla = sl ? h[1] : h[0], hlb = sl ? h[0] : h[1], hra = sr ? h[3] : h[2], hrb = sr ? h[2] : h[3];
    const uint32_t r0 = sp ? ra : la, r1 = sp ? rb : lb, r2 = sp ? la : ra, r3 = sp ? lb : rb;
    const float t1 = sp ? rtb : ltb, t2 = sp ? lta : rta, t3 = sp ? ltb : rtb;
    const bool h0 = sp ? hra : hla, h1 = sp ? hrb : hlb, h2 = sp ? hla : hra, h3 = sp ? hlb : hrb;
    const bool any1 = h0 || h1, any2 = any1 || h2;
    if (h3 && any2) st.pushBounded(c.sp, r3, t3);
    if (h2 && any1) st.pushBounded(c.sp, r2, t2);
    if (h1 && h0) st.pushBounded(c.sp, r1, t1);
    c.ref = h0 ? r0 : (h1 ? r1 : (h2 ? r2 : r3));
    if (!any2 && !h3) cloudPop(st, c);
}

// The lane's traversal from the start, by the binary tree's steps and the tests
// in leaf order: for a ray whose two-level walk accepted a NaN distance (a
// degenerate surfel's).  After one, the next surfel is accepted at any
// distance, so the best rises, and boxes tested two levels early against the
// smaller one are missing from the stack.  On the lane's own state and surfel by
// surfel: it runs hardly ever, and its registers would count for every wave (a
// second kind of step in the waves' loop cost 3 to 5 % of every case).
__device__ __forceinline__ void cloudAgain(const DevScene& S, uint32_t rootRef, const LaneStack& st, CloudLane& c) {
    c.best = __builtin_huge_valf();
    c.bestIdx = kInvalid;
    c.sp = c.base;
    c.ref = rootRef;
    while (c.ref != kRefDone) {
        if (c.ref & kLeafBit) {
            const uint32_t first = leafFirst(c.ref), cnt = leafCount(c.ref);
#pragma unroll 1
            for (uint32_t k = 0; k < cnt; ++k) {
                const SurfelGeo& g = S.geo[first + k];
                const F3 n = mk3(g.nx, g.ny, g.nz);
                const float nd = dot(n, c.d);
                if (fabsf(nd) < 1e-6f) continue;
                const float t = dot(n, mk3(g.px, g.py, g.pz) - c.o) / nd;
                if (t <= 1e-5f || t >= c.best) continue;
                if (surfelR2(g, c.o + c.d * t) >= 1.0f) continue;
                c.best = t;
                c.bestIdx = first + k;
            }
            cloudPop(st, c);
        } else {
            const float4* n = reinterpret_cast<const float4*>(S.nodes + c.ref);
            const float4 p = n[0], q = n[1], r = n[2];
            const uint2 refs = reinterpret_cast<const uint2*>(S.nodes + c.ref)[6];  // left, right (not the padding)
            float tl = __builtin_huge_valf(), tr = __builtin_huge_valf();
            const bool hl = slab(c.o, c.inv, p.x, p.y, p.z, p.w, q.x, q.y, c.best, 1e-6f, tl);
            const bool hr = slab(c.o, c.inv, q.z, q.w, r.x, r.y, r.z, r.w, c.best, 1e-6f, tr);
            const bool left = hl && (!hr || tl <= tr);
            if (hl && hr) st.pushBounded(c.sp, left ? refs.y : refs.x, left ? tr : tl);
            c.ref = left ? refs.x : refs.y;
            if (!hl && !hr) cloudPop(st, c);
        }
    }
}

// A wave's leaf tests, packed: the (lane, surfel) pairs of up to 16 lanes at
// a leaf take one test each on all 64 lanes, four neighbouring lanes (a quad)
// per leaf.  A step of four tests one after the other costs the wave the same
// for one lane at a leaf as for 64, and few are there at a time (the walk:
// 7.5 leaves and 48 nodes per query).  A pair reads its lane's ray through the
// LDS crossbar; the quad's smallest accepted distance, the first of equal
// ones, is what the loop in leaf order ends with.  Every lane of the wave
// calls it; returns whether this lane's leaf was tested.
//
// The support test keeps its two IEEE divisions: deciding r2 < 1 by products
// outside a band of 4e-6 around the rim took as long (800x800x16 on 1M surfels
// 47.7 ms that way, 47.3 so; room of 100k surfels 24.5 and 24.4).
__device__ __forceinline__ int laneGet(int v, uint32_t from) { return __builtin_amdgcn_ds_bpermute((int)(from << 2), v); }
__device__ __forceinline__ float laneGetF(float v, uint32_t from) {
    return __int_as_float(laneGet(__float_as_int(v), from));
}
template <int kCtrl>
__device__ __forceinline__ float quadGet(float v) {  // of the lane that the quad permutation names
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, true));
}
constexpr uint32_t kLeafLanes = 16;

__device__ __forceinline__ bool cloudLeafRound(const DevScene& S, CloudLane& c, bool leaf) {
    const uint32_t lane = __lane_id();
    const unsigned long long m = __builtin_amdgcn_ballot_w64(leaf);
    const uint32_t n = (uint32_t)__popcll(m);
    const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    // Lane r of `owner` holds the r-th lane at a leaf (a permutation: the
    // other lanes follow).
    const uint32_t place = leaf ? below : n + (lane - below);
    const uint32_t owner = (uint32_t)__builtin_amdgcn_ds_permute((int)(place << 2), (int)lane);
    const uint32_t r = lane >> 2, k = lane & 3u;
    const uint32_t from = (uint32_t)laneGet((int)owner, r);
    const uint32_t ref = (uint32_t)laneGet((int)c.ref, from);
    const F3 o = mk3(laneGetF(c.o.x, from), laneGetF(c.o.y, from), laneGetF(c.o.z, from));
    const F3 d = mk3(laneGetF(c.d.x, from), laneGetF(c.d.y, from), laneGetF(c.d.z, from));
    const float best = laneGetF(c.best, from);
    float t = 0.0f;
    bool inside = false;  // hit, in front, in the support: all tests but that against best
    if (r < n && k < leafCount(ref)) {
        const float4* g = reinterpret_cast<const float4*>(S.geo + (leafFirst(ref) + k));
        const float4 g0 = g[0], g1 = g[1], g2 = g[2], g3 = g[3];
        const F3 pn = mk3(g1.x, g1.y, g1.z), p = mk3(g0.x, g0.y, g0.z);
        const float nd = dot(pn, d);
        t = dot(pn, p - o) / nd;
        const F3 x = o + d * t;
        const F3 q = x - p;
        const float a = dot(mk3(g2.x, g2.y, g2.z), q), b = dot(mk3(g3.x, g3.y, g3.z), q);
        const float uu = a / g0.w, vv = b / g1.w;
        inside = !(uu * uu + vv * vv >= 1.0f) && !(fabsf(nd) < 1e-6f) && !(t <= 1e-5f);
    }
    const bool ok = inside && !(t >= best);
    unsigned long long wins;
    float nt;
    if (__builtin_amdgcn_ballot_w64(ok && !(t < best)) == 0ull) {
        float q = ok ? t : __builtin_huge_valf();
        q = fminf(q, quadGet<0xB1>(q));
        q = fminf(q, quadGet<0x4E>(q));
        wins = __builtin_amdgcn_ballot_w64(ok && t == q);
        nt = laneGetF(q, (below << 2) & 63u);
    } else {
        // A NaN distance (a degenerate surfel or ray) was accepted: the tests
        // one after the other, each against the best before it (none is beyond
        // a NaN best).  A lane that accepted one, also if another took its
        // place, ends here with a NaN best (traceWave).
        const unsigned long long in = __builtin_amdgcn_ballot_w64(inside);
        const uint32_t mine = (uint32_t)(in >> (lane & 60u));
        const float t0 = quadGet<0x00>(t), t1 = quadGet<0x55>(t), t2 = quadGet<0xAA>(t), t3 = quadGet<0xFF>(t);
        float now = best;
        uint32_t win = 4u;
        bool was = false;
        if ((mine & 1u) && !(t0 >= now)) { now = t0; win = 0u; was = was || now != now; }
        if ((mine & 2u) && !(t1 >= now)) { now = t1; win = 1u; was = was || now != now; }
        if ((mine & 4u) && !(t2 >= now)) { now = t2; win = 2u; was = was || now != now; }
        if ((mine & 8u) && !(t3 >= now)) { now = t3; win = 3u; was = was || now != now; }
        if (was) now = __builtin_nanf("");
        wins = __builtin_amdgcn_ballot_w64(win == k);
        nt = laneGetF(now, (below << 2) & 63u);
        if (leaf && below < kLeafLanes && nt != nt) c.sp = c.base;
    }
    const bool tested = leaf && below < kLeafLanes;
    const uint32_t won = (uint32_t)(wins >> ((below << 2) & 63u)) & 15u;
    if (tested && won) {
        c.best = nt;
        c.bestIdx = leafFirst(c.ref) + (uint32_t)__ffs((int)won) - 1u;
    }
    return tested;
}

// intersectTriangle (KernelHelpers.h:248-277)
__device__ __forceinline__ bool intersectTri(F3 o, F3 d, F3 v0, F3 v1, F3 v2, float tMin, float& tOut) {
    const F3 e1 = v1 - v0, e2 = v2 - v0;
    const F3 h = cross(d, e2);
    const float a = dot(e1, h);
    if (fabsf(a) < 1.0e-4f) return false;
    const float f = 1.0f / a;
    const F3 s = o - v0;
    const float u = f * dot(s, h);
    if (u < 0.0f || u > 1.0f) return false;
    const F3 q = cross(s, e1);
    const float v = f * dot(d, q);
    if (v < 0.0f || u + v > 1.0f) return false;
    const float t = f * dot(e2, q);
    if (t <= tMin) return false;
    tOut = t;
    return true;
}

// intersectBLASMesh (IntersectionKernels.h:37-105)
template <bool kCount>
__device__ bool traverseMesh(const DevScene& S, const DevInstance& I, F3 o, F3 d, const LaneStack& st,
                             uint32_t base, LocalHit& out, Work& w) {
    const F3 inv = safeInvDir(d);
    float best = __builtin_huge_valf();
    float te;
    if (kCount) w.aabb++;  // the reference slab-tests the root when it pops it
    if (!slab(o, inv, I.rmnx, I.rmny, I.rmnz, I.rmxx, I.rmxy, I.rmxz, best, 1e-6f, te)) {
        if (kCount) w.pops++;
        return false;
    }
    bool firstPop = true;
    uint32_t sp = base;
    st.push(sp, I.rootRef, te);
    bool any = false;
    uint32_t bestTri = 0;
    while (sp > base) {
        const uint2 e = st.get(--sp);
        if (kCount) {
            w.pops++;
            if (!firstPop) w.aabb++;  // re-test of a popped box (root already counted)
            firstPop = false;
        }
        if (__uint_as_float(e.y) > best) continue;
        const uint32_t ref = e.x;
        if (ref & kLeafBit) {
            const uint32_t first = leafFirst(ref), cnt = leafCount(ref);
            if (kCount) w.prims += cnt;
            for (uint32_t k = 0; k < cnt; ++k) {
                const TriGeo tg = S.tris[first + k];
                float t;
                if (intersectTri(o, d, mk3(tg.v0x, tg.v0y, tg.v0z), mk3(tg.v1x, tg.v1y, tg.v1z),
                                 mk3(tg.v2x, tg.v2y, tg.v2z), 1e-4f, t) &&
                    t < best && t > 0.0f) {
                    best = t;
                    any = true;
                    bestTri = first + k;
                }
            }
            continue;
        }
        const float4* nd4 = reinterpret_cast<const float4*>(S.nodes + ref);
        const float4 a = nd4[0], b = nd4[1], c = nd4[2];
        const uint2 refs = reinterpret_cast<const uint2*>(S.nodes + ref)[6];  // left, right (not the padding)
        if (kCount) w.aabb += 2;
        float tl = __builtin_huge_valf(), tr = __builtin_huge_valf();
        const bool hl = slab(o, inv, a.x, a.y, a.z, a.w, b.x, b.y, best, 1e-6f, tl);
        const bool hr = slab(o, inv, b.z, b.w, c.x, c.y, c.z, c.w, best, 1e-6f, tr);
        if (hl && hr) {
            if (tl <= tr) {
                st.push(sp, refs.y, tr);
                st.push(sp, refs.x, tl);
            } else {
                st.push(sp, refs.x, tl);
                st.push(sp, refs.y, tr);
            }
        } else if (hl) {
            st.push(sp, refs.x, tl);
        } else if (hr) {
            st.push(sp, refs.y, tr);
        }
    }
    if (!any) return false;
    out.prim = bestTri;
    out.pos = toWorldPoint(I.o2w, o + d * best);
    return true;
}

// intersectScene, FirstHit mode (IntersectionKernels.h:954-1097).  The TLAS
// stack shares the lane's LDS stack below the BLAS entries.
// The scene's top level (TLAS nodes and instances), read where it lies in
// global memory (TopGlobal) or from a copy in LDS that a workgroup makes when
// it starts (TopLds: every lane of a wave reads the same few nodes and
// instances, which the LDS broadcasts without using the vector-memory path).
struct TopGlobal {
    const TlasNode* tlas;
    const DevInstance* inst;
};
constexpr uint32_t kTopLdsTlas = 15, kTopLdsInst = 8;
struct TopLds {
    TlasNode tlas[kTopLdsTlas];
    DevInstance inst[kTopLdsInst];
};
__host__ __device__ inline bool topFitsLds(const DevScene& S) {
    return S.nTlas <= kTopLdsTlas && S.nInst <= kTopLdsInst;
}
// Copy of the top level into LDS by the whole workgroup (then a barrier).
__device__ inline void loadTopLds(const DevScene& S, TopLds& t) {
    const uint32_t nt = S.nTlas * (uint32_t)(sizeof(TlasNode) / 4), ni = S.nInst * (uint32_t)(sizeof(DevInstance) / 4);
    const uint32_t* gt = reinterpret_cast<const uint32_t*>(S.tlas);
    const uint32_t* gi = reinterpret_cast<const uint32_t*>(S.inst);
    uint32_t* lt = reinterpret_cast<uint32_t*>(t.tlas);
    uint32_t* li = reinterpret_cast<uint32_t*>(t.inst);
    for (uint32_t k = threadIdx.x; k < nt; k += blockDim.x) lt[k] = gt[k];
    for (uint32_t k = threadIdx.x; k < ni; k += blockDim.x) li[k] = gi[k];
    __syncthreads();
}

// One query, its work counted as the reference's.
template <typename Top>
__device__ void intersectScene(const DevScene& S, const Top& top, F3 o, F3 d, const LaneStack& st, Hit& h, Work& w) {
    h.inst = kInvalid;
    if (S.nTlas == 0) return;
    const F3 inv = safeInvDir(d);
    float bestW = __builtin_huge_valf();
    uint32_t sp = 0;
    st.push(sp, 0u, 0.0f);
    while (sp > 0) {
        const uint32_t ni = st.get(--sp).x;
        const TlasNode nd = top.tlas[ni];
        w.pops++;
        w.aabb++;
        float te;
        if (!slab(o, inv, nd.mnx, nd.mny, nd.mnz, nd.mxx, nd.mxy, nd.mxz, bestW, 0.0f, te)) continue;
        if (nd.count == 0) {
            const TlasNode L = top.tlas[nd.left], R = top.tlas[nd.right];
            w.aabb += 2;
            float tl = __builtin_huge_valf(), tr = __builtin_huge_valf();
            const bool hl = slab(o, inv, L.mnx, L.mny, L.mnz, L.mxx, L.mxy, L.mxz, bestW, 0.0f, tl);
            const bool hr = slab(o, inv, R.mnx, R.mny, R.mnz, R.mxx, R.mxy, R.mxz, bestW, 0.0f, tr);
            if (hl && hr) {
                if (tl <= tr) {
                    st.push(sp, nd.right, 0.0f);
                    st.push(sp, nd.left, 0.0f);
                } else {
                    st.push(sp, nd.left, 0.0f);
                    st.push(sp, nd.right, 0.0f);
                }
            } else if (hl) {
                st.push(sp, nd.left, 0.0f);
            } else if (hr) {
                st.push(sp, nd.right, 0.0f);
            }
            continue;
        }
        const uint32_t ii = nd.left;
        const DevInstance& I = top.inst[ii];
        if (I.empty) continue;
        // toObjectSpace (KernelHelpers.h:217-227)
        float hv[4];
        mulv4(I.w2o, o.x, o.y, o.z, 1.0f, hv);
        const F3 oo = divs(mk3(hv[0], hv[1], hv[2]), hv[3]);
        mulv4(I.w2o, d.x, d.y, d.z, 0.0f, hv);
        const F3 od = normalize(mk3(hv[0], hv[1], hv[2]));
        LocalHit lh;
        bool acc;
        if (I.type == kGeoMesh)
            acc = traverseMesh<true>(S, I, oo, od, st, sp, lh, w);
        else
            acc = traverseCloud(S, I, oo, od, st, sp, lh, w);
        if (acc) {
            const float tw = dot(lh.pos - o, d);
            if (tw > 0.0f && tw < bestW) {
                bestW = tw;
                h.pos = lh.pos;
                h.inst = ii;
                h.prim = lh.prim;
            }
        }
    }
}

// Queries of a whole wave (intersectScene for every lane, FirstHit mode), by
// lanes that move on by themselves: a lane whose query ends hands its hit to
// the job, takes its next ray and starts again while the others still
// traverse.
//
// With one query per lane run to the wave's longest, and each iteration
// stepping the lanes at a leaf and the lanes at a node, the traversals were bound
// by vector instructions of which 16 % (photon trace) to 49 % (camera walk, shared
// samples) of the lanes took part; a query of 1M clustered surfels visits 50 nodes
// of the binary tree and 7.5 leaves.  So a wave takes one kind of step at a time,
// for the lanes that are at that kind: a leaf round (cloudLeafRound, 100 vector
// instructions; a node step has 170) once kLeafMin lanes or 1 / kLeafShare of those
// that traverse wait at a leaf, and the ends and starts of queries once 1 /
// kEndShare of the lanes that were traversing have ended.
//
// Camera walk of 16 passes at 800x800 on 1M surfels: 41.6 ms before, 28.4 now (87.5
// and 45.4 with independent samples).  Vector instructions take all of its cycles
// with shared samples, 84 % with independent ones, where L1 accesses take 80 %; a
// sixth of its time passes after the last pixel is drawn, while the longest pixels
// end.  kLeafMin 6, 8, 10, 16: 5 % slower to 2 % slower; kEndShare 1 and 3: 40 % and
// 5 % slower.  The photon and adjoint traces run the same with other values (within
// 1 %).
//
// Job: bool finish(bool done, const Hit&, const Work&, F3& o, F3& d) takes
// the hits of the lanes with done set (and the work of their queries in
// counting mode) and returns whether the lane goes on with a new ray (o, d),
// bool fetch(bool idle, F3& o, F3& d) gives idle lanes new work; both are
// called by every lane of the wave.  drained(): no more work to fetch
// (uniform over the wave).  kGoesOn: finish may give a lane a new ray.
// Counting mode runs the counting traversal, query by query.
constexpr uint32_t kLeafMin = 12, kLeafShare = 2, kEndShare = 2;

template <bool kCount, typename Top, typename Job>
__device__ __forceinline__ void traceWave(const DevScene& S, const Top& top, const LaneStack& st, Job& job) {
    if constexpr (kCount) {
        F3 o = mk3(0, 0, 0), d = mk3(0, 0, 1);
        bool has = false;
        Hit h{};
        Work w{};
        while (true) {
            has = job.finish(has, h, w, o, d);
            if (job.fetch(!has, o, d)) has = true;
            if (!__any(has)) {
                if (job.drained()) return;
                continue;
            }
            if (has) {
                w = Work{};
                intersectScene(S, top, o, d, st, h, w);
            }
        }
    }
    enum : uint32_t { kIdle, kTop, kCloud, kEnd };
    uint32_t state = kIdle;
    F3 o = mk3(0, 0, 0), d = mk3(0, 0, 1);
    CloudLane c{};
    c.ref = kRefDone;
    Hit h{};
    float bestW = 0.0f;
    uint32_t inst = 0;  // instance being traversed
    while (true) {
        // Ends and starts of queries, until the lanes that got a ray are in
        // the cloud (a ray that misses it ends here at once).
        while (true) {
            if (state == kCloud && c.ref == kRefDone) {
                if (c.best != c.best) cloudAgain(S, top.inst[inst].rootRef, st, c);  // a NaN distance was accepted
                if (c.bestIdx != kInvalid) {
                    const F3 x = c.o + c.d * c.best;
                    const float tw = dot(x - o, d);
                    if (tw > 0.0f && tw < bestW) {
                        bestW = tw;
                        h.pos = x;
                        h.inst = inst;
                        h.prim = c.bestIdx;
                    }
                }
                c.sp = c.base;
                state = kTop;
            }
            if (state == kTop) {
                const F3 inv = safeInvDir(d);
                state = kEnd;
                while (c.sp > 0) {
                    const uint32_t ni = st.get(--c.sp).x;
                    const TlasNode nd = top.tlas[ni];
                    float te;
                    if (!slab(o, inv, nd.mnx, nd.mny, nd.mnz, nd.mxx, nd.mxy, nd.mxz, bestW, 0.0f, te)) continue;
                    if (nd.count == 0) {
                        const TlasNode L = top.tlas[nd.left], R = top.tlas[nd.right];
                        float tl = __builtin_huge_valf(), tr = __builtin_huge_valf();
                        const bool hl = slab(o, inv, L.mnx, L.mny, L.mnz, L.mxx, L.mxy, L.mxz, bestW, 0.0f, tl);
                        const bool hr = slab(o, inv, R.mnx, R.mny, R.mnz, R.mxx, R.mxy, R.mxz, bestW, 0.0f, tr);
                        const bool left = hl && (!hr || tl <= tr);
                        if (hl && hr) st.push(c.sp, left ? nd.right : nd.left, 0.0f);
                        if (hl || hr) st.push(c.sp, left ? nd.left : nd.right, 0.0f);
                        continue;
                    }
                    const uint32_t ii = nd.left;
                    const DevInstance& I = top.inst[ii];
                    if (I.empty) continue;
                    // toObjectSpace (KernelHelpers.h:217-227)
                    float hv[4];
                    mulv4(I.w2o, o.x, o.y, o.z, 1.0f, hv);
                    const F3 oo = divs(mk3(hv[0], hv[1], hv[2]), hv[3]);
                    mulv4(I.w2o, d.x, d.y, d.z, 0.0f, hv);
                    const F3 od = normalize(mk3(hv[0], hv[1], hv[2]));
                    if (I.type == kGeoMesh) {
                        LocalHit lh;
                        Work w{};
                        if (traverseMesh<false>(S, I, oo, od, st, c.sp, lh, w)) {
                            const float tw = dot(lh.pos - o, d);
                            if (tw > 0.0f && tw < bestW) {
                                bestW = tw;
                                h.pos = lh.pos;
                                h.inst = ii;
                                h.prim = lh.prim;
                            }
                        }
                    } else if (cloudBegin(I, oo, od, c.sp, c)) {
                        inst = ii;
                        state = kCloud;
                        break;
                    }
                }
            }
            const bool more = job.finish(state == kEnd, h, Work{}, o, d);
            if (state == kEnd) state = more ? kTop : kIdle;
            if (job.fetch(state == kIdle, o, d)) state = kTop;
            if (state == kTop) {
                bestW = __builtin_huge_valf();
                h.inst = kInvalid;
                c.sp = 0;
                if (S.nTlas) st.push(c.sp, 0u, 0.0f);
            }
            if (!__any(state == kTop)) break;
        }
        const uint32_t started = (uint32_t)__popcll(__ballot(state == kCloud));
        if (started == 0u) {
            if (job.drained()) break;
            continue;
        }
        // (Without more rays for the lanes that end there is nothing to leave
        // the others for.)
        const uint32_t stay = !Job::kGoesOn && job.drained() ? 0u : started - (started + kEndShare - 1u) / kEndShare;
        while (true) {
            const bool run = state == kCloud && c.ref != kRefDone;
            const bool leaf = run && (c.ref & kLeafBit);
            const uint32_t running = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(run));
            if (running <= stay) break;
            const uint32_t leaves = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(leaf));
            if (leaves >= kLeafMin || leaves * kLeafShare >= running) {
                if (cloudLeafRound(S, c, leaf)) cloudPop(st, c);
            } else {
                if (run && !leaf) cloudNode(S, st, c);
            }
        }
    }
}

// Gradient of alpha_geom (intersectSurfel, KernelHelpers.h:637-669) with
// respect to the surfel's center, raw tangents, scales and beta, for the
// object-space ray (o, d): a reverse pass through the test's expressions
// (orthonormal frame from normalize(t_u) and Gram-Schmidt t_v, plane hit,
// (u, v) from the raw tangents, alpha = (1 - r^2)^(4 e^beta)).  g[0..2]
// center, g[3..5] t_u, g[6..8] t_v, g[9] s_u, g[10] s_v, g[11] beta.  False
// if the ray misses the support.
__device__ bool alphaGradient(const SurfelGeo& s, F3 o, F3 d, float g[12]) {
    const F3 p = mk3(s.px, s.py, s.pz), tu = mk3(s.tux, s.tuy, s.tuz), tv = mk3(s.tvx, s.tvy, s.tvz);
    const float lu = sqrtf(dot(tu, tu));
    const F3 uh = tu * (1.0f / lu);
    const float sdot = dot(uh, tv);
    const F3 wv = tv - uh * sdot;
    const float lw = sqrtf(dot(wv, wv));
    const F3 vh = wv * (1.0f / lw);
    const F3 m = cross(uh, vh);
    const float lm = sqrtf(dot(m, m));
    const F3 n = m * (1.0f / lm);
    const float nd = dot(n, d);
    if (fabsf(nd) < 1e-6f) return false;
    const F3 po = p - o;
    const float t = dot(n, po) / nd;
    const F3 r = (o + d * t) - p;
    const float U = dot(tu, r) / s.su, V = dot(tv, r) / s.sv;
    const float R = U * U + V * V;
    if (!(R < 1.0f)) return false;
    const float k = s.e4b;
    const float a = pow_r(1.0f - R, k);
    const float dadR = -k * a / (1.0f - R);
    const float gU = dadR * 2.0f * U, gV = dadR * 2.0f * V;
    const F3 gr = tu * (gU / s.su) + tv * (gV / s.sv);
    const float gt = dot(gr, d);
    const float gnp = gt / nd, gnd = -gt * t / nd;
    const F3 gp = n * gnp - gr;
    const F3 gn = po * gnp + d * gnd;
    const F3 gm = (gn - n * dot(n, gn)) * (1.0f / lm);
    F3 guh = cross(vh, gm);
    const F3 gvh = cross(gm, uh);
    const F3 gw = (gvh - vh * dot(vh, gvh)) * (1.0f / lw);
    F3 gtv = r * (gV / s.sv) + (gw - uh * dot(uh, gw));
    guh = guh - gw * sdot - tv * dot(uh, gw);
    const F3 gtu = r * (gU / s.su) + (guh - uh * dot(uh, guh)) * (1.0f / lu);
    g[0] = gp.x; g[1] = gp.y; g[2] = gp.z;
    g[3] = gtu.x; g[4] = gtu.y; g[5] = gtu.z;
    g[6] = gtv.x; g[7] = gtv.y; g[8] = gtv.z;
    g[9] = -gU * U / s.su;
    g[10] = -gV * V / s.sv;
    g[11] = a * (float)log((double)(1.0f - R)) * k;
    return true;
}

// buildIntersectionNormal (KernelHelpers.h:480-503)
__device__ __forceinline__ F3 hitNormal(const DevScene& S, const Hit& h) {
    const DevInstance& I = S.inst[h.inst];
    if (I.type == kGeoMesh) {
        const TriGeo tg = S.tris[h.prim];
        const F3 p0 = toWorldPoint(I.o2w, mk3(tg.v0x, tg.v0y, tg.v0z));
        const F3 p1 = toWorldPoint(I.o2w, mk3(tg.v1x, tg.v1y, tg.v1z));
        const F3 p2 = toWorldPoint(I.o2w, mk3(tg.v2x, tg.v2y, tg.v2z));
        return normalize(cross(p1 - p0, p2 - p0));
    }
    const SurfelShade sh = S.shade[h.prim];
    return mk3(sh.nsx, sh.nsy, sh.nsz);
}

// sampleCosineHemisphere(rng, n, dir, pdf) (KernelHelpers.h:317-337)
__device__ __forceinline__ void sampleCosine(Rng& rng, F3 n, F3& dir, float& pdf) {
    const float u1 = rng.nextFloat();
    const float u2 = rng.nextFloat();
    const float z = sqrtf(1.0f - u1);
    const float r = sqrtf(1.0f - z * z);
    const float phi = 2.0f * kPi * u2;
    const float x = r * cos_r(phi);
    const float y = r * sin_r(phi);
    const F3 up = fabsf(n.z) < 0.999f ? mk3(0, 0, 1) : mk3(1, 0, 0);
    const F3 tang = normalize(cross(up, n));
    const F3 bit = cross(n, tang);
    dir = normalize(tang * x + bit * y + n * z);
    pdf = fmaxf(0.0f, dot(dir, n)) / kPi;
}

// sampleUniformHemisphereAroundNormal (KernelHelpers.h:551-596)
__device__ __forceinline__ void sampleUniformHemi(Rng& rng, F3 normal, F3& dir, float& pdf) {
    const F3 n = normalize(normal);
    const float u1 = rng.nextFloat();
    const float u2 = rng.nextFloat();
    const float z = u1;
    const float phi = 2.0f * kPi * u2;
    const float r = sqrtf(fmaxf(0.0f, 1.0f - z * z));
    const float x = r * cos_r(phi);
    const float y = r * sin_r(phi);
    const float sign = copysignf(1.0f, n.z);
    const float a = -1.0f / (sign + n.z);
    const float b = n.x * n.y * a;
    const F3 t = mk3(1.0f + sign * n.x * n.x * a, sign * b, -sign * n.x);
    const F3 bt = mk3(b, sign + n.y * n.y * a, -n.y);
    dir = normalize(t * x + bt * y + n * z);
    pdf = 1.0f / (2.0f * kPi);
}

// applyRussianRoulette (KernelHelpers.h:1612-1657)
__device__ __forceinline__ bool russianRoulette(Rng& rng, uint32_t bounce, F3& T, uint32_t start) {
    if (bounce < start) return true;
    if (!isfinite(T.x) || !isfinite(T.y) || !isfinite(T.z)) return false;
    const float lum = 0.2126f * T.x + 0.7152f * T.y + 0.0722f * T.z;
    const float p = fminf(fmaxf(lum, 0.0f), 0.99f);
    if (rng.nextFloat() > p) return false;
    float c = 1.0f / p;
    c = fminf(c, 10.0f);
    T = T * c;
    return true;
}

// sampleMeshAreaLight (KernelHelpers.h:340-449)
__device__ bool sampleLight(const DevScene& S, Rng& rng, F3& pos, F3& dir, F3& power) {
    const uint32_t lc = S.nLights;
    if (lc == 0) return false;
    const float ul = rng.nextFloat();
    const uint32_t li = min((uint32_t)(ul * (float)lc), lc - 1u);
    const DevLight L = S.lights[li];
    if (L.triCount == 0u || L.area <= 0.0f) return false;
    const float ut = rng.nextFloat();
    uint32_t lo = 0u, hi = L.triCount - 1u;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1u;
        if (ut <= S.emTris[L.triOffset + mid].cdf) hi = mid;
        else lo = mid + 1u;
    }
    const TriGeo tg = S.tris[S.emTris[L.triOffset + lo].tri];
    const F3 v0 = mk3(tg.v0x, tg.v0y, tg.v0z), v1 = mk3(tg.v1x, tg.v1y, tg.v1z), v2 = mk3(tg.v2x, tg.v2y, tg.v2z);
    const float u1 = rng.nextFloat();
    const float u2 = rng.nextFloat();
    const float s1 = sqrtf(u1);
    const float b0 = 1.0f - s1, b1 = s1 * (1.0f - u2), b2 = s1 * u2;
    const F3 xo = v0 * b0 + v1 * b1 + v2 * b2;
    const float* o2w = S.inst[L.instance].o2w;
    const F3 p0 = toWorldPoint(o2w, v0), p1 = toWorldPoint(o2w, v1), p2 = toWorldPoint(o2w, v2);
    const F3 e0 = p1 - p0, e1 = p2 - p0;
    F3 n = mk3(e0.y * e1.z - e0.z * e1.y, e0.z * e1.x - e0.x * e1.z, e0.x * e1.y - e0.y * e1.x);
    const float nl = sqrtf(dot(n, n));
    if (nl <= 0.0f) return false;
    n = divs(n, nl);
    float pdf;
    sampleCosine(rng, n, dir, pdf);
    pos = toWorldPoint(o2w, xo);
    power = mk3(L.cr, L.cg, L.cb) * L.power;
    return true;
}

// worldToCellClamped (KernelHelpers.h:920-934)
__device__ __forceinline__ void worldToCell(const DevGrid& g, F3 p, int& x, int& y, int& z) {
    const F3 f = divv(p - mk3(g.ox, g.oy, g.oz), mk3(g.cx, g.cy, g.cz));
    x = min(max((int)floorf(f.x), 0), g.rx - 1);
    y = min(max((int)floorf(f.y), 0), g.ry - 1);
    z = min(max((int)floorf(f.z), 0), g.rz - 1);
}

// Rows of the grid that can hold a photon within radius r of a point of the
// box [qlo, qhi] (one point: qlo = qhi): a row (cy, cz) is skipped when its
// y-z extent lies farther than r from the box, and otherwise its x range
// shrinks to the chords of the sphere.  Every bound is widened by a margin,
// 1e-3 of a cell plus 2e-6 of the coordinates, far above the binary32 rounding
// of worldToCell, of the distance test and of the bounds themselves (a dozen
// roundings of 6e-8 relative to the coordinates), and boundary cells, which
// also hold the photons that worldToCell clamps into them, extend to infinity.
// A photon in a skipped cell therefore fails the reference's d2 > r2 test, so
// skipping it leaves the sum unchanged.  Nothing here enters a sum, so the
// bounds need no correctly rounded operations: with an IEEE square root and
// two IEEE divisions per row the 25 rows of a gather cost more vector
// instructions than its photons.
struct GridRows {
    float c, inv;          // cell size, 1 / cell size
    float ylo, yhi, zlo, zhi;  // gaps to the faces of cell 0: ylo + i c and yhi - i c to cell i's
    float x0, x1;          // the box's x range, widened, in cells
    float room;            // r^2 and a little

    __device__ __forceinline__ GridRows(const DevGrid& g, F3 qlo, F3 qhi, float r2) {
        c = g.cx;
        inv = g.inv;
        const float m = 1e-3f * c;
        const float mx = m + 2e-6f * (fmaxf(fabsf(qlo.x), fabsf(qhi.x)) + fabsf(g.ox) + g.radius);
        const float my = m + 2e-6f * (fmaxf(fabsf(qlo.y), fabsf(qhi.y)) + fabsf(g.oy) + g.radius);
        const float mz = m + 2e-6f * (fmaxf(fabsf(qlo.z), fabsf(qhi.z)) + fabsf(g.oz) + g.radius);
        ylo = g.oy - my - qhi.y;
        yhi = qlo.y - g.oy - my - c;
        zlo = g.oz - mz - qhi.z;
        zhi = qlo.z - g.oz - mz - c;
        x0 = (qlo.x - mx - g.ox) * inv;
        x1 = (qhi.x + mx - g.ox) * inv;
        room = r2 * 1.001f;
    }
    __device__ __forceinline__ float gap(float lo, float hi, int i, int res) const {
        const float t = (float)i * c;
        const float a = i == 0 ? 0.0f : lo + t, b = i == res - 1 ? 0.0f : hi - t;
        return fmaxf(fmaxf(a, b), 0.0f);
    }
    // what slice cz leaves of room
    __device__ __forceinline__ float slice(const DevGrid& g, int cz) const {
        const float d = gap(zlo, zhi, cz, g.rz);
        return room - d * d;
    }
    __device__ __forceinline__ bool span(const DevGrid& g, float left, int cy, int lx, int hx, int& ax, int& bx) const {
        const float d = gap(ylo, yhi, cy, g.ry);
        const float rest = left - d * d;
        const float hw = __builtin_amdgcn_sqrtf(fmaxf(rest, 0.0f)) * inv;
        // The first and last cells have no outer face (photons beyond the grid
        // are stored there): a point beyond it keeps them.
        ax = min(max((int)floorf(x0 - hw), lx), g.rx - 1);
        bx = max(min((int)floorf(x1 + hw), hx), 0);
        return rest >= 0.0f && ax <= bx;
    }
};

typedef __attribute__((address_space(4))) const float4 ConstF4;
typedef __attribute__((address_space(4))) const float ConstF;
typedef __attribute__((address_space(4))) const uint32_t ConstU32;

__device__ __forceinline__ float waveMinF(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ float waveMaxF(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// A photon's tests and its part of the sum (its power is stored divided by
// the disc's area, k_cell_payload).
__device__ __forceinline__ void gatherPhoton(F3& E, F3 q, F3 n, float r2, const float4& pp, const float4& dp, float pz) {
    const F3 dd = mk3(pp.x, pp.y, pp.z) - q;
    // dot(n, -dir) == dot(-n, dir) exactly (negation is exact).
    const float cosine = dot(n, -mk3(dp.x, dp.y, dp.z));
    const float d2 = dot(dd, dd);
    if (!(cosine < 0.0f) && !(d2 > r2)) E = E + mk3(pp.w, dp.w, pz);
}

// The gather of a full wave whose points share one cell box and lie close
// together (qlo..qhi, within kWaveSpread of the radius on every axis): the
// rows and photons are the same for every lane, so they are walked once for
// the wave with scalar loads, and each lane applies its own tests to every
// photon of the rows' spans for the whole wave.  A lane adds exactly the
// photons of its own box that pass its tests, in the same order as the
// per-lane walk, so the sums are the same to the bit.
constexpr float kWaveSpread = 0.5f;
__device__ F3 gatherWave(const DevGrid& g, F3 q, F3 n, F3 qlo, F3 qhi, float r2, int lx, int ly, int lz, int hx,
                         int hy, int hz) {
    F3 E = mk3(0, 0, 0);
    auto addPhoton = [&](const float4& pp, const float4& dp, float pz) { gatherPhoton(E, q, n, r2, pp, dp, pz); };
    const GridRows rows(g, qlo, qhi, r2);
    const ConstF4* pos = (const ConstF4*)g.posPow;
    const ConstF4* dir = (const ConstF4*)g.dirPow;
    const ConstF* pzs = (const ConstF*)g.powZ;
    const ConstU32* cs = (const ConstU32*)g.cellStart;
    for (int cz = lz; cz <= hz; ++cz) {
        const float left = rows.slice(g, cz);
        for (int cy = ly; cy <= hy; ++cy) {
            int ax, bx;
            if (!rows.span(g, left, cy, lx, hx, ax, bx)) continue;
            ax = __builtin_amdgcn_readfirstlane(ax);
            bx = __builtin_amdgcn_readfirstlane(bx);
            const uint32_t row = (uint32_t)((cz * g.ry + cy) * g.rx);
            __asm__ volatile("");
            uint32_t j = cs[row + ax];
            const uint32_t b = cs[row + bx + 1];
            for (; j + 4 <= b; j += 4) {
                const float4 p0 = make_float4(pos[j].x, pos[j].y, pos[j].z, pos[j].w);
                const float4 p1 = make_float4(pos[j + 1].x, pos[j + 1].y, pos[j + 1].z, pos[j + 1].w);
                const float4 p2 = make_float4(pos[j + 2].x, pos[j + 2].y, pos[j + 2].z, pos[j + 2].w);
                const float4 p3 = make_float4(pos[j + 3].x, pos[j + 3].y, pos[j + 3].z, pos[j + 3].w);
                const float4 d0 = make_float4(dir[j].x, dir[j].y, dir[j].z, dir[j].w);
                const float4 d1 = make_float4(dir[j + 1].x, dir[j + 1].y, dir[j + 1].z, dir[j + 1].w);
                const float4 d2 = make_float4(dir[j + 2].x, dir[j + 2].y, dir[j + 2].z, dir[j + 2].w);
                const float4 d3 = make_float4(dir[j + 3].x, dir[j + 3].y, dir[j + 3].z, dir[j + 3].w);
                const float z0 = pzs[j], z1 = pzs[j + 1], z2 = pzs[j + 2], z3 = pzs[j + 3];
                addPhoton(p0, d0, z0);
                addPhoton(p1, d1, z1);
                addPhoton(p2, d2, z2);
                addPhoton(p3, d3, z3);
            }
            for (; j < b; ++j)
                addPhoton(make_float4(pos[j].x, pos[j].y, pos[j].z, pos[j].w),
                          make_float4(dir[j].x, dir[j].y, dir[j].z, dir[j].w), pzs[j]);
        }
    }
    return E;
}

// gatherDiffuseIrradianceAtPoint (KernelHelpers.h:990-1037).  Photons are
// stored sorted by (cell, deposit index), so the cells of one grid row form
// one contiguous range; summation order equals the reference's cell-by-cell,
// photon-by-photon order.  Cells that cannot hold an accepted photon are not
// scanned (GridRows).  Memory-level parallelism: the row bounds of a whole
// z-slice are loaded before any photon of that slice, and photons are loaded
// two at a time (added in order).  Counting mode counts the reference's
// cells and photons (the whole box), not the scanned ones.  kWave (the
// camera gather, whose waves hold cell-sorted points, with shared seeds
// often the same point several times): a wave whose points share a cell box
// and lie close together gathers through gatherWave.
constexpr int kSliceRows = 6;  // cells per axis: 4 + 1, +1 for rounding

template <bool kCount, bool kWave = false>
__device__ F3 gatherIrradiance(const DevGrid& g, F3 q, F3 n, Work& w) {
    if (kCount) w.gathers++;
    if (!g.valid) return mk3(0, 0, 0);
    const float r = g.radius;
    const float r2 = r * r;
    int lx, ly, lz, hx, hy, hz;
    worldToCell(g, q - mk3(r, r, r), lx, ly, lz);
    worldToCell(g, q + mk3(r, r, r), hx, hy, hz);
    F3 E = mk3(0, 0, 0);
    bool waveDone = false;
    if (kWave && !kCount && __builtin_amdgcn_ballot_w64(true) == ~0ull) {
        const int ulx = __builtin_amdgcn_readfirstlane(lx), uly = __builtin_amdgcn_readfirstlane(ly),
                  ulz = __builtin_amdgcn_readfirstlane(lz), uhx = __builtin_amdgcn_readfirstlane(hx),
                  uhy = __builtin_amdgcn_readfirstlane(hy), uhz = __builtin_amdgcn_readfirstlane(hz);
        if (__builtin_amdgcn_ballot_w64(lx != ulx || ly != uly || lz != ulz || hx != uhx || hy != uhy || hz != uhz) ==
            0ull) {
            const F3 qlo = mk3(waveMinF(q.x), waveMinF(q.y), waveMinF(q.z));
            const F3 qhi = mk3(waveMaxF(q.x), waveMaxF(q.y), waveMaxF(q.z));
            const F3 ext = qhi - qlo;
            if (fmaxf(fmaxf(ext.x, ext.y), ext.z) <= kWaveSpread * r) {
                E = gatherWave(g, q, n, qlo, qhi, r2, ulx, uly, ulz, uhx, uhy, uhz);
                waveDone = true;
            }
        }
    }
    if (!waveDone) {
    auto addPhoton = [&](const float4& pp, const float4& dp, float pz) { gatherPhoton(E, q, n, r2, pp, dp, pz); };
    const GridRows rows(g, q, q, r2);
    for (int cz = lz; cz <= hz; ++cz) {
        const float left = rows.slice(g, cz);
        for (int cy0 = ly; cy0 <= hy; cy0 += kSliceRows) {
            uint32_t ra[kSliceRows], rb[kSliceRows];
#pragma unroll
            for (int k = 0; k < kSliceRows; ++k) {
                const int cy = cy0 + k;
                ra[k] = rb[k] = 0u;
                int ax, bx;
                if (cy <= hy && rows.span(g, left, cy, lx, hx, ax, bx)) {
                    const uint32_t row = (uint32_t)((cz * g.ry + cy) * g.rx);
                    ra[k] = g.cellStart[row + ax];
                    rb[k] = g.cellStart[row + bx + 1];
                }
            }
#pragma unroll
            for (int k = 0; k < kSliceRows; ++k) {
                if (kCount && cy0 + k <= hy) {
                    const uint32_t row = (uint32_t)((cz * g.ry + cy0 + k) * g.rx);
                    w.cells += (uint32_t)(hx - lx + 1);
                    w.photons += g.cellStart[row + hx + 1] - g.cellStart[row + lx];
                    for (int cx = lx; cx <= hx; ++cx) w.cellsNE += g.cellStart[row + cx + 1] > g.cellStart[row + cx];
                }
                uint32_t j = ra[k];
                const uint32_t b = rb[k];
                // Two at a time, then the last: rows hold few photons (2 to 3
                // of the 1M-surfel workload's map).
                for (; j + 2 <= b; j += 2) {
                    const float4 p0 = g.posPow[j], p1 = g.posPow[j + 1];
                    const float4 d0 = g.dirPow[j], d1 = g.dirPow[j + 1];
                    const float z0 = g.powZ[j], z1 = g.powZ[j + 1];
                    addPhoton(p0, d0, z0);
                    addPhoton(p1, d1, z1);
                }
                if (j < b) addPhoton(g.posPow[j], g.dirPow[j], g.powZ[j]);
            }
        }
    }
    }
    const uint32_t T = *g.attempted;
    const uint32_t D = min(T, g.capacity);
    if (D == 0u) return mk3(0, 0, 0);
    return E * ((float)T / (float)D);
}

// makePrimaryRayFromPixelJitteredFov (KernelHelpers.h:764-796)
struct DevCamera {
    float invView[16];
    uint32_t W, H;
    float fx, fy;
};

__device__ __forceinline__ void primaryRay(const DevCamera& c, float px, float py, float jx, float jy, F3& o,
                                           F3& d) {
    const float W = (float)c.W, H = (float)c.H;
    const float u = px + 0.5f + jx;
    const float v = py + 0.5f + jy;
    const float vf = H - v;
    const float ndcX = 2.0f * u / W - 1.0f;
    const float ndcY = 2.0f * vf / H - 1.0f;
    const F3 dc = normalize(mk3(ndcX * (0.5f * W) / c.fx, ndcY * (0.5f * H) / c.fy, -1.0f));
    d = transformDirection(c.invView, dc);
    o = transformPoint(c.invView, mk3(0, 0, 0));
}

}  // namespace pale
