// pale_kernels.hip -- gfx950 kernels of the beta-surfel photon-mapping
// renderer and its opacity adjoint.
//
// Wavefront structure: every bounce is one traversal kernel over a ray queue
// followed by a stable (order-preserving) compaction of its outputs.  Queue
// slot = rank in the previous queue, so each ray meets the per-item random
// stream the reference's sequential order gives it (the reference seeds every
// work item from its queue slot, PrimalKernels.cpp:80-82,
// AdjointKernels.cpp:99-101).  Counts stay on the device; no kernel waits for
// the host.
#include <mutex>
#include <algorithm>
#include <cstddef>
#include <vector>

#include "pale_kernels.h"

namespace pale {

namespace {

constexpr uint32_t kScanThreads = 256;
constexpr uint32_t kTileSpan = kTile / kScanThreads;  // items per thread

enum : uint32_t { kNone = 0, kNullT = 1, kReflectS = 2, kTransmitS = 3, kProjection = 4 };

__device__ __forceinline__ uint32_t laneId() { return __lane_id(); }

// Wave-level count of a predicate, one atomic per wave.
__device__ __forceinline__ void waveCount(bool pred, unsigned long long* counter) {
    const unsigned long long m = __ballot(pred);
    if (laneId() == __ffsll((long long)__ballot(1)) - 1 && m) atomicAdd(counter, (unsigned long long)__popcll(m));
}

__device__ __forceinline__ uint32_t waveSum(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Flush a thread's work counters: one atomic per counter per wave.  Every
// lane of the wave must call this.
__device__ __forceinline__ void flushWork(const Work& w, DevState* st, int cls) {
    const uint32_t v[7] = {waveSum(w.pops), waveSum(w.aabb), waveSum(w.prims), waveSum(w.gathers),
                           waveSum(w.cells), waveSum(w.cellsNE), waveSum(w.photons)};
    if (__lane_id() == 0) {
#pragma unroll
        for (int k = 0; k < 7; ++k)
            if (v[k]) atomicAdd(&st->work[cls][k], (unsigned long long)v[k]);
    }
}

__device__ __forceinline__ void addWork(Work& w, const Work& q) {
    w.pops += q.pops;
    w.aabb += q.aabb;
    w.prims += q.prims;
}

// Exclusive scan over a 256-thread block; `total` receives the block sum.
__device__ __forceinline__ uint32_t blockExclusiveScan(uint32_t v, uint32_t& total) {
    __shared__ uint32_t waveTotals[kScanThreads / 64 + 1];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= (uint32_t)o) x += y;
    }
    if (lane == 63u) waveTotals[wave] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t s = 0;
        for (uint32_t w = 0; w < kScanThreads / 64; ++w) {
            const uint32_t t = waveTotals[w];
            waveTotals[w] = s;
            s += t;
        }
        waveTotals[kScanThreads / 64] = s;
    }
    __syncthreads();
    const uint32_t excl = x - v + waveTotals[wave];
    total = waveTotals[kScanThreads / 64];
    __syncthreads();
    return excl;
}

__device__ __forceinline__ uint32_t loadCount(const uint32_t* count, uint32_t maxItems) {
    const uint32_t n = *count;
    return n < maxItems ? n : maxItems;
}

__device__ __forceinline__ LaneStack laneStack(uint2* lds, uint32_t depth) {
    return LaneStack{(LdsUint2*)(lds + threadIdx.x), depth, nullptr, depth};
}

// A trace's stack: its first inLds entries in LDS, the rest in the lane's part
// of the spill area, so that more waves fit on a CU; spill == nullptr: all in
// LDS.
__device__ __forceinline__ LaneStack walkStack(uint2* lds, uint32_t depth, uint2* spill, uint32_t inLds) {
    if (!spill) return laneStack(lds, depth);
    const uint32_t l = blockIdx.x * kTraceBlock + threadIdx.x;
    return LaneStack{(LdsUint2*)(lds + threadIdx.x), depth, spill + (size_t)l * (depth - inLds), inLds};
}

__device__ __forceinline__ float4 f4(F3 v, float w) { return make_float4(v.x, v.y, v.z, w); }
__device__ __forceinline__ float u2f(uint32_t u) { return __uint_as_float(u); }
__device__ __forceinline__ uint32_t f2u(float f) { return __float_as_uint(f); }

}  // namespace

// ---------------------------------------------------------------- small --
__global__ void k_fill(uint32_t* p, uint32_t n, uint32_t v) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    do {
        p[i] = v;
    } while (nextItem(i, gridDim.x * blockDim.x, n));
}
__global__ void k_fillf(float* p, uint32_t n, float v) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    do {
        p[i] = v;
    } while (nextItem(i, gridDim.x * blockDim.x, n));
}
__global__ void k_iota(uint32_t* p, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    do {
        p[i] = i;
    } while (nextItem(i, gridDim.x * blockDim.x, n));
}

// Between the launches of the photon stage.  Seed schedule of
// submitPhotonMappingKernel (SyclBridge.cpp:83-143): one draw per emitter
// launch, per executed bounce and per camera.  bounce kNextDraw always draws
// (an emitter launch, a camera); a bounce takes over the queue that the launch
// before it wrote and draws only if it is not empty; kNextEnd only adds the
// last bounce's deposits (photonCount counts deposit attempts, the reference's
// counter T; only the first `cap` are stored).  The next bounce may pass a
// reservoir's capacity if the deposits so far plus one per queued photon do.
// The tile states of the next compaction are cleared.
__global__ __launch_bounds__(256) void k_photon_next(DevState* st, const uint32_t* table, uint32_t len, int bounce,
                                                     uint32_t resvCap, TileStates ts, uint32_t tiles) {
    for (uint32_t k = threadIdx.x; k < tiles; k += blockDim.x) ts.state[k] = 0ull;
    if (threadIdx.x < kTraceRegions) st->traceNext[threadIdx.x * kCursorStride] = 0u;
    if (threadIdx.x != 0) return;
    const uint32_t deposits = st->photonCount + st->depTotal;
    st->photonCount = deposits;
    st->depTotal = 0;
    st->ticket = 0;
    if (bounce == kNextEnd) return;
    if (bounce >= 0) {
        const uint32_t q = st->extTotal;
        st->qCount = q;
        st->resv = (resvCap && q && (uint64_t)deposits + (uint64_t)q > (uint64_t)resvCap) ? 1u : 0u;
        if (q == 0) return;
    }
    const uint32_t c = st->cursor;
    st->number = c < len ? table[c] : 0u;
    st->cursor = c + 1;
}

// Between the bounces of the adjoint: the queue and the events that the bounce
// before wrote are taken over, the tile states cleared.  In a batch (nSegs > 0)
// also where each segment's rays start and end in the queue (it stays in
// segment order: raygen writes it so, compaction is stable; segFirst has the
// first of every segment present, kInvalid for the others, whose first and end
// become 0), the places of the views' groups for the trace's interleaved order
// (K segments x the most rays of one), and segNext cleared for the bounce.
__global__ __launch_bounds__(256) void k_adj_next(DevState* st, int bounce, uint32_t poolCap, TileStates ts,
                                                  uint32_t tiles, uint32_t* segFirst, uint32_t* segEnd,
                                                  uint32_t* segNext, uint32_t nSegs, uint4* groups, uint32_t nGroups,
                                                  const uint32_t* groupSegs) {
    for (uint32_t k = threadIdx.x; k < tiles; k += blockDim.x) ts.state[k] = 0ull;
    if (threadIdx.x < kTraceRegions) st->traceNext[threadIdx.x * kCursorStride] = 0u;
    __shared__ uint32_t sQueue;
    if (threadIdx.x == 0) {
        const uint32_t n = st->evPool + st->evTotal;
        st->evPool = n < poolCap ? n : poolCap;
        st->evTotal = 0;
        st->ticket = 0;
        if (bounce > 0) st->qCount = st->extTotal;
        sQueue = st->qCount;
    }
    if (!nSegs || bounce == kNextEnd) return;
    __syncthreads();
    if (threadIdx.x < 64u) {
        uint32_t after = sQueue;  // where the segment after this chunk starts
        for (uint32_t base = (nSegs - 1u) & ~63u;; base -= 64u) {
            const uint32_t s = base + threadIdx.x;
            const uint32_t first = s < nSegs ? segFirst[s] : kInvalid;
            uint32_t m = first;  // the smallest first of this and later segments (they ascend)
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t v = __shfl_down(m, o, 64);
                if (threadIdx.x + (uint32_t)o < 64u) m = min(m, v);
            }
            const uint32_t next = __shfl_down(m, 1, 64);
            const uint32_t end = min(threadIdx.x < 63u ? next : kInvalid, after);
            if (s < nSegs) {
                segFirst[s] = first == kInvalid ? 0u : first;
                segEnd[s] = first == kInvalid ? 0u : end;
            }
            after = min(after, (uint32_t)__shfl(m, 0, 64));
            if (base == 0u) break;
        }
    }
    __syncthreads();
    for (uint32_t s = threadIdx.x; s < nSegs; s += blockDim.x) segNext[s] = kInvalid;
    for (uint32_t g = threadIdx.x; g < nGroups; g += blockDim.x) {
        const uint4 gr = groups[g];
        uint32_t most = 0;
        for (uint32_t k = 0; k < gr.y; ++k) {
            const uint32_t s = groupSegs[gr.x + k];
            most = max(most, segEnd[s] - segFirst[s]);
        }
        groups[g].w = most;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    uint32_t place = 0;
    for (uint32_t g = 0; g < nGroups; ++g) {
        groups[g].z = place;
        place += groups[g].y * groups[g].w;
    }
}

// Start of a served view: its passes draw from `number` (+ pass); the
// camera-gather counters restart, the photon map's stay.
__global__ void k_begin_view(DevState* st, uint32_t number) {
    if (blockIdx.x != 0) return;
    const uint32_t t = threadIdx.x;
    if (t < 8) st->work[kWorkGather][t] = 0ull;
    if (t == 0) {
        st->number = number;
        st->gatherQ = 0ull;
        st->entries = 0u;
        st->overflow = 0u;
    }
}

// ------------------------------------------------------- compaction --
// Offsets of a launch's items in the compacted outputs, in one pass: the
// workgroups take tiles of kTile items in ticket order, publish their tile's
// counts, add up those of the tiles before until one has published its prefix,
// and publish their own (decoupled look-back, Merrill and Garland 2016).  A
// tile's ticket is drawn by a running workgroup, and a workgroup waits only for
// earlier tickets after it has published its own counts, so every wait ends.
// The writers of the outputs then go on with them in registers: with staged
// outputs, flags, a count, a scan and a scatter launch per output a bounce took
// 9 launches (adjoint: 12) instead of 3 and moved every ray, deposit and event
// twice more.  Per bounce at 640,000 rays those took about 260 us of an adjoint
// bounce; k_adj_shade takes 126 us with the shading in it.
//
// A tile's state is one word, so that its parts are seen together: 2 bits of
// what it holds, 31 bits for each of two counts.
__device__ __forceinline__ uint32_t tileTicket(uint32_t* ticket) {
    __shared__ uint32_t t;
    if (threadIdx.x == 0) t = atomicAdd(ticket, 1u);
    __syncthreads();
    return t;
}
constexpr uint64_t kTileCounts = 1ull << 62, kTilePrefix = 2ull << 62, kTileValue = (1ull << 62) - 1ull;

// Publishes the tile's sum, returns the sum of the tiles before it.  One whole
// wave of the workgroup calls it.
__device__ __forceinline__ uint64_t lookBack(unsigned long long* state, uint32_t tile, uint64_t sum) {
    const uint32_t lane = laneId();
    uint64_t before = 0;
    if (tile > 0u) {
        if (lane == 0) __hip_atomic_store(state + tile, kTileCounts | sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int64_t at = (int64_t)tile - 1;
        while (true) {
            const int64_t t = at - (int64_t)lane;
            const uint64_t w =
                t >= 0 ? __hip_atomic_load(state + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : kTilePrefix;
            const unsigned long long prefix = __ballot((w & kTilePrefix) != 0ull), none = __ballot((w >> 62) == 0ull);
            const uint32_t p = prefix ? (uint32_t)__ffsll((long long)prefix) - 1u : 64u;
            if (none && (uint32_t)__ffsll((long long)none) - 1u < p) {
                __builtin_amdgcn_s_sleep(2);
                continue;
            }
            uint64_t c = lane <= p ? (w & kTileValue) : 0ull;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
            before += c;
            if (p < 64u) break;
            at -= 64;
        }
    }
    if (lane == 0)
        __hip_atomic_store(state + tile, kTilePrefix | (before + sum), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return before;
}

struct TileOffset {
    uint32_t a, b;        // this thread's places
    uint32_t endA, endB;  // the counts up to and with this tile
};
// Every thread of the workgroup calls it.
__device__ __forceinline__ TileOffset tileOffsets(TileStates ts, uint32_t tile, bool a, bool b) {
    __shared__ uint32_t waveA[kTile / 64], waveB[kTile / 64];
    __shared__ uint64_t sBase, sSum;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const unsigned long long ma = __ballot(a), mb = __ballot(b);
    if (lane == 0) {
        waveA[wave] = (uint32_t)__popcll(ma);
        waveB[wave] = (uint32_t)__popcll(mb);
    }
    __syncthreads();
    if (wave == 0) {
        uint64_t v = lane < kTile / 64 ? ((uint64_t)waveA[lane] << 31) | waveB[lane] : 0ull;
        const uint64_t own = v;
#pragma unroll
        for (int o = 1; o < (int)(kTile / 64); o <<= 1) {
            const uint64_t y = __shfl_up(v, o, 64);
            if (lane >= (uint32_t)o) v += y;
        }
        const uint64_t sum = __shfl(v, kTile / 64 - 1, 64);
        if (lane < kTile / 64) {
            waveA[lane] = (uint32_t)((v - own) >> 31);
            waveB[lane] = (uint32_t)((v - own) & 0x7FFFFFFFull);
        }
        const uint64_t before = lookBack(ts.state, tile, sum);
        if (lane == 0) {
            sBase = before;
            sSum = sum;
        }
    }
    __syncthreads();
    const uint64_t base = sBase, end = sBase + sSum;
    const unsigned long long below = (1ull << lane) - 1ull;
    return TileOffset{(uint32_t)(base >> 31) + waveA[wave] + (uint32_t)__popcll(ma & below),
                      (uint32_t)(base & 0x7FFFFFFFull) + waveB[wave] + (uint32_t)__popcll(mb & below),
                      (uint32_t)(end >> 31), (uint32_t)(end & 0x7FFFFFFFull)};
}

// ------------------------------------------------------- queue traces --
// Rays of a queue for the waves of a persistent grid: 64 consecutive rays (a
// unit) at a time, given to the wave's lanes as they fall idle.  A wave starts
// with the unit at its own place in the grid; the units after those go round
// the regions, and the waves of a region claim them from its counter.  With one
// counter and every unit claimed from it, the claims bounded the trace: 36
// bounces of 1M photons in a 100k-surfel room 18.4 ms, with the first units
// given 15.7 ms, with a counter per region 15.1 ms; 6 adjoint bounces of 167k
// rays in a 775-surfel scene 340 us against 170 us.
struct QueueCursor {
    uint32_t* next;      // claims of the region, zero at the start of a launch
    uint32_t end;        // rays to hand out
    uint32_t regions, region, own;  // own: units that the waves start with
    uint32_t at, to;     // the wave's untaken rays
    bool empty;

    __device__ QueueCursor(uint32_t* n, uint32_t e) : end(e) {
        const uint32_t waves = blockDim.x / 64u;
        regions = min(kTraceRegions, gridDim.x);
        region = blockIdx.x % regions;
        next = n + region * kCursorStride;
        own = gridDim.x * waves;
        at = (blockIdx.x * waves + __builtin_amdgcn_readfirstlane(threadIdx.x / 64u)) * 64u;
        to = min(at + 64u, end);
        empty = at >= end;
    }
    // Every lane of the wave calls it; false: no ray for this lane now (t
    // stays as it is).
    __device__ __forceinline__ bool take(bool want, uint32_t& t) {
        const unsigned long long need = __ballot(want);
        if (!need || empty) return false;
        const uint32_t lane = laneId();
        if (at >= to) {
            uint64_t base = (uint64_t)own * 64u;
            if (base < end) {
                const uint32_t leader = (uint32_t)__ffsll((long long)need) - 1u;
                uint32_t claim = 0;
                if (lane == leader) claim = atomicAdd(next, 1u);
                claim = __builtin_amdgcn_readlane(claim, leader);
                base += ((uint64_t)claim * regions + region) * 64u;
            }
            if (base >= end) {
                empty = true;
                return false;
            }
            at = (uint32_t)base;
            to = min(at + 64u, end);
        }
        const uint32_t mine = at + (uint32_t)__popcll(need & ((1ull << lane) - 1ull));
        const bool got = want && mine < to;
        if (got) t = mine;
        at = min(at + (uint32_t)__popcll(need), to);
        return got;
    }
};

// ---------------------------------------------------------- emission --
// launchRayGenEmitterKernel (PrimalKernels.cpp:13-62)
__global__ __launch_bounds__(kTile) void k_emit(DevScene S, DevState* st, uint32_t P, float invEmitted, RayQueue out,
                                                uint32_t outCap, TileStates ts) {
    const uint32_t tile = tileTicket(&st->ticket);
    if (tile * kTile >= P) {
        if (P == 0u) st->extTotal = 0u;
        return;
    }
    const uint32_t i = tile * kTile + threadIdx.x;
    F3 pos, dir, power;
    bool ok = false;
    if (i < P) {
        Rng rng(perItemSeed(st->number, i));
        ok = sampleLight(S, rng, pos, dir, power);
    }
    const TileOffset at = tileOffsets(ts, tile, ok, false);
    if (ok && at.a < outCap) {
        const F3 T = (power * (float)S.nLights) * invEmitted;
        out.o[at.a] = f4(pos, u2f(kInvalid));
        out.d[at.a] = f4(dir, u2f(0u));
        out.T[at.a] = f4(T, 0.0f);
    }
    if (threadIdx.x == 0 && tile == (P - 1u) / kTile) st->extTotal = min(at.endA, outCap);
}

// ---------------------------------------------------- photon bounce --
// Closest hits of a queue's rays, on a persistent grid.
struct QueueHits {
    float4* pos;     // hit point, instance (bits; kInvalid: miss)
    uint32_t* prim;  // primitive
    __device__ __forceinline__ Hit load(uint32_t i) const {
        const float4 p = pos[i];
        return Hit{ld3(p), f2u(p.w), prim[i]};
    }
};

template <bool kCount, bool kGroups>
struct QueueJob {
    static constexpr bool kGoesOn = false;
    const RayQueue& in;
    const HitArrays& hits;
    const TraceParams& tp;
    QueueCursor queue;  // of queue indices, or of places of the view groups
    uint32_t i = 0;
    Work w{};

    __device__ __forceinline__ bool drained() const { return queue.empty; }
    __device__ __forceinline__ bool fetch(bool idle, F3& o, F3& d) {
        uint32_t t;
        if (!queue.take(idle, t)) return false;
        i = t;
        if (kGroups && tp.groups) {
            // Place t -> (view group, segment, rank) -> queue index.
            uint32_t lo = 0, hi = tp.nGroups;  // last group whose first place <= t
            while (hi - lo > 1u) {
                const uint32_t mid = (lo + hi) >> 1;
                if (tp.groups[mid].z <= t)
                    lo = mid;
                else
                    hi = mid;
            }
            const uint4 gr = tp.groups[lo];
            const uint32_t local = t - gr.z;
            if (t < gr.z || local >= gr.y * gr.w) return false;
            const uint32_t s = tp.groupSegs[gr.x + local % gr.y], r = local / gr.y;
            if (r >= tp.segEnd[s] - tp.segFirst[s]) return false;
            i = tp.segFirst[s] + r;
        }
        o = ld3(in.o[i]);
        d = ld3(in.d[i]);
        return true;
    }
    __device__ __forceinline__ bool finish(bool done, const Hit& h, const Work& wl, F3&, F3&) {
        if (!done) return false;
        if (kCount) addWork(w, wl);
        hits.pos[i] = f4(h.pos, u2f(h.inst));
        hits.prim[i] = h.prim;
        return false;
    }
};

// What a hit makes of a photon or an adjoint ray is left to the shade kernels,
// one full wave after the other: at the end of the traversal it ran on half
// empty waves, its registers spilled and kept the trace at 4 waves per SIMD.
// The trace waits for its nodes: 5 waves (87 VGPRs, no spill) against 4 take
// 4 % off the rays of 1M surfels and nothing off those of 100k.  Together with
// the compaction in the shade kernels: backward pass of 800x800 rays on 1M
// surfels 26.0 -> 21.2 ms, step of a 4k scene 2.05 -> 1.82 ms.
template <bool kCount, bool kTopLds, bool kAdjoint>
__device__ __forceinline__ void queueTrace(const DevScene& S, DevState* st, const RayQueue& in, const HitArrays& hits,
                                           const TraceParams& tp) {
    extern __shared__ uint2 s_stack[];
    __shared__ TopLds sTop;
    if (kTopLds) loadTopLds(S, sTop);
    const LaneStack stk = walkStack(s_stack, S.stackDepth, tp.spill, tp.inLds);
    const uint32_t n = st->qCount;
    uint32_t end = n;
    if (kAdjoint && tp.groups) {
        const uint4 last = tp.nGroups ? tp.groups[tp.nGroups - 1u] : make_uint4(0u, 0u, 0u, 0u);
        end = last.z + last.y * last.w;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0)
        atomicAdd(kAdjoint ? &st->adjointQ : &st->photonQ, (unsigned long long)n);
    QueueJob<kCount, kAdjoint> job{in, hits, tp, QueueCursor(st->traceNext, end)};
    if (kTopLds)
        traceWave<kCount>(S, sTop, stk, job);
    else
        traceWave<kCount>(S, TopGlobal{S.tlas, S.inst}, stk, job);
    if (kCount) flushWork(job.w, st, kAdjoint ? kWorkAdjoint : kWorkPhoton);
}

template <bool kCount, bool kTopLds>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(5))) void k_photon_trace(
    DevScene S, DevState* st, RayQueue in, HitArrays hits, TraceParams tp) {
    queueTrace<kCount, kTopLds, false>(S, st, in, hits, tp);
}
template <bool kCount, bool kTopLds>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(5))) void k_adj_trace(
    DevScene S, DevState* st, RayQueue in, HitArrays hits, TraceParams tp) {
    queueTrace<kCount, kTopLds, true>(S, st, in, hits, tp);
}

// launchIntersectKernel (PrimalKernels.cpp:65-321) for one queue: what the hit
// of ray i deposits and the ray that goes on, written in queue order.
__global__ __launch_bounds__(kTile) void k_photon_shade(DevScene S, DevState* st, RayQueue in, HitArrays hitArrays,
                                                        RayQueue out, uint32_t outCap, PhotonArrays map,
                                                        PhotonArrays staged, TraceParams tp, Reservoir rs,
                                                        TileStates ts) {
    const uint32_t n = st->qCount;
    const uint32_t tile = tileTicket(&st->ticket);
    if (tile * kTile >= n) {
        if (n == 0u && tile == 0u && threadIdx.x == 0) st->extTotal = st->depTotal = 0u;
        return;
    }
    const QueueHits hits{hitArrays.pos, hitArrays.prim};
    const uint32_t i = tile * kTile + threadIdx.x;
    const bool resv = st->resv != 0u;
    bool ef = false, df = false;
    F3 no = mk3(0, 0, 0), nT = mk3(0, 0, 0), ndir = mk3(0, 0, 0);
    float4 depPos, depDir;
    float depZ = 0.0f;
    uint32_t bounce = 0;
    if (i < n) {
        Rng rng(perItemSeed(st->number, i));
        // depositPhotonSurface past capacity (KernelHelpers.h:1705-1718): the
        // attempt index comes from the probe pass; accept with probability
        // cap / (attempt + 1), then pick the slot (two draws of this item).
        auto reservoirDraws = [&]() {
            if (!resv) return;
            const uint32_t a = rs.attempt[i];
            uint32_t sl = kNoSlot;
            if (a >= rs.cap) {
                const float u = rng.nextFloat();
                const float accept = (float)rs.cap / (float)(a + 1u);
                if (u < accept) sl = rng.nextUint() % rs.cap;
            }
            rs.slot[i] = sl;
            if (sl != kNoSlot) {
                staged.posPow[i] = depPos;
                staged.dirPow[i] = depDir;
                staged.powZ[i] = depZ;
            }
        };
        if (resv) rs.slot[i] = kNoSlot;
        const float4 d4 = in.d[i];
        const F3 d = ld3(d4), T = ld3(in.T[i]);
        bounce = f2u(d4.w);
        const Hit h = hits.load(i);
        if (h.inst != kInvalid) {
            const DevInstance& I = S.inst[h.inst];
            ndir = d;
            bool spawn = false;
            if (I.type == kGeoMesh) {
                const F3 ng = hitNormal(S, h);
                df = true;
                depPos = f4(h.pos, T.x);
                depDir = f4(d, T.y);
                depZ = T.z;
                reservoirDraws();
                const DevMaterial m = S.mats[I.material];
                float pdf;
                sampleCosine(rng, ng, ndir, pdf);
                no = h.pos + ng * 1e-6f;
                nT = T * mk3(m.r, m.g, m.b);
                spawn = true;
            } else {
                const float u = rng.nextFloat();
                const SurfelShade sh = S.shade[h.prim];
                const float hAlpha = surfelAlpha(S.geo[h.prim], h.pos);
                if (u < tp.qNull) {
                    const float att = 1.0f - hAlpha * sh.opacity;
                    const float wn = att / tp.qNull;
                    no = h.pos + d * 1e-5f;
                    nT = T * wn;
                    spawn = true;
                } else if (u < tp.qNull + tp.qReflect) {
                    const F3 nc = mk3(sh.nsx, sh.nsy, sh.nsz);
                    const float sc = dot(nc, -d);
                    const int sign = sc >= 0.0f ? 1 : -1;
                    const F3 on = (float)sign * nc;
                    const F3 flux = divs(T, tp.qReflect);
                    df = true;
                    depPos = f4(h.pos, flux.x);
                    depDir = f4(d, flux.y);
                    depZ = flux.z;
                    reservoirDraws();
                    float pdf;
                    sampleUniformHemi(rng, on, ndir, pdf);
                    const float cosT = fmaxf(0.0f, dot(ndir, on));
                    const F3 fs = (sh.alpha_r * mk3(sh.ar, sh.ag, sh.ab)) * kInvPi;
                    const float alpha = hAlpha * sh.opacity;
                    const F3 w = divs(((alpha / tp.qReflect) * fs) * cosT, pdf);
                    no = h.pos + on * 1e-5f;
                    nT = T * w;
                    spawn = true;
                } else if (u < tp.qNull + tp.qReflect + tp.qTransmit) {
                    const F3 nc = mk3(sh.nsx, sh.nsy, sh.nsz);
                    const float sc = dot(nc, -d);
                    const int sign = sc >= 0.0f ? 1 : -1;
                    const F3 on = (float)sign * nc;
                    float pdf;
                    sampleUniformHemi(rng, on, ndir, pdf);
                    const float cosT = fmaxf(0.0f, dot(ndir, on));
                    const F3 fs = (0.0f * mk3(sh.ar, sh.ag, sh.ab)) * kInvPi;  // alpha_t = 0
                    const float alpha = hAlpha * sh.opacity;
                    const F3 w = divs(((alpha / tp.qReflect) * fs) * cosT, pdf);
                    no = h.pos + (-on) * 1e-5f;
                    nT = T * w;
                    spawn = true;
                }
            }
            ef = spawn && russianRoulette(rng, bounce + 1, nT, tp.rrStart);
        }
    }
    const TileOffset at = tileOffsets(ts, tile, ef, df);
    if (ef && at.a < outCap) {
        out.o[at.a] = f4(no, in.o[i].w);
        out.d[at.a] = f4(ndir, u2f(bounce + 1));
        out.T[at.a] = f4(nT, 0.0f);
    }
    if (df) {
        const uint32_t j = st->photonCount + at.b;
        if (j < rs.cap) {
            map.posPow[j] = depPos;
            map.dirPow[j] = depDir;
            map.powZ[j] = depZ;
        }
    }
    if (threadIdx.x == 0 && tile == (n - 1u) / kTile) {
        st->extTotal = min(at.endA, outCap);
        st->depTotal = at.endB;
    }
}

// Which items of a reservoir bounce deposit (the hit and the first draw of
// k_photon_shade), so that every deposit learns its attempt index in queue order
// before its random stream is used.
__global__ __launch_bounds__(256) void k_photon_probe(DevScene S, const DevState* st, HitArrays hitArrays,
                                                      uint8_t* depFlags, TraceParams tp) {
    if (!st->resv) return;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= st->qCount) return;
    const Hit h = QueueHits{hitArrays.pos, hitArrays.prim}.load(i);
    uint8_t df = 0;
    if (h.inst != kInvalid) {
        if (S.inst[h.inst].type == kGeoMesh) {
            df = 1;
        } else {
            Rng rng(perItemSeed(st->number, i));
            const float u = rng.nextFloat();
            df = (u >= tp.qNull && u < tp.qNull + tp.qReflect) ? 1 : 0;
        }
    }
    depFlags[i] = df;
}

// attempt[i] = photonCount + rank of item i among the depositing items.
__global__ __launch_bounds__(kScanThreads) void k_resv_rank(const uint8_t* flags, const DevState* st,
                                                            const uint32_t* tiles, uint32_t* attempt) {
    if (!st->resv) return;
    const uint32_t n = st->qCount;
    const uint32_t first = blockIdx.x * kTile + threadIdx.x * kTileSpan;
    uint8_t f[kTileSpan];
    uint32_t s = 0;
#pragma unroll
    for (uint32_t k = 0; k < kTileSpan; ++k) {
        f[k] = (first + k < n) ? flags[first + k] : 0;
        s += f[k];
    }
    uint32_t total;
    uint32_t off = blockExclusiveScan(s, total) + tiles[blockIdx.x] + st->photonCount;
#pragma unroll
    for (uint32_t k = 0; k < kTileSpan; ++k) {
        if (f[k]) attempt[first + k] = off++;
    }
}

__global__ __launch_bounds__(256) void k_resv_claim(const DevState* st, Reservoir rs) {
    if (!st->resv) return;
    const uint32_t n = st->qCount;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t sl = rs.slot[i];
    if (sl != kNoSlot) atomicMax(&rs.owner[sl], rs.attempt[i]);
}

__global__ __launch_bounds__(256) void k_resv_write(const DevState* st, Reservoir rs, PhotonArrays dep,
                                                    PhotonArrays raw) {
    if (!st->resv) return;
    const uint32_t n = st->qCount;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t sl = rs.slot[i];
    if (sl == kNoSlot || rs.owner[sl] != rs.attempt[i]) return;
    raw.posPow[sl] = dep.posPow[i];
    raw.dirPow[sl] = dep.dirPow[i];
    raw.powZ[sl] = dep.powZ[i];
}

// ------------------------------------------- ranks of a full map's deposits --
__global__ __launch_bounds__(kScanThreads) void k_tile_count(const uint8_t* flags, const uint32_t* count,
                                                             uint32_t maxItems, uint32_t* tiles) {
    const uint32_t n = loadCount(count, maxItems);
    const uint32_t base = blockIdx.x * kTile + threadIdx.x * kTileSpan;
    uint32_t s = 0;
#pragma unroll
    for (uint32_t k = 0; k < kTileSpan; ++k)
        if (base + k < n) s += flags[base + k];
    uint32_t total;
    blockExclusiveScan(s, total);
    if (threadIdx.x == 0) tiles[blockIdx.x] = total;
}

// Exclusive scan of the tile sums (one workgroup).
__global__ __launch_bounds__(1024) void k_tile_scan(uint32_t* tiles, const uint32_t* count, uint32_t maxItems) {
    __shared__ uint32_t sums[1024 / 64 + 1];
    const uint32_t numTiles = ceilDiv(loadCount(count, maxItems), kTile);
    uint32_t carry = 0;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    for (uint32_t base = 0; base < numTiles; base += 1024) {
        const uint32_t idx = base + threadIdx.x;
        const uint32_t v = idx < numTiles ? tiles[idx] : 0u;
        uint32_t x = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (lane >= (uint32_t)o) x += y;
        }
        if (lane == 63u) sums[wave] = x;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t s = 0;
            for (uint32_t w = 0; w < 1024 / 64; ++w) {
                const uint32_t t = sums[w];
                sums[w] = s;
                s += t;
            }
            sums[1024 / 64] = s;
        }
        __syncthreads();
        if (idx < numTiles) tiles[idx] = carry + x - v + sums[wave];
        carry += sums[1024 / 64];
        __syncthreads();
    }
}

// ------------------------------------------------------ photon grid --
// computePhotonCellIdsAndPermutation + countPhotonsPerCell
// (PrimalKernels.cpp:796-858).
__global__ __launch_bounds__(256) void k_cell_count(GridParams g, const DevState* st, uint32_t cap,
                                                    const float4* posPow, uint32_t* cellId, uint32_t* cellCount) {
    const uint32_t n = min(st->photonCount, cap);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 p = posPow[i];
    const F3 f = divv(mk3(p.x, p.y, p.z) - mk3(g.ox, g.oy, g.oz), mk3(g.cell, g.cell, g.cell));
    const int x = min(max((int)floorf(f.x), 0), g.rx - 1);
    const int y = min(max((int)floorf(f.y), 0), g.ry - 1);
    const int z = min(max((int)floorf(f.z), 0), g.rz - 1);
    const uint32_t c = (uint32_t)((z * g.ry + y) * g.rx + x);
    cellId[i] = c;
    atomicAdd(&cellCount[c], 1u);
}

// Exclusive scan of the counts of a grid's cells (or of an image's pixels) in
// one pass: the tiles' sums by look-back, 16 bytes per lane and load; out[n] =
// the sum of all.  in and out are the starts of their allocations.  Every count
// is read and every start written once; what bounds it is how fast the tiles'
// prefixes follow each other, so the tiles are large: 125M cells 0.60 ms at 8192
// items, 0.46 ms at 16384, 0.42 ms at 32768, where small grids (64k cells) take
// 8.1 instead of 6.8 us.  Scans of tiles, one workgroup's scan of their sums and
// its addition moved the starts three times: 1.36 ms, and 14.3 us.
__global__ __launch_bounds__(kScanBlock) void k_scan(const uint32_t* in, uint32_t* out, uint32_t n,
                                                     unsigned long long* scratch) {
    constexpr uint32_t kLoads = kScanTile / (kScanBlock * 4u), kWaves = kScanBlock / 64u;
    constexpr uint32_t kPer = (kLoads * kWaves + 63u) / 64u;  // wave sums per lane of the wave that scans them
    __shared__ uint32_t sums[kLoads * kWaves];
    __shared__ uint32_t sBase;
    const uint32_t tile = tileTicket(reinterpret_cast<uint32_t*>(scratch));
    const uint32_t first = tile * kScanTile + threadIdx.x * 4u, lane = laneId(), wave = threadIdx.x >> 6;
    uint4 v[kLoads];
    uint32_t off[kLoads];
#pragma unroll
    for (uint32_t k = 0; k < kLoads; ++k) {
        const uint32_t i = first + k * (kScanBlock * 4u);
        if (wholeFour(i, n))
            v[k] = *reinterpret_cast<const uint4*>(in + i);
        else
            v[k] = make_uint4(i < n ? in[i] : 0u, i + 1u < n ? in[i + 1u] : 0u, i + 2u < n ? in[i + 2u] : 0u, 0u);
    }
#pragma unroll
    for (uint32_t k = 0; k < kLoads; ++k) {
        const uint32_t s = v[k].x + v[k].y + v[k].z + v[k].w;
        uint32_t t = s;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(t, o, 64);
            if (lane >= (uint32_t)o) t += y;
        }
        off[k] = t - s;
        if (lane == 63u) sums[k * kWaves + wave] = t;
    }
    __syncthreads();
    if (wave == 0) {
        uint32_t v[kPer], own = 0;
#pragma unroll
        for (uint32_t k = 0; k < kPer; ++k) {
            v[k] = lane * kPer + k < kLoads * kWaves ? sums[lane * kPer + k] : 0u;
            own += v[k];
        }
        uint32_t t = own;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(t, o, 64);
            if (lane >= (uint32_t)o) t += y;
        }
        uint32_t first = t - own;
#pragma unroll
        for (uint32_t k = 0; k < kPer; ++k) {
            if (lane * kPer + k < kLoads * kWaves) sums[lane * kPer + k] = first;
            first += v[k];
        }
        const uint32_t total = __shfl(t, 63, 64);
        const uint64_t before = lookBack(scratch + 1, tile, total);
        if (lane == 0) {
            sBase = (uint32_t)before;
            if (tile == (n - 1u) / kScanTile) out[n] = (uint32_t)before + total;
        }
    }
    __syncthreads();
    const uint32_t base = sBase;
#pragma unroll
    for (uint32_t k = 0; k < kLoads; ++k) {
        const uint32_t i = first + k * (kScanBlock * 4u);
        uint4 o;
        o.x = base + sums[k * kWaves + wave] + off[k];
        o.y = o.x + v[k].x;
        o.z = o.y + v[k].y;
        o.w = o.z + v[k].z;
        if (wholeFour(i, n)) {
            *reinterpret_cast<uint4*>(out + i) = o;
        } else {
            if (i < n) out[i] = o.x;
            if (i + 1u < n) out[i + 1u] = o.y;
            if (i + 2u < n) out[i + 2u] = o.z;
        }
    }
}

// scatterPhotonsIntoCells (PrimalKernels.cpp:861-893).  The decrement leaves
// cellCount zeroed for the next build.
__global__ __launch_bounds__(256) void k_cell_scatter(const DevState* st, uint32_t cap, const uint32_t* cellId,
                                                      const uint32_t* cellStart, uint32_t* cellCount,
                                                      uint32_t* sortedIdx) {
    const uint32_t n = min(st->photonCount, cap);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t c = cellId[i];
    const uint32_t slot = cellStart[c] + atomicSub(&cellCount[c], 1u) - 1u;
    if (slot < n) sortedIdx[slot] = i;
}

// Order each cell by deposit index: the reference's sequential scatter
// order, which makes every gather sum in the same order.  A wave takes 64
// consecutive cells and sorts each one of up to 64 photons together: lane j
// holds photon j of the cell and its place is the number of smaller indices
// (indices are distinct).  Larger cells go to a list for k_cell_sort_big.
constexpr uint32_t kWaveCell = 64;
constexpr uint32_t kBlockCell = 4096;

__global__ __launch_bounds__(256) void k_cell_sort(uint32_t total, const uint32_t* cellStart, uint32_t* sortedIdx,
                                                   DevState* st, uint32_t* bigList) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t lane = laneId();
    uint32_t a = 0, n = 0;
    if (c < total) {
        a = cellStart[c];
        n = cellStart[c + 1] - a;
    }
    const unsigned long long big = __ballot(n > kWaveCell);
    if (big) {
        const uint32_t leader = (uint32_t)__ffsll((long long)big) - 1u;
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(&st->bigCells, (uint32_t)__popcll(big));
        base = __shfl(base, (int)leader, 64);
        if (n > kWaveCell) bigList[base + (uint32_t)__popcll(big & ((1ull << lane) - 1ull))] = c;
    }
    unsigned long long todo = __ballot(n >= 2u && n <= kWaveCell);
    while (todo) {
        const uint32_t j = (uint32_t)__ffsll((long long)todo) - 1u;
        todo &= todo - 1ull;
        const uint32_t ca = __shfl(a, (int)j, 64), cn = __shfl(n, (int)j, 64);
        const uint32_t x = lane < cn ? sortedIdx[ca + lane] : 0xFFFFFFFFu;
        uint32_t r = 0;
        for (uint32_t m = 0; m < cn; ++m) r += __shfl(x, (int)m, 64) < x ? 1u : 0u;
        if (lane < cn) sortedIdx[ca + r] = x;
    }
}

// Cells of more than 64 photons, one workgroup each: the cell in LDS, each
// photon's place = the number of smaller indices.  A cell beyond the LDS
// tile (more than 4096 photons, which clustered scenes of millions of
// photons do not reach) is sorted by one thread.
__global__ __launch_bounds__(256) void k_cell_sort_big(const DevState* st, const uint32_t* bigList,
                                                       const uint32_t* cellStart, uint32_t* sortedIdx) {
    __shared__ uint32_t v[kBlockCell];
    const uint32_t nb = st->bigCells;
    for (uint32_t q = blockIdx.x; q < nb; q += gridDim.x) {
        const uint32_t c = bigList[q];
        const uint32_t a = cellStart[c], n = cellStart[c + 1] - a;
        if (n <= kBlockCell) {
            for (uint32_t j = threadIdx.x; j < n; j += blockDim.x) v[j] = sortedIdx[a + j];
            __syncthreads();
            for (uint32_t j = threadIdx.x; j < n; j += blockDim.x) {
                const uint32_t x = v[j];
                uint32_t r = 0;
                for (uint32_t m = 0; m < n; ++m) r += v[m] < x ? 1u : 0u;
                sortedIdx[a + r] = x;
            }
            __syncthreads();
        } else if (threadIdx.x == 0) {
            for (uint32_t j = a + 1; j < a + n; ++j) {
                const uint32_t x = sortedIdx[j];
                uint32_t k = j;
                while (k > a && sortedIdx[k - 1] > x) {
                    sortedIdx[k] = sortedIdx[k - 1];
                    --k;
                }
                sortedIdx[k] = x;
            }
        }
    }
}

// The gather's copy: photons in cell order, their power times 1 / (pi r^2),
// the factor that every gather applies to it.
__global__ __launch_bounds__(256) void k_cell_payload(const DevState* st, uint32_t cap, const uint32_t* sortedIdx,
                                                      PhotonArrays raw, PhotonArrays sorted, float radius) {
    const uint32_t n = min(st->photonCount, cap);
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const uint32_t k = sortedIdx[j];
    const float invArea = 1.0f / (kPi * (radius * radius));
    float4 p = raw.posPow[k], d = raw.dirPow[k];
    p.w *= invArea;
    d.w *= invArea;
    sorted.posPow[j] = p;
    sorted.dirPow[j] = d;
    sorted.powZ[j] = raw.powZ[k] * invArea;
}

// ---------------------------------------------------- camera gather --
// launchCameraGatherKernel (PrimalKernels.cpp:500-653), split in stages so
// that the irradiance gathers, which dominate the pass, run in grid-cell
// order instead of pixel order:
//
//   k_cam_init      primary ray of every pixel (the reference's jitter);
//   k_cam_trace     persistent lanes walk each pixel's layers (closest-hit
//                   queries only) and append the hit of every layer, in layer
//                   order within the pixel.  Where a layer's ray starts does
//                   not depend on what the hits weigh, so the walk reads no
//                   shading record and evaluates no alpha;
//   k_entry_key     entry -> place in its pixel's layer list, and a
//                   counting sort of the gather entries by photon-grid cell;
//   k_entry_gather  one irradiance gather per entry, neighbouring lanes on
//                   neighbouring points (shared photon rows, similar loops),
//                   with the hit's normal, colour factor k and alpha; E * k
//                   and alpha * opacity go to the entry's place in the layer
//                   list;
//   k_cam_composite per pixel over the layers in order, w = tr * alpha *
//                   opacity, C = C + w * (E * k), then the reference's
//                   framebuffer update.
//
// Every value is computed by the same expressions as in the reference's
// single loop, and the per-pixel sums run in layer order, so the image is
// bit-identical.  If the entry buffer fills, a pixel stops before the layer
// that did not fit and resumes from there in the next round.
enum : uint32_t { kPixActive = 0u, kPixFinished = 1u, kPixFlushed = 2u };
constexpr uint32_t kEntryMesh = 0x80000000u;

__global__ __launch_bounds__(256) void k_cam_init(DevCamera cam, const DevState* st, uint32_t pass, int decorrelate,
                                                  PixelArrays px) {
    const uint32_t npx = cam.W * cam.H;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npx) return;
    const uint32_t seed = decorrelate ? st->number + pass : st->number;
    Rng rng(perItemSeed(seed, i));
    const float jx = rng.nextFloat() - 0.5f;
    const float jy = rng.nextFloat() - 0.5f;
    F3 o, d;
    primaryRay(cam, (float)(i % cam.W), (float)(i / cam.W), jx, jy, o, d);
    px.ot[i] = f4(o, 1.0f);
    px.dl[i] = f4(d, 0.0f);
    px.cs[i] = make_float4(0.0f, 0.0f, 0.0f, u2f(kPixActive));
    px.cnt[i] = 0u;
}

// Slot -> pixel maps of the layer walk.  Pixels are handed out in 8x8 tiles
// (a wave's first rays are neighbours); the order does not change any
// pixel's result.  ImageMap: the tiles of one image.  BatchMap: a list of
// tiles of several images (views x passes).
struct ImageMap {
    uint32_t width, height, tilesX;
    __device__ __forceinline__ uint32_t slots() const { return tilesX * ((height + 7u) / 8u) * 64u; }
    __device__ __forceinline__ bool locate(uint32_t slot, uint32_t& p) const {
        const uint32_t tile = slot >> 6, within = slot & 63u;
        const uint32_t pxx = (tile % tilesX) * 8u + (within & 7u);
        const uint32_t pxy = (tile / tilesX) * 8u + (within >> 3);
        p = pxy * width + pxx;
        return pxx < width && pxy < height;
    }
};

// Segment and pixel of a slot of a batch (see BatchDesc::tiles); false if
// the pixel lies outside the image (right and bottom tile edges).
__device__ __forceinline__ bool batchSlot(const uint4* tiles, uint32_t slot, uint32_t& seg, uint32_t& pxx,
                                          uint32_t& pxy, const BatchSeg*& s, const BatchSeg* segs) {
    const uint4 e = tiles[slot >> 6];
    const uint32_t j = slot - (e.z << 6);
    const uint32_t q = j / e.w;
    seg = e.x + (j - q * e.w);
    s = segs + seg;
    const uint32_t tilesX = s->tilesX;
    pxx = (e.y % tilesX) * 8u + (q & 7u);
    pxy = (e.y / tilesX) * 8u + (q >> 3);
    return pxx < s->W && pxy < s->H;
}

struct BatchMap {
    const uint4* tiles;
    const BatchSeg* segs;
    const BatchHeader* hdr;
    __device__ __forceinline__ uint32_t slots() const { return hdr->nTiles * 64u; }
    __device__ __forceinline__ bool locate(uint32_t slot, uint32_t& p) const {
        uint32_t seg, pxx, pxy;
        const BatchSeg* s;
        if (!batchSlot(tiles, slot, seg, pxx, pxy, s, segs)) return false;
        p = s->slotBase + pxy * s->W + pxx;
        return true;
    }
};

// Slots a wave of the layer walk claims at a time from its region.
constexpr uint32_t kWalkUnit = 64;
// Entries a wave claims at a time, and the slot of an entry it left unused.
constexpr uint32_t kEntryClaim = 512;
constexpr uint32_t kNoSlotOfEntry = 0xFFFFFFFFu;

// The layers of a pixel, one closest-hit query each: a lane appends the entry
// of its hit and goes on behind it until its pixel ends, then draws another.
template <bool kCount, typename Map, typename Top>
struct CameraJob {
    static constexpr bool kGoesOn = true;
    const DevScene& S;
    const Top& top;
    DevState* st;
    const Map& map;
    const PixelArrays& px;
    const EntryArrays& ent;
    uint32_t cap;
    uint32_t* cursor;
    uint32_t tiles, region;
    uint32_t emptyRegions = 0;
    uint32_t chunkNext = 0, chunkEnd = 0;  // the wave's untaken slots
    bool begun = false;                    // the wave has taken its first unit
    bool exhausted = false;
    // Entries are claimed entClaim at a time: one claim per entry append made
    // every wave wait for an atomic on the one counter of the grid, and with
    // queries that end a few lanes at a time the walk took 58 ms that way
    // against 38 ms (1M surfels, 800x800, 16 shared-seed passes).  What a wave
    // has claimed and not used when it ends is marked as holes (leaveHoles).
    uint32_t entClaim;
    uint32_t entNext = 0, entEnd = 0;
    uint32_t layers = 0;  // of the wave
    uint32_t pixel = 0, r = 0;  // r: entries of the pixel this round
    Work w{};

    __device__ __forceinline__ bool drained() const { return exhausted; }

    __device__ __forceinline__ void leaveHoles() const {
        for (uint32_t e = entNext + laneId(); e < min(entEnd, cap); e += 64u)
            ent.qs[e] = make_uint2(kNoSlotOfEntry, 0u);
    }

    // Draws pixels for the idle lanes until each has one or the slots run out
    // (a lane that drew a finished pixel, or none, draws again).
    __device__ __forceinline__ bool fetch(bool idle, F3& o, F3& d) {
        const uint32_t lane = laneId();
        bool got = false;
        while (!exhausted) {
            const unsigned long long need = __ballot(idle && !got);
            if (!need) break;
            // The wave claims a whole 64-slot unit (a few pixels in all their
            // passes) of its region and keeps what its lanes have not taken
            // for its next draws: its lanes stay on neighbouring rays.
            // Claiming only what the lanes need interleaves the waves' draws
            // and scatters each wave over many pixels (the walk took 17 %
            // longer, 28 % with decorrelated passes).
            if (chunkNext >= chunkEnd) {
                // Slots [lo, hi) of the current region; cursor[region] counts
                // the slots claimed from it this round.
                const uint32_t lo = (uint32_t)(((uint64_t)region * tiles) / kTraceRegions) * 64u;
                const uint32_t hi = (uint32_t)(((uint64_t)(region + 1u) * tiles) / kTraceRegions) * 64u;
                // The first units are the waves' own by their place in the
                // grid; after them a region's counter is read before it is
                // advanced, as each wave finds all regions used up once
                // (QueueCursor has what claims cost; with the waves' first
                // entries given as well, 16 passes of 155x130 on 1.1k surfels
                // 580 -> 174 us, nothing at 800x800 on 1M surfels).
                const uint32_t waves = kTraceBlock / 64u;
                uint32_t base;
                if (!begun) {
                    begun = true;
                    base = lo + ((blockIdx.x / kTraceRegions) * waves + __builtin_amdgcn_readfirstlane(threadIdx.x / 64u)) *
                                    kWalkUnit;
                } else {
                    const uint32_t blocks = (gridDim.x + kTraceRegions - 1u - region) / kTraceRegions;
                    base = lo + blocks * waves * kWalkUnit;
                    if (base < hi)
                        base += __builtin_amdgcn_readfirstlane(
                            *reinterpret_cast<volatile const uint32_t*>(cursor + region * kCursorStride));
                    if (base < hi) {
                        const uint32_t leader = (uint32_t)__ffsll((long long)need) - 1u;
                        if (lane == leader) base = lo + blocks * waves * kWalkUnit + atomicAdd(cursor + region * kCursorStride, kWalkUnit);
                        base = __builtin_amdgcn_readlane(base, leader);
                    }
                }
                if (base >= hi) {
                    // Used up (it stays so): the next region, done after all.
                    if (++emptyRegions == kTraceRegions) exhausted = true;
                    region = (region + 1u) % kTraceRegions;
                    continue;
                }
                chunkNext = base;
                chunkEnd = min(base + kWalkUnit, hi);
                if (__builtin_amdgcn_readfirstlane(*reinterpret_cast<volatile const uint32_t*>(&st->overflow)) != 0u) {
                    exhausted = true;
                    break;
                }
            }
            if (idle && !got) {
                const uint32_t slot = chunkNext + (uint32_t)__popcll(need & ((1ull << lane) - 1ull));
                uint32_t p = 0;
                if (slot < chunkEnd && map.locate(slot, p) && f2u(px.cs[p].w) == kPixActive) {
                    pixel = p;
                    got = true;
                    o = ld3(px.ot[p]);
                    d = ld3(px.dl[p]);
                    r = 0;
                }
            }
            chunkNext = min(chunkNext + (uint32_t)__popcll(need), chunkEnd);
        }
        return got;
    }

    __device__ __forceinline__ bool finish(bool done, const Hit& h, const Work& wl, F3& o, F3& d) {
        const uint32_t lane = laneId();
        const bool want = done && h.inst != kInvalid;
        const bool mesh = want && top.inst[h.inst].type == kGeoMesh;
        // Append of the entries, in lane order: from the wave's claimed
        // range, then from a new one.
        const unsigned long long m = __ballot(want);
        uint32_t e = 0xFFFFFFFFu;
        if (m) {
            const uint32_t count = (uint32_t)__popcll(m), mine = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            const uint32_t left = entEnd - entNext, taken = min(count, left);
            e = entNext + mine;
            entNext += taken;
            if (taken < count) {
                const uint32_t leader = (uint32_t)__ffsll((long long)m) - 1u, claim = max(entClaim, count - taken);
                uint32_t base = 0;
                if (lane == leader) base = atomicAdd(&st->entries, claim);
                base = __builtin_amdgcn_readlane(base, leader);
                if (mine >= taken) e = base + (mine - taken);
                entNext = base + (count - taken);
                entEnd = base + claim;
            }
        }
        const bool full = want && e >= cap;
        bool more = false;
        layers += (uint32_t)__popcll(__ballot(done && !full));
        if (done) {
            if (full) {
                // No room: stop before this layer, resume next round.
                float* ot = reinterpret_cast<float*>(px.ot + pixel);
                ot[0] = o.x;
                ot[1] = o.y;
                ot[2] = o.z;
                st->overflow = 1u;
                px.cnt[pixel] = r;
            } else {
                if (kCount) addWork(w, wl);
                if (want) {
                    ent.qa[e] = f4(h.pos, u2f(h.inst));
                    ent.qb[e] = f4(d, u2f(h.prim));
                    ent.qs[e] = make_uint2(pixel, r | (mesh ? kEntryMesh : 0u));
                    ++r;
                }
                more = want && !mesh;
                if (more) {
                    o = h.pos + d * 1e-4f;
                } else {
                    px.cnt[pixel] = r;
                    px.cs[pixel].w = u2f(kPixFinished);
                }
            }
        }
        if (__any(full)) exhausted = true;
        return more;
    }
};

// Entries that a wave of the layer walk claims at a time: at most an eighth of
// the buffer is claimed ahead; 0 (below 64): what it appends.  Else every wave
// starts with kEntryOwn entries at its place in the grid.
constexpr uint32_t kEntryOwn = 64;
__host__ __device__ __forceinline__ uint32_t entryClaim(uint32_t cap, uint32_t waves) {
    const uint32_t a = cap / (8u * waves), share = a < kEntryClaim ? a : kEntryClaim;
    return share < kEntryOwn ? 0u : share;
}
// Start of a round of the layer walk.
__global__ void k_walk_begin(DevState* st, uint32_t* cursor, uint32_t entries) {
    if (threadIdx.x < kTraceRegions) cursor[threadIdx.x * kCursorStride] = 0u;
    if (threadIdx.x == 0) {
        st->entries = entries;
        st->overflow = 0u;
    }
}

template <bool kCount, typename Map, typename Top>
__device__ __forceinline__ void camTrace(const DevScene& S, const Top& top, DevState* st, const Map& map,
                                         const PixelArrays& px, const EntryArrays& ent, uint32_t cap, uint32_t* cursor,
                                         const LaneStack& stk) {
    CameraJob<kCount, Map, Top> job{S, top, st, map, px, ent, cap, cursor, map.slots() >> 6, blockIdx.x % kTraceRegions};
    const uint32_t waves = gridDim.x * (kTraceBlock / 64u);
    job.entClaim = entryClaim(cap, waves);
    if (job.entClaim) {
        job.entNext = (blockIdx.x * (kTraceBlock / 64u) + threadIdx.x / 64u) * kEntryOwn;
        job.entEnd = job.entNext + kEntryOwn;
    }
    traceWave<kCount>(S, top, stk, job);
    job.leaveHoles();
    if (laneId() == 0 && job.layers) atomicAdd(&st->gatherQ, (unsigned long long)job.layers);
    if (kCount) flushWork(job.w, st, kWorkGather);
}

// 5 waves per SIMD (96 VGPRs without spills since the walk shades nothing, and
// kWalkLdsEntries of its stack in LDS): 57.6 -> 50.6 ms against 4 with
// independent samples, 35.7 -> 33.4 ms shared (16 passes of 800x800, 1M
// surfels); 6 waves spill 11 registers and run the same.
template <bool kCount, typename Map, bool kTopLds>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(5))) void k_cam_trace(
    DevScene S, DevState* st, Map map, PixelArrays px, EntryArrays ent, uint32_t cap, uint32_t* cursor,
    uint2* spill, uint32_t inLds) {
    extern __shared__ uint2 s_stack[];
    __shared__ TopLds sTop;
    if (kTopLds) loadTopLds(S, sTop);
    const LaneStack stk = walkStack(s_stack, S.stackDepth, spill, inLds);
    if (kTopLds)
        camTrace<kCount>(S, sTop, st, map, px, ent, cap, cursor, stk);
    else
        camTrace<kCount>(S, TopGlobal{S.tlas, S.inst}, st, map, px, ent, cap, cursor, stk);
}

// The lanes of a wave that hold the same key, wherever they sit: the lowest
// of them (the group's head), their number and this lane's rank among them.
// One pass per distinct key of the wave; every lane of the wave calls it.
struct KeyGroup {
    uint32_t head, len, rank;
};
__device__ __forceinline__ KeyGroup keyGroup(uint32_t key) {
    const uint32_t lane = laneId();
    unsigned long long todo = __ballot(1);
    KeyGroup g{lane, 1u, 0u};
    while (todo) {
        const uint32_t leader = (uint32_t)__ffsll((long long)todo) - 1u;
        const uint32_t lk = __shfl(key, (int)leader, 64);
        const unsigned long long peers = __ballot(key == lk);
        if (key == lk) {
            g.head = leader;
            g.len = (uint32_t)__popcll(peers);
            g.rank = (uint32_t)__popcll(peers & ((1ull << lane) - 1ull));
        }
        todo &= ~peers;
    }
    return g;
}

constexpr uint32_t kNoCell = 0xFFFFFFFFu;


// Place of every entry in its slot's layer-ordered list; grid cell and
// per-cell count of the gather entries (the cell of worldToCellClamped,
// KernelHelpers.h:920-934).  An emitter gathers nothing: its contribution is
// written here.  Neighbouring entries come from neighbouring lanes of the
// layer walk, so a wave holds few distinct cells: one atomic per distinct cell
// of the wave.  The entry kernels stride over the entries with a bounded grid:
// the count is known only on the device and the capacity is far above it.  The
// loop is uniform over the block, so whole waves take part in the run
// detection.
__global__ __launch_bounds__(256) void k_entry_key(DevScene S, GridParams g, uint32_t shift, const DevState* st, uint32_t cap,
                                                   PixelArrays px, EntryArrays ent, uint32_t* cellCount) {
    const uint32_t n = min(st->entries, cap);
    for (uint32_t i0 = blockIdx.x * blockDim.x; i0 < n; i0 += gridDim.x * blockDim.x) {
        const uint32_t i = i0 + threadIdx.x;
        uint32_t c = kNoCell;
        if (i < n) {
            const uint2 s = ent.qs[i];
            if (s.x != kNoSlotOfEntry) {  // else claimed and not used by its wave
                const uint32_t pos = px.off[s.x] + (s.y & ~kEntryMesh);
                ent.pos[i] = pos;
                const float4 a = ent.qa[i];
                bool gather = true;
                if (s.y & kEntryMesh) {
                    const DevMaterial m = S.mats[S.inst[f2u(a.w)].material];
                    if (m.power > 0.0f) {
                        ent.contrib[pos] = f4(vmin(mk3(m.r, m.g, m.b) * m.power, mk3(1.0f, 1.0f, 1.0f)), 1.0f);
                        gather = false;
                    }
                }
                if (gather) {
                    const F3 f = divv(mk3(a.x, a.y, a.z) - mk3(g.ox, g.oy, g.oz), mk3(g.cell, g.cell, g.cell));
                    const int x = min(max((int)floorf(f.x), 0), g.rx - 1);
                    const int y = min(max((int)floorf(f.y), 0), g.ry - 1);
                    const int z = min(max((int)floorf(f.z), 0), g.rz - 1);
                    c = (uint32_t)((z * g.ry + y) * g.rx + x) >> shift;
                }
            }
            ent.cell[i] = c;
        }
        const KeyGroup r = keyGroup(c);
        if (laneId() == r.head && c != kNoCell) atomicAdd(&cellCount[c], r.len);
    }
}

// Counting-sort scatter of the gather entries; leaves cellCount zeroed.  The
// lanes of a wave with the same cell take their places with one atomic.
__global__ __launch_bounds__(256) void k_entry_scatter(const DevState* st, uint32_t cap, const uint32_t* cellStart,
                                                       uint32_t* cellCount, EntryArrays ent) {
    const uint32_t n = min(st->entries, cap);
    for (uint32_t i0 = blockIdx.x * blockDim.x; i0 < n; i0 += gridDim.x * blockDim.x) {
        const uint32_t i = i0 + threadIdx.x;
        const uint32_t c = i < n ? ent.cell[i] : kNoCell;
        const KeyGroup r = keyGroup(c);
        const uint32_t lane = laneId();
        uint32_t base = 0;
        if (lane == r.head && c != kNoCell) base = cellStart[c] + atomicSub(&cellCount[c], r.len) - r.len;
        base = __shfl(base, (int)r.head, 64);
        if (c != kNoCell) ent.sorted[base + r.rank] = i;
    }
}

// One irradiance gather per entry in cell order, and what the hit makes of it:
// the radiance E * k and alpha * opacity (a mesh: 1) go to the entry's place in
// the slot's layer list (the products the reference's loop forms,
// PrimalKernels.cpp:583-585, :620, :626-628).
//
// Bound by vector instructions with shared seeds (issued in all of the cycles;
// 72 % with independent samples, 48 GB a launch at 0.39 of the HBM rate), then
// by the latency of the rows' dependent loads: 5 waves per SIMD (at most 96 VGPRs) instead of 4.  12.2 ->
// 8.8 ms and 18.1 -> 14.0 ms for the 102 M gathers of the 1M-surfel step: row
// bounds without IEEE divisions and square roots (GridRows; -1.0, -1.8 ms),
// photons two at a time instead of four (-1.6 ms), the fifth wave (-0.6 ms).
// The hit's alpha and shading (taken over from the layer walk) add 0.5 ms.
template <bool kCount>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void k_entry_gather(
    DevScene S, DevGrid G, DevState* st, const uint32_t* nGather, EntryArrays ent) {
    // One lane per entry (a one-shot grid over the capacity): gathers vary
    // in cost, and fresh waves take the place of finished ones, which a
    // strided loop would not.
    const uint32_t n = *nGather;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    Work w{};
    if (i < n) {
        const uint32_t e = ent.sorted[i];
        const float4 a = ent.qa[e], b = ent.qb[e];
        const uint32_t pos = ent.pos[e], prim = f2u(b.w);
        F3 nrm, k;
        float ae = 1.0f;
        if (ent.qs[e].y & kEntryMesh) {
            const Hit h{ld3(a), f2u(a.w), prim};
            nrm = hitNormal(S, h);
            const DevMaterial m = S.mats[S.inst[h.inst].material];
            k = mk3(m.r, m.g, m.b) * kInvPi;
        } else {
            const SurfelShade sh = S.shade[prim];
            nrm = mk3(sh.nsx, sh.nsy, sh.nsz);
            if (dot(nrm, -ld3(b)) < 0.0f) nrm = -nrm;
            k = (sh.alpha_r * mk3(sh.ar, sh.ag, sh.ab)) * kInvPi;
            ae = sh.opacity * surfelAlpha(S.geo[prim], ld3(a));
        }
        const F3 E = gatherIrradiance<kCount, true>(G, ld3(a), nrm, w);
        ent.contrib[pos] = f4(E * k, ae);
    }
    if (kCount) flushWork(w, st, kWorkGather);
}

// fb == nullptr (batches): a finished pixel keeps its colour in cs and the
// framebuffer update is left to k_batch_resolve.  nDev: device-side count.
// C = C + w * (E * k) over the pixel's layers in order, w = tr * alpha *
// opacity; a pixel that goes on in another round keeps its tr.
__global__ __launch_bounds__(256) void k_cam_composite(uint32_t npx, const uint32_t* nDev, PixelArrays px,
                                                       EntryArrays ent, float invSpp, float4* fb) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (nDev ? min(*nDev, npx) : npx)) return;
    const float4 cs = px.cs[p];
    const uint32_t status = f2u(cs.w);
    if (status == kPixFlushed) return;
    F3 C = mk3(cs.x, cs.y, cs.z);
    const uint32_t first = px.off[p], cnt = px.cnt[p];
    float tr = px.ot[p].w;
    for (uint32_t j = 0; j < cnt; ++j) {
        const float4 c = ent.contrib[first + j];
        const float w = tr * c.w;
        C = C + w * ld3(c);
        tr = tr * (1.0f - c.w);
    }
    // The next round's slot scan must see zero for every pixel it did not
    // touch, finished ones included.
    px.cnt[p] = 0u;
    if (status == kPixFinished) {
        if (fb) {
            const float4 f = fb[p];
            fb[p] = make_float4(C.x * invSpp + f.x, C.y * invSpp + f.y, C.z * invSpp + f.z, 1.0f * invSpp + f.w);
        }
        px.cs[p] = make_float4(C.x, C.y, C.z, u2f(kPixFlushed));
    } else {
        px.cs[p] = make_float4(C.x, C.y, C.z, u2f(kPixActive));
        px.ot[p].w = tr;
    }
}

// Primary rays of a batch: one thread per tile pixel; the same jitter and
// ray as k_cam_init for (view, pass) with seed = view seed + pass.
__global__ __launch_bounds__(256) void k_batch_init(BatchDesc b, PixelArrays px) {
    const uint32_t t = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (t >= b.hdr->nTiles) return;
    uint32_t seg, pxx, pxy;
    const BatchSeg* sp;
    if (!batchSlot(b.tiles, t * 64u + (threadIdx.x & 63u), seg, pxx, pxy, sp, b.segs)) return;
    const BatchSeg s = *sp;
    const uint32_t pixel = pxy * s.W + pxx, slot = s.slotBase + pixel;
    Rng rng(perItemSeed(s.seed, pixel));
    const float jx = rng.nextFloat() - 0.5f;
    const float jy = rng.nextFloat() - 0.5f;
    F3 o, d;
    primaryRay(b.cams[s.view], (float)pxx, (float)pxy, jx, jy, o, d);
    px.ot[slot] = f4(o, 1.0f);
    px.dl[slot] = f4(d, 0.0f);
    px.cs[slot] = make_float4(0.0f, 0.0f, 0.0f, u2f(kPixActive));
    px.cnt[slot] = 0u;
}

// Framebuffer update of a batch, per view pixel over the view's passes in
// pass order: the sequence of k_cam_composite's updates.
__global__ __launch_bounds__(256) void k_batch_resolve(BatchDesc b, PixelArrays px, float4* fb) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= b.hdr->nResolve) return;
    uint32_t lo = 0, hi = b.hdr->nRuns - 1u;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1u) >> 1;
        if (b.runs[mid].resolveBase <= i)
            lo = mid;
        else
            hi = mid - 1u;
    }
    const BatchRun r = b.runs[lo];
    const uint32_t pixel = i - r.resolveBase;
    float4 f = fb[r.fbOffset + pixel];
    for (uint32_t k = 0; k < r.numSegs; ++k) {
        const float4 c = px.cs[b.segs[r.firstSeg + k].slotBase + pixel];
        f = make_float4(c.x * r.invSpp + f.x, c.y * r.invSpp + f.y, c.z * r.invSpp + f.z, 1.0f * r.invSpp + f.w);
    }
    fb[r.fbOffset + pixel] = f;
}

// launchPostProcessKernel (PostprocessKernel.cpp:11-106), float LDR output.
__global__ __launch_bounds__(256) void k_post(const float4* fb, float4* ldr, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float invGamma = 1.0f / 2.2f;
    const float4 v = fb[i];
    float c[3] = {v.x, v.y, v.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float x = c[k] * 1.0f;
        x = fmaxf(x, 0.0f);
        x = pow_r(x, invGamma);
        x = fminf(fmaxf(x, 0.0f), 1.0f);
        c[k] = x;
    }
    ldr[i] = make_float4(c[0], c[1], c[2], 1.0f);
}

// ---------------------------------------------------------- adjoint --
// launchRayGenAdjointKernel (AdjointKernels.cpp:15-84).  The adjoint seeds
// from PathTracerSettings::random.number (default 42, setting adjoint_seed);
// with adjoint_decorrelate the host passes adjoint_seed + sample instead.
__global__ __launch_bounds__(256) void k_adj_raygen(DevCamera cam, const float* dloss, RayQueue q,
                                                    PendingArrays pend, DevState* st, uint32_t seed) {
    const uint32_t npx = cam.W * cam.H;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) st->qCount = npx;
    if (i >= npx) return;
    Rng rng(perItemSeed((uint64_t)seed, i));
    const float jx = rng.nextFloat() - 0.5f;
    const float jy = rng.nextFloat() - 0.5f;
    F3 o, d;
    primaryRay(cam, (float)(i % cam.W), (float)(i / cam.W), jx, jy, o, d);
    q.o[i] = f4(o, u2f(i));
    q.d[i] = f4(d, u2f(0u));
    q.T[i] = make_float4(dloss[3 * (size_t)i], dloss[3 * (size_t)i + 1], dloss[3 * (size_t)i + 2], 0.0f);
    pend.p0[i] = make_float4(0.0f, 0.0f, 0.0f, u2f(kNone));
}

// Adjoint primary rays of a batch: one thread per tile pixel, the jitter and
// ray of k_adj_raygen for the pixel of its view; queue index = slot.
__global__ __launch_bounds__(256) void k_adj_raygen_batch(BatchDesc b, const float* dloss, RayQueue q,
                                                          PendingArrays pend, DevState* st, uint32_t* segFirst) {
    const uint32_t t = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (blockIdx.x == 0 && threadIdx.x == 0) st->qCount = b.hdr->nSlots;
    if (t >= b.hdr->nTiles) return;
    uint32_t seg, pxx, pxy;
    const BatchSeg* sp;
    if (!batchSlot(b.tiles, t * 64u + (threadIdx.x & 63u), seg, pxx, pxy, sp, b.segs)) return;
    const BatchSeg s = *sp;
    const uint32_t pixel = pxy * s.W + pxx, slot = s.slotBase + pixel;
    Rng rng(perItemSeed((uint64_t)s.seed, pixel));
    const float jx = rng.nextFloat() - 0.5f;
    const float jy = rng.nextFloat() - 0.5f;
    F3 o, d;
    primaryRay(b.cams[s.view], (float)pxx, (float)pxy, jx, jy, o, d);
    if (pixel == 0u) segFirst[seg] = slot;
    const size_t src = 3 * ((size_t)s.pixOffset + pixel);
    q.o[slot] = f4(o, u2f(slot));
    q.d[slot] = f4(d, u2f(0u));
    q.T[slot] = make_float4(dloss[src], dloss[src + 1], dloss[src + 2], u2f(seg));
    pend.p0[slot] = make_float4(0.0f, 0.0f, 0.0f, u2f(kNone));
}

// launchAdjointIntersectKernel (AdjointKernels.cpp:87-386) for one queue: the
// pending event that the hit of ray i completes, the event it makes and the ray
// that goes on, written in queue order; segNext gets the first place of every
// segment that goes on (a batch).
__global__ __launch_bounds__(kTile) void k_adj_shade(DevScene S, DevState* st, uint32_t bounceIndex, RayQueue in,
                                                     HitArrays hitArrays, RayQueue out, uint32_t outCap,
                                                     EventArrays pool, uint32_t poolCap, PendingArrays pend,
                                                     uint32_t pendCap, TraceParams tp, uint32_t* segNext,
                                                     TileStates ts) {
    const uint32_t n = st->qCount;
    const uint32_t tile = tileTicket(&st->ticket);
    if (tile * kTile >= n) {
        if (n == 0u && tile == 0u && threadIdx.x == 0) st->extTotal = st->evTotal = 0u;
        return;
    }
    const QueueHits hits{hitArrays.pos, hitArrays.prim};
    const uint32_t i = tile * kTile + threadIdx.x;
    bool ef = false, vf = false;
    F3 no = mk3(0, 0, 0), nT = mk3(0, 0, 0), ndir = mk3(0, 0, 0);
    float4 e0, e1, e2, e3, e4, e5;
    uint32_t seg = 0, path = 0, bounce = 0;
    if (i < n) {
        const float4 o4 = in.o[i], d4 = in.d[i], T4 = in.T[i];
        const Hit h = hits.load(i);
        seg = f2u(T4.w);
        const uint32_t rank = tp.segFirst ? i - tp.segFirst[seg] : i;
        const float invS = tp.segs ? tp.segs[seg].invSpp : tp.invSpp;
        Rng rng(perItemSeed((uint64_t)(tp.segs ? tp.segs[seg].seed : tp.seed), rank));
        const F3 o = ld3(o4), d = ld3(d4), T = ld3(T4);
        path = f2u(o4.w);
        bounce = f2u(d4.w);
        const uint32_t dpx = !tp.debug ? 0u
                             : tp.segs ? tp.segs[seg].pixOffset + (path - tp.segs[seg].slotBase)
                                       : tp.debugBase + path;
        if (h.inst != kInvalid) {
            const DevInstance& I = S.inst[h.inst];
            const bool cloud = I.type == kGeoCloud;
            const float hAlpha = cloud ? surfelAlpha(S.geo[h.prim], h.pos) : 0.0f;
            F3 on, ng = mk3(0, 0, 0), dir;
            float pdf;
            SurfelShade sh{};
            if (!cloud) {
                ng = hitNormal(S, h);
                sampleCosine(rng, ng, dir, pdf);
                on = ng;
            } else {
                sh = S.shade[h.prim];
                const F3 nc = mk3(sh.nsx, sh.nsy, sh.nsz);
                const float sc = dot(nc, -d);
                const int sign = sc >= 0.0f ? 1 : -1;
                on = (float)sign * nc;
                sampleUniformHemi(rng, on, dir, pdf);
            }
            // Complete the pending interaction with this hit as its endpoint.
            if (path < pendCap) {
                const float4 p0 = pend.p0[path];
                const uint32_t kind = f2u(p0.w);
                const bool reflectDone = kind == kReflectS && cloud;
                const bool nullDone = kind == kNullT;
                if (reflectDone || nullDone) {
                    const float4 p1 = pend.p1[path];
                    const uint2 p2 = pend.p2[path];
                    const F3 Tp = ld3(p1) * (reflectDone ? tp.qReflect : tp.qNull);
                    const float endCos = fmaxf(0.0f, dot(dir, on));
                    e0 = f4(h.pos, u2f(kind));
                    if (reflectDone) {
                        e1 = f4(on, u2f(h.prim));
                        e2 = f4(Tp, hAlpha);
                        e3 = make_float4(u2f(S.inst[p2.y].material), pdf, endCos, invS);
                        if (tp.fullGradients || tp.debug) {  // this ray hit the endpoint surfel
                            e4 = f4(o, 0.0f);
                            e5 = f4(d, u2f(dpx));
                        }
                    } else {
                        e1 = f4(on, u2f(p2.x));
                        e2 = f4(Tp, p1.w);
                        e3 = make_float4(u2f(cloud ? kGeoCloud : kGeoMesh), u2f(cloud ? h.prim : I.material), endCos,
                                         invS);
                        if (tp.fullGradients) {  // the ray that crossed the pending surfel
                            e4 = pend.p3[path];
                            e5 = pend.p4[path];
                            e5.w = u2f(dpx);
                        } else if (tp.debug) {
                            e5 = make_float4(0.0f, 0.0f, 0.0f, u2f(dpx));
                        }
                    }
                    vf = true;
                    pend.p0[path] = make_float4(0.0f, 0.0f, 0.0f, u2f(kNone));
                }
            }
            bool spawn = false;
            uint32_t newKind = kNone;
            F3 pT = mk3(0, 0, 0);
            float pAlpha = 0.0f;
            uint2 pIds = make_uint2(kInvalid, kInvalid);
            ndir = dir;
            bool projection = false;
            if (!cloud) {
                const DevMaterial m = S.mats[I.material];
                const F3 base = mk3(m.r, m.g, m.b);
                no = h.pos + ng * 1e-6f;
                nT = T * base;
                spawn = true;
                newKind = kReflectS;
                pT = T * base;
                pIds = make_uint2(kInvalid, h.inst);
            } else {
                const float u = rng.nextFloat();
                if (u < tp.qNull) {
                    const float att = 1.0f - hAlpha * sh.opacity;
                    const float wn = att / tp.qNull;
                    no = h.pos + d * 1e-5f;
                    ndir = d;
                    nT = T * wn;
                    spawn = true;
                    newKind = kNullT;
                    pT = divs(T, tp.qNull);
                    pAlpha = hAlpha;
                    pIds = make_uint2(h.prim, kInvalid);
                } else if (u < tp.qNull + tp.qReflect) {
                    const F3 fs = (sh.alpha_r * mk3(sh.ar, sh.ag, sh.ab)) * kInvPi;
                    const float cosT = fmaxf(0.0f, dot(dir, on));
                    const float alpha = hAlpha * sh.opacity;
                    const F3 mult = divs((alpha / tp.qReflect) * (fs * cosT), pdf);
                    no = h.pos + on * 1e-5f;
                    nT = T * mult;
                    spawn = true;
                    projection = bounceIndex == 0;
                } else if (u < tp.qNull + tp.qReflect + tp.qTransmit) {
                    const float alpha = hAlpha * sh.opacity;
                    const float w = (alpha * 0.0f) / tp.qTransmit;  // alpha_t = 0
                    const F3 nc = mk3(sh.nsx, sh.nsy, sh.nsz);
                    const float sc = dot(nc, -d);
                    const int sign = sc >= 0.0f ? 1 : -1;
                    const F3 ot = (float)sign * nc;
                    float p2df;
                    sampleUniformHemi(rng, ot, ndir, p2df);
                    no = h.pos + (-ot) * 1e-5f;
                    nT = (T * w) * mk3(sh.ar, sh.ag, sh.ab);
                    spawn = true;
                }
            }
            if (spawn && russianRoulette(rng, bounce + 1, nT, tp.rrStart)) {
                if (newKind != kNone && path < pendCap) {
                    pend.p0[path] = f4(h.pos, u2f(newKind));
                    pend.p1[path] = f4(pT, pAlpha);
                    pend.p2[path] = pIds;
                    if (tp.fullGradients && newKind == kNullT) {
                        pend.p3[path] = f4(o, 0.0f);
                        pend.p4[path] = f4(d, 0.0f);
                    }
                }
                if (projection && path < pendCap) {
                    e0 = f4(h.pos, u2f(kProjection));
                    e1 = f4(on, u2f(h.prim));
                    e2 = f4(divs(T, tp.qReflect), hAlpha);
                    e3 = make_float4(0.0f, 0.0f, 0.0f, invS);
                    if (tp.fullGradients || tp.debug) {
                        e4 = f4(o, 0.0f);
                        e5 = f4(d, u2f(dpx));
                    }
                    vf = true;
                }
                ef = true;
            }
        }
    }
    const TileOffset at = tileOffsets(ts, tile, ef, vf);
    if (vf) {
        const uint32_t j = st->evPool + at.b;
        if (j < poolCap) {
            pool.e0[j] = e0;
            pool.e1[j] = e1;
            pool.e2[j] = e2;
            pool.e3[j] = e3;
            if (pool.e4) {
                pool.e4[j] = e4;
                pool.e5[j] = e5;
            }
        }
    }
    if (ef && at.a < outCap) {
        out.o[at.a] = f4(no, u2f(path));
        out.d[at.a] = f4(ndir, u2f(bounce + 1));
        out.T[at.a] = f4(nT, u2f(seg));
    }
    if (segNext) {
        // The wave's first ray of each segment; the value read first spares
        // the atomic of the waves behind the segment's start.
        const uint32_t lane = laneId();
        const unsigned long long m = __ballot(ef), before = m & ((1ull << lane) - 1ull);
        const uint32_t prev = before ? 63u - (uint32_t)__clzll((long long)before) : lane;
        const uint32_t prevSeg = __shfl(seg, (int)prev, 64);
        if (ef && (!before || prevSeg != seg) && at.a < segNext[seg]) atomicMin(segNext + seg, at.a);
    }
    if (threadIdx.x == 0 && tile == (n - 1u) / kTile) {
        st->extTotal = min(at.endA, outCap);
        st->evTotal = at.endB;
    }
}

// Counting sort of the pooled events by the photon-grid cell of their
// gather point, so the transport's irradiance gathers run in cell order.
// Cell of every pooled event and per-cell counts; neighbouring events come
// from neighbouring pixels, so equal cells arrive in runs: one atomic per
// run (the loop is uniform over the block, as in k_entry_key).
__global__ __launch_bounds__(256) void k_event_key(GridParams g, uint32_t shift, const DevState* st, uint32_t cap, EventArrays ev,
                                                   uint32_t* cell, uint32_t* cellCount) {
    const uint32_t n = min(st->evPool, cap);
    for (uint32_t i0 = blockIdx.x * blockDim.x; i0 < n; i0 += gridDim.x * blockDim.x) {
        const uint32_t i = i0 + threadIdx.x;
        uint32_t c = kNoCell;
        if (i < n) {
            const float4 a = ev.e0[i];
            const F3 f = divv(mk3(a.x, a.y, a.z) - mk3(g.ox, g.oy, g.oz), mk3(g.cell, g.cell, g.cell));
            const int x = min(max((int)floorf(f.x), 0), g.rx - 1);
            const int y = min(max((int)floorf(f.y), 0), g.ry - 1);
            const int z = min(max((int)floorf(f.z), 0), g.rz - 1);
            c = (uint32_t)((z * g.ry + y) * g.rx + x) >> shift;
            cell[i] = c;
        }
        const KeyGroup r = keyGroup(c);
        if (laneId() == r.head && c != kNoCell) atomicAdd(&cellCount[c], r.len);
    }
}

// Counting-sort scatter of the events (order within a cell: any; the
// transport's FP32 atomics sum in device order anyway); leaves cellCount
// zeroed.
__global__ __launch_bounds__(256) void k_event_scatter(const DevState* st, uint32_t cap, const uint32_t* cell,
                                                       const uint32_t* cellStart, uint32_t* cellCount,
                                                       uint32_t* sorted) {
    const uint32_t n = min(st->evPool, cap);
    for (uint32_t i0 = blockIdx.x * blockDim.x; i0 < n; i0 += gridDim.x * blockDim.x) {
        const uint32_t i = i0 + threadIdx.x;
        const uint32_t c = i < n ? cell[i] : kNoCell;
        const KeyGroup r = keyGroup(c);
        const uint32_t lane = laneId();
        uint32_t base = 0;
        if (lane == r.head && c != kNoCell) base = cellStart[c] + atomicSub(&cellCount[c], r.len) - r.len;
        base = __shfl(base, (int)r.head, 64);
        if (c != kNoCell) sorted[base + r.rank] = i;
    }
}

// Full-gradient contribution of one event: d(alpha_geom)/d(geometry) of
// surfel `prim` for the recorded ray, times eta * w (w = the event's weight
// sum_rgb(T * Lo) * invSpp with its sign).
// c[] = the surfel's 16 accumulator columns (position 0-2, t_u 3-5, t_v 6-8,
// scale 9-10, albedo 11-13, beta 15).
__device__ void addGeometryGradient(const DevScene& S, uint32_t prim, float4 ro, float4 rd, float w, float c[16]) {
    const DevInstance& I = S.inst[S.cloudInst];
    float hv[4];
    mulv4(I.w2o, ro.x, ro.y, ro.z, 1.0f, hv);
    const F3 oo = divs(mk3(hv[0], hv[1], hv[2]), hv[3]);
    mulv4(I.w2o, rd.x, rd.y, rd.z, 0.0f, hv);
    const F3 od = normalize(mk3(hv[0], hv[1], hv[2]));
    float g[12];
    if (!alphaGradient(S.geo[prim], oo, od, g)) return;
    const float f = S.shade[prim].opacity * w;
#pragma unroll
    for (int k = 0; k < 11; ++k) c[k] += g[k] * f;
    c[15] += g[11] * f;
}

// Sums v over each run of equal keys among consecutive lanes of the wave
// into the run's first lane (a segmented suffix reduction by shuffles);
// returns whether this lane heads its run.  Every lane of the wave calls it.
template <int kN>
__device__ __forceinline__ bool runReduce(uint32_t key, float (&v)[kN]) {
    const uint32_t lane = laneId();
    const uint32_t next = __shfl_down(key, 1, 64);
    const uint32_t prev = __shfl_up(key, 1, 64);
    const unsigned long long ends = __ballot(lane == 63u || next != key);
    const uint32_t end = lane + (uint32_t)__ffsll((long long)(ends >> lane)) - 1u;
#pragma unroll
    for (uint32_t o = 1; o < 64; o <<= 1) {
#pragma unroll
        for (int k = 0; k < kN; ++k) {
            const float t = __shfl_down(v[k], o, 64);
            if (lane + o <= end) v[k] += t;
        }
    }
    return lane == 0u || prev != key;
}

// launchAdjointTransportKernel (AdjointKernels.cpp:389-509), one lane per
// pooled event.  Each event carries the 1/spp of the view whose adjoint ray
// made it (e3.w).
template <bool kCount>
__global__ __launch_bounds__(256) void k_adj_transport(DevScene S, DevGrid G, DevState* st, uint32_t poolCap,
                                                       EventArrays ev, const uint32_t* sorted, float* grad,
                                                       float* full, float* debugImg) {
    const uint32_t n = min(st->evPool, poolCap);
    if (blockIdx.x * blockDim.x >= n) return;  // the grid covers the pool's capacity
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = i < n;
    Work w{};
    // Contributions of this lane's event: opacity in c[0], the full
    // gradient's columns in c[1 + column]; lanes of a wave that follow one
    // another with the same target surfel (events are cell-sorted, so runs
    // are common) add theirs up before one lane issues the atomics.
    float c[17];
#pragma unroll
    for (int k = 0; k < 17; ++k) c[k] = 0.0f;
    uint32_t target = 0xFFFFFFFFu;
    if (active) {
        const uint32_t j = sorted[i];
        const float4 e0 = ev.e0[j], e1 = ev.e1[j], e2 = ev.e2[j], e3 = ev.e3[j];
        const uint32_t kind = f2u(e0.w);
        target = f2u(e1.w);
        const float invSpp = e3.w;
        const F3 T = ld3(e2);
        const float a = e2.w;
        const F3 E = gatherIrradiance<kCount>(G, ld3(e0), ld3(e1), w);
        float val = 0.0f;
        if (kind == kProjection) {
            const SurfelShade sh = S.shade[target];
            const F3 fr = (sh.alpha_r * mk3(sh.ar, sh.ag, sh.ab)) * kInvPi;
            const F3 Lr = fr * E;
            const F3 g = (a * T) * Lr;
            val = fsum(g) * invSpp;
            if (full) {
                addGeometryGradient(S, target, ev.e4[j], ev.e5[j], fsum(T * Lr) * invSpp, c + 1);
                const F3 ga = ((a * sh.opacity * sh.alpha_r * kInvPi) * (T * E)) * invSpp;
                c[1 + 11] += ga.x;
                c[1 + 12] += ga.y;
                c[1 + 13] += ga.z;
            }
        } else if (kind == kNullT) {
            F3 base;
            float power;
            if (f2u(e3.x) == kGeoMesh) {
                const DevMaterial m = S.mats[f2u(e3.y)];
                base = mk3(m.r, m.g, m.b);
                power = m.power;
            } else {
                const SurfelShade es = S.shade[f2u(e3.y)];
                base = es.alpha_r * mk3(es.ar, es.ag, es.ab);
                power = 0.0f;
            }
            const F3 Lr = (E * base) * kInvPi;
            F3 Le = mk3(0, 0, 0);
            if (power > 0.0f && S.nLights > 0) Le = (base * (power / (kPi * S.lights[0].area))) * e3.z;
            const F3 Lo = Le + Lr;
            const F3 g = ((-a) * T) * Lo;
            val = fsum(g) * invSpp;
            if (full) addGeometryGradient(S, target, ev.e4[j], ev.e5[j], -(fsum(T * Lo) * invSpp), c + 1);
        } else if (kind == kReflectS) {
            const DevMaterial m = S.mats[f2u(e3.x)];
            const F3 Lo = (E * mk3(m.r, m.g, m.b)) * kInvPi;
            const F3 p = divs(T, e3.y);
            const F3 g = (p * Lo) * a;
            val = fsum(g) * invSpp;
            if (full) addGeometryGradient(S, target, ev.e4[j], ev.e5[j], fsum(p * Lo) * invSpp, c + 1);
        }
        c[0] = val;
        if (debugImg) {
            float* px = debugImg + 4 * (size_t)f2u(ev.e5[j].w);
            atomicAdd(px, val);
            atomicAdd(px + 1, val);
            atomicAdd(px + 2, val);
            __hip_atomic_store(px + 3, 1.0f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    bool head;
    if (full) {
        head = runReduce(target, c);
    } else {
        float v[1] = {c[0]};
        head = runReduce(target, v);
        c[0] = v[0];
    }
    if (head && target != 0xFFFFFFFFu) {
        atomicAdd(&grad[target], c[0]);
        if (full) {
            float* out = full + (size_t)target * 16;
#pragma unroll
            for (int k = 0; k < 16; ++k)
                if (k != 14 && c[1 + k] != 0.0f) atomicAdd(out + k, c[1 + k]);
        }
    }
    waveCount(active, &st->events);
    if (kCount) flushWork(w, st, kWorkAdjoint);
}

// ------------------------------------------------------ diagnostics --
// A caller's rays by the renderer's own traversal.  2M incoherent rays against
// 100k and 1M clustered surfels: 1.4 and 1.7 ms; one query per lane, run to the
// wave's longest: 2.5 and 3.1 ms by the binary tree, 2.9 and 3.3 ms by quad nodes.
struct ProbeJob {
    static constexpr bool kGoesOn = false;
    const DevScene& S;
    const float *org, *dir;
    int32_t *inst, *prim;
    float *t, *pos, *alpha;
    QueueCursor queue;
    size_t i = 0;

    __device__ __forceinline__ bool drained() const { return queue.empty; }
    __device__ __forceinline__ bool fetch(bool idle, F3& o, F3& d) {
        uint32_t k;
        if (!queue.take(idle, k)) return false;
        i = k;
        o = mk3(org[3 * i], org[3 * i + 1], org[3 * i + 2]);
        d = mk3(dir[3 * i], dir[3 * i + 1], dir[3 * i + 2]);
        return true;
    }
    __device__ __forceinline__ bool finish(bool done, const Hit& h, const Work&, F3& o, F3& d) {
        if (!done) return false;
        const bool hit = h.inst != kInvalid;
        const F3 x = hit ? h.pos : mk3(0, 0, 0);
        inst[i] = hit ? (int32_t)h.inst : -1;
        prim[i] = hit ? (int32_t)h.prim : -1;
        t[i] = hit ? dot(x - o, d) : 0.0f;
        pos[3 * i] = x.x;
        pos[3 * i + 1] = x.y;
        pos[3 * i + 2] = x.z;
        alpha[i] = hit && S.inst[h.inst].type == kGeoCloud ? surfelAlpha(S.geo[h.prim], x) : 0.0f;
        return false;
    }
};
__global__ __launch_bounds__(kTraceBlock) void k_trace_rays(DevScene S, DevState* st, uint32_t n, const float* o,
                                                            const float* d, int32_t* inst, int32_t* prim, float* t,
                                                            float* pos, float* alpha) {
    extern __shared__ uint2 s_stack[];
    ProbeJob job{S, o, d, inst, prim, t, pos, alpha, QueueCursor(st->traceNext, n)};
    traceWave<false>(S, TopGlobal{S.tlas, S.inst}, laneStack(s_stack, S.stackDepth), job);
}

// Full-gradient array (16 floats per surfel) into the ABI's arrays.
__global__ __launch_bounds__(256) void k_split_gradients(const float* full, uint32_t n, float* position,
                                                         float* tangentU, float* tangentV, float* scale,
                                                         float* albedo, float* beta) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float* g = full + (size_t)i * 16;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (position) position[3 * (size_t)i + k] = g[k];
        if (tangentU) tangentU[3 * (size_t)i + k] = g[3 + k];
        if (tangentV) tangentV[3 * (size_t)i + k] = g[6 + k];
        if (albedo) albedo[3 * (size_t)i + k] = g[11 + k];
    }
    if (scale) {
        scale[2 * (size_t)i] = g[9];
        scale[2 * (size_t)i + 1] = g[10];
    }
    if (beta) beta[i] = g[15];
}

// Opacity of every surfel from device memory (BVH order).
__global__ __launch_bounds__(256) void k_set_opacity(SurfelShade* shade, const float* opacity, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) shade[i].opacity = opacity[i];
}

// apply_point_optimization with the parameters already in device memory:
// each surfel's intersection and shading records from the same binary32
// expressions as the host's refreshSurfels (orthonormal frame of
// intersectSurfel, KernelHelpers.h:646-648; shading normal
// normalize(cross(t_u, t_v)), :497-501; 4 e^beta), so that both paths give
// identical records.  The values are written as given (no clamp or
// normalisation), as the reference's apply_point_optimization writes them
// (pale_bindings.cpp:853-1056); alpha_r is kept.  `raw` receives the
// parameters for the host mirror.
__global__ __launch_bounds__(256) void k_apply_points(SurfelGeo* geo, SurfelShade* shade, float* raw,
                                                      DevPointArrays a, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const F3 p = mk3(a.position[3 * i], a.position[3 * i + 1], a.position[3 * i + 2]);
    const F3 tu = mk3(a.tangent_u[3 * i], a.tangent_u[3 * i + 1], a.tangent_u[3 * i + 2]);
    const F3 tv = mk3(a.tangent_v[3 * i], a.tangent_v[3 * i + 1], a.tangent_v[3 * i + 2]);
    const float su = a.scale[2 * i], sv = a.scale[2 * i + 1];
    const F3 alb = mk3(a.albedo[3 * i], a.albedo[3 * i + 1], a.albedo[3 * i + 2]);
    const float op = a.opacity[i], beta = a.beta[i];
    const F3 u = normalize(tu);
    const F3 v = normalize(tv - u * dot(u, tv));
    const F3 nrm = normalize(cross(u, v));
    SurfelGeo g;
    g.px = p.x; g.py = p.y; g.pz = p.z; g.su = su;
    g.nx = nrm.x; g.ny = nrm.y; g.nz = nrm.z; g.sv = sv;
    g.tux = tu.x; g.tuy = tu.y; g.tuz = tu.z; g.e4b = 4.0f * exp_r(beta);
    g.tvx = tv.x; g.tvy = tv.y; g.tvz = tv.z; g.pad = 0.0f;
    geo[i] = g;
    const F3 ns = normalize(cross(tu, tv));
    SurfelShade h;
    h.nsx = ns.x; h.nsy = ns.y; h.nsz = ns.z; h.opacity = op;
    h.ar = alb.x; h.ag = alb.y; h.ab = alb.z; h.alpha_r = shade[i].alpha_r;
    shade[i] = h;
    float4* r = reinterpret_cast<float4*>(raw) + 4 * (size_t)i;
    r[0] = make_float4(p.x, p.y, p.z, tu.x);
    r[1] = make_float4(tu.y, tu.z, tv.x, tv.y);
    r[2] = make_float4(tv.z, su, sv, alb.x);
    r[3] = make_float4(alb.y, alb.z, op, beta);
}

// Irradiance estimate at given points (gatherDiffuseIrradianceAtPoint,
// KernelHelpers.h:990-1037) for tests of the gather on its own.
__global__ __launch_bounds__(256) void k_gather_points(DevGrid G, uint32_t n, const float* q, const float* nrm,
                                                       float* out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    Work w{};
    const F3 E = gatherIrradiance<false>(G, mk3(q[3 * i], q[3 * i + 1], q[3 * i + 2]),
                                         mk3(nrm[3 * i], nrm[3 * i + 1], nrm[3 * i + 2]), w);
    out[3 * i] = E.x;
    out[3 * i + 1] = E.y;
    out[3 * i + 2] = E.z;
}

// A node's quad node.  The children's own boxes are not stored: the traversal
// takes their entries from the union of their children's, so a node is written
// two levels deep only where those unions are the children's boxes (always,
// unless a box has NaN or no extent); otherwise, and where `levels` is 1, its two
// children take a slot each.
__global__ __launch_bounds__(256) void k_quad_nodes(const WideNode* nodes, QuadNode* quads, uint32_t first, uint32_t n,
                                                    uint32_t levels) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const WideNode w = nodes[first + i];
    struct Box {
        float b[6];  // min xyz, max xyz
    };
    const Box child[2] = {{{w.lminx, w.lminy, w.lminz, w.lmaxx, w.lmaxy, w.lmaxz}},
                          {{w.rminx, w.rminy, w.rminz, w.rmaxx, w.rmaxy, w.rmaxz}}};
    const uint32_t ref[2] = {w.left, w.right};
    Box box[4];
    uint32_t refs[4];
    bool whole = levels == 2u;
    for (int c = 0; c < 2; ++c) {
        box[2 * c] = box[2 * c + 1] = child[c];
        refs[2 * c] = ref[c];
        refs[2 * c + 1] = kInvalid;
        if (ref[c] & kLeafBit) continue;
        const WideNode g = nodes[ref[c]];
        const Box l = {{g.lminx, g.lminy, g.lminz, g.lmaxx, g.lmaxy, g.lmaxz}};
        const Box r = {{g.rminx, g.rminy, g.rminz, g.rmaxx, g.rmaxy, g.rmaxz}};
        for (int a = 0; a < 6; ++a) {
            const float u = a < 3 ? fminf(l.b[a], r.b[a]) : fmaxf(l.b[a], r.b[a]);
            whole = whole && u == child[c].b[a] && l.b[a] == l.b[a] && r.b[a] == r.b[a];
            if (a < 3) whole = whole && l.b[a] <= l.b[a + 3] && r.b[a] <= r.b[a + 3];
        }
        box[2 * c] = l;
        box[2 * c + 1] = r;
        refs[2 * c] = g.left;
        refs[2 * c + 1] = g.right;
    }
    QuadNode q;
    for (int k = 0; k < 4; ++k) {
        const Box& b = whole ? box[k] : child[k >> 1];
        q.mnx[k] = b.b[0];
        q.mny[k] = b.b[1];
        q.mnz[k] = b.b[2];
        q.mxx[k] = b.b[3];
        q.mxy[k] = b.b[4];
        q.mxz[k] = b.b[5];
        q.ref[k] = whole ? refs[k] : ((k & 1) ? kInvalid : ref[k >> 1]);
        q.pad[k] = 0u;
    }
    quads[first + i] = q;
}

// ------------------------------------------------------------ launchers --
static inline uint32_t blocks(uint32_t n, uint32_t b) { return ceilDiv(n, b); }
// Grid of the light per-item kernels (keys and scatters of the entry and
// event sorts) that stride over buffers whose count is known only on the
// device: 256 CUs x 32 workgroups of 256 lanes.
constexpr uint32_t kEntryBlocks = 8192;
static inline size_t stackBytes(const DevScene& S) { return (size_t)S.stackDepth * sizeof(uint2) * kTraceBlock; }

void launchFill(hipStream_t s, uint32_t* p, uint32_t n, uint32_t v) {
    if (n) k_fill<<<min(blocks(n, 256), 65535u), 256, 0, s>>>(p, n, v);
}
void launchFillF(hipStream_t s, float* p, uint32_t n, float v) {
    if (n) k_fillf<<<min(blocks(n, 256), 65535u), 256, 0, s>>>(p, n, v);
}
void launchIota(hipStream_t s, uint32_t* p, uint32_t n) {
    if (n) k_iota<<<min(blocks(n, 256), 65535u), 256, 0, s>>>(p, n);
}
static inline uint32_t tilesOf(uint32_t rays) { return blocks(rays, kTile); }
void launchPhotonNext(hipStream_t s, DevState* st, const uint32_t* table, uint32_t len, int bounce, uint32_t resvCap,
                      TileStates ts, uint32_t rays) {
    k_photon_next<<<1, 256, 0, s>>>(st, table, len, bounce, resvCap, ts, tilesOf(rays));
}
void launchBeginView(hipStream_t s, DevState* st, uint32_t number) { k_begin_view<<<1, 64, 0, s>>>(st, number); }
void launchEmit(hipStream_t s, const DevScene& S, DevState* st, uint32_t P, float invEmitted, RayQueue out,
                uint32_t outCap, TileStates ts) {
    k_emit<<<tilesOf(max(P, 1u)), kTile, 0, s>>>(S, st, P, invEmitted, out, outCap, ts);
}
// Persistent grid of a trace kernel: as many workgroups as fit on the device.
// Renderers on several host threads share the cache.
static uint32_t traceGrid(const void* kernel, size_t lds) {
    struct Entry {
        const void* kernel;
        size_t lds;
        int dev;
        uint32_t grid;
    };
    static std::mutex lock;
    static std::vector<Entry> cache;  // a few kernels, one LDS size per stack depth
    int dev = 0, cus = 0, perCu = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> guard(lock);
    for (const Entry& e : cache)
        if (e.kernel == kernel && e.lds == lds && e.dev == dev) return e.grid;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, kernel, kTraceBlock, lds);
    cache.push_back(Entry{kernel, lds, dev, (uint32_t)std::max(1, cus) * (uint32_t)std::max(1, perCu)});
    return cache.back().grid;
}
template <bool kCount, typename Map, bool kTopLds>
static uint32_t camTraceGrid(size_t lds) {
    return traceGrid(reinterpret_cast<const void*>(&k_cam_trace<kCount, Map, kTopLds>), lds);
}

uint32_t queueTraceLanes(const DevScene& S, uint32_t rays, uint32_t inLds) {
    const size_t lds = (size_t)min(S.stackDepth, inLds) * sizeof(uint2) * kTraceBlock;
    uint32_t grid = 0;
    const auto add = [&](auto k) { grid = std::max(grid, traceGrid(reinterpret_cast<const void*>(k), lds)); };
    add(&k_photon_trace<false, false>);
    add(&k_photon_trace<false, true>);
    add(&k_photon_trace<true, false>);
    add(&k_photon_trace<true, true>);
    add(&k_adj_trace<false, false>);
    add(&k_adj_trace<false, true>);
    add(&k_adj_trace<true, false>);
    add(&k_adj_trace<true, true>);
    return min(grid, blocks(rays, kTraceBlock)) * kTraceBlock;
}

void launchQueueTrace(hipStream_t s, const DevScene& S, DevState* st, uint32_t maxRays, RayQueue in, HitArrays hits,
                      TraceParams tp, bool adjoint, bool count) {
    if (!maxRays) return;
    using Kernel = void (*)(DevScene, DevState*, RayQueue, HitArrays, TraceParams);
    static constexpr Kernel kernels[2][2][2] = {
        {{&k_photon_trace<false, false>, &k_photon_trace<false, true>},
         {&k_photon_trace<true, false>, &k_photon_trace<true, true>}},
        {{&k_adj_trace<false, false>, &k_adj_trace<false, true>}, {&k_adj_trace<true, false>, &k_adj_trace<true, true>}}};
    const size_t lds = tp.spill ? (size_t)tp.inLds * sizeof(uint2) * kTraceBlock : stackBytes(S);
    const Kernel k = kernels[adjoint][count][topFitsLds(S)];
    const uint32_t g = min(traceGrid(reinterpret_cast<const void*>(k), lds), blocks(maxRays, kTraceBlock));
    k<<<g, kTraceBlock, lds, s>>>(S, st, in, hits, tp);
}

void launchPhotonShade(hipStream_t s, const DevScene& S, DevState* st, uint32_t maxRays, RayQueue in, HitArrays hits,
                       RayQueue out, uint32_t outCap, PhotonArrays map, PhotonArrays staged, TraceParams tp,
                       Reservoir rs, uint8_t* depFlags, uint32_t* tiles, TileStates ts) {
    if (!maxRays) return;
    if (rs.attempt) {
        // The map can fill during this render: which deposit, their ranks.
        const uint32_t* qCount =
            reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(st) + offsetof(DevState, qCount));
        const uint32_t nt = blocks(maxRays, kTile);
        k_photon_probe<<<blocks(maxRays, 256), 256, 0, s>>>(S, st, hits, depFlags, tp);
        k_tile_count<<<nt, kScanThreads, 0, s>>>(depFlags, qCount, maxRays, tiles);
        k_tile_scan<<<1, 1024, 0, s>>>(tiles, qCount, maxRays);
        k_resv_rank<<<nt, kScanThreads, 0, s>>>(depFlags, st, tiles, rs.attempt);
    }
    k_photon_shade<<<tilesOf(maxRays), kTile, 0, s>>>(S, st, in, hits, out, outCap, map, staged, tp, rs, ts);
    if (rs.attempt) {
        k_resv_claim<<<blocks(maxRays, 256), 256, 0, s>>>(st, rs);
        k_resv_write<<<blocks(maxRays, 256), 256, 0, s>>>(st, rs, staged, map);
    }
}

void launchExclusiveScan(hipStream_t s, const uint32_t* in, uint32_t* out, uint32_t n, unsigned long long* scratch) {
    if (!n) return;
    const uint32_t tiles = blocks(n, kScanTile);
    launchFill(s, reinterpret_cast<uint32_t*>(scratch), 2u * (tiles + 1u), 0u);
    k_scan<<<tiles, kScanBlock, 0, s>>>(in, out, n, scratch);
}
void launchBuildGrid(hipStream_t s, const GridParams& g, DevState* st, uint32_t cap, PhotonArrays raw,
                     PhotonArrays sorted, uint32_t* cellId, uint32_t* sortedIdx, uint32_t* cellCount,
                     uint32_t* cellStart, unsigned long long* scan, float radius) {
    const uint32_t pb = blocks(cap, 256);
    k_cell_count<<<pb, 256, 0, s>>>(g, st, cap, raw.posPow, cellId, cellCount);
    launchExclusiveScan(s, cellCount, cellStart, g.total, scan);
    k_cell_scatter<<<pb, 256, 0, s>>>(st, cap, cellId, cellStart, cellCount, sortedIdx);
    // cellId is free once the photons are scattered: it holds the list of
    // large cells.
    launchFill(s, reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(st) + offsetof(DevState, bigCells)), 1, 0u);
    k_cell_sort<<<blocks(g.total, 256), 256, 0, s>>>(g.total, cellStart, sortedIdx, st, cellId);
    k_cell_sort_big<<<min(pb, 2048u), 256, 0, s>>>(st, cellId, cellStart, sortedIdx);
    k_cell_payload<<<pb, 256, 0, s>>>(st, cap, sortedIdx, raw, sorted, radius);
}


void launchCamInit(hipStream_t s, const DevCamera& cam, const DevState* st, uint32_t pass, int decorrelate,
                   PixelArrays px) {
    const uint32_t npx = cam.W * cam.H;
    if (npx) k_cam_init<<<blocks(npx, 256), 256, 0, s>>>(cam, st, pass, decorrelate, px);
}

// LDS of one layer-walk workgroup: the in-LDS part of its lanes' stacks.
static size_t walkLdsBytes(const DevScene& S, const uint2* spill, uint32_t inLds) {
    return spill ? (size_t)inLds * sizeof(uint2) * kTraceBlock : stackBytes(S);
}

size_t walkSpillBytes(const DevScene& S, uint32_t inLds) {
    if (S.stackDepth <= inLds) return 0;
    const size_t lds = (size_t)inLds * sizeof(uint2) * kTraceBlock;
    const uint32_t grid =
        std::max(std::max(std::max(camTraceGrid<false, BatchMap, false>(lds), camTraceGrid<true, BatchMap, false>(lds)),
                          std::max(camTraceGrid<false, ImageMap, false>(lds), camTraceGrid<true, ImageMap, false>(lds))),
                 std::max(std::max(camTraceGrid<false, BatchMap, true>(lds), camTraceGrid<true, BatchMap, true>(lds)),
                          std::max(camTraceGrid<false, ImageMap, true>(lds), camTraceGrid<true, ImageMap, true>(lds))));
    return (size_t)(S.stackDepth - inLds) * grid * kTraceBlock * sizeof(uint2);
}

// A round of the layer walk over `slots` slots, on `fraction` of the lanes that
// the device holds.
template <typename Map>
static void walkRound(hipStream_t s, const DevScene& S, DevState* st, const Map& map, uint32_t slots, PixelArrays px,
                      EntryArrays ent, uint32_t cap, uint32_t* cursor, uint2* spill, uint32_t inLds, float fraction,
                      bool count) {
    inLds = std::max(1u, inLds);
    if (S.stackDepth <= inLds) spill = nullptr;
    const size_t lds = walkLdsBytes(S, spill, inLds);
    const bool top = topFitsLds(S);
    const auto k = count ? (top ? &k_cam_trace<true, Map, true> : &k_cam_trace<true, Map, false>)
                         : (top ? &k_cam_trace<false, Map, true> : &k_cam_trace<false, Map, false>);
    const uint32_t full = traceGrid(reinterpret_cast<const void*>(k), lds);
    const uint32_t g = min(max(1u, (uint32_t)((float)full * fraction)), blocks(slots, kTraceBlock));
    const uint32_t waves = g * (kTraceBlock / 64u);
    k_walk_begin<<<1, 64, 0, s>>>(st, cursor, entryClaim(cap, waves) ? waves * kEntryOwn : 0u);
    k<<<g, kTraceBlock, lds, s>>>(S, st, map, px, ent, cap, cursor, spill, inLds);
}
void launchCamTrace(hipStream_t s, const DevScene& S, DevState* st, uint32_t npx, uint32_t width, PixelArrays px,
                    EntryArrays ent, uint32_t cap, uint32_t* cursor, uint2* spill, uint32_t inLds, bool count) {
    if (npx)
        walkRound(s, S, st, ImageMap{width, npx / width, (width + 7u) / 8u}, npx, px, ent, cap, cursor, spill, inLds,
                  1.0f, count);
}

void launchBatchInit(hipStream_t s, BatchDesc b, uint32_t maxTiles, PixelArrays px) {
    if (maxTiles) k_batch_init<<<blocks(maxTiles, 4), 256, 0, s>>>(b, px);
}

void launchCamTraceBatch(hipStream_t s, const DevScene& S, DevState* st, BatchDesc b, uint32_t maxSlots,
                         PixelArrays px, EntryArrays ent, uint32_t cap, uint32_t* cursor, uint2* spill,
                         uint32_t inLds, float gridFraction, bool count) {
    if (maxSlots)
        walkRound(s, S, st, BatchMap{b.tiles, b.segs, b.hdr}, maxSlots, px, ent, cap, cursor, spill, inLds, gridFraction,
                  count);
}

void launchCamCompositeBatch(hipStream_t s, uint32_t maxSlots, const BatchHeader* hdr, PixelArrays px,
                             EntryArrays ent) {
    if (maxSlots)
        k_cam_composite<<<blocks(maxSlots, 256), 256, 0, s>>>(maxSlots, &hdr->nSlots, px, ent, 0.0f, nullptr);
}

void launchBatchResolve(hipStream_t s, BatchDesc b, uint32_t maxResolve, PixelArrays px, float4* fb) {
    if (maxResolve) k_batch_resolve<<<blocks(maxResolve, 256), 256, 0, s>>>(b, px, fb);
}

void launchEntrySort(hipStream_t s, const DevScene& S, const GridParams& g, DevState* st, uint32_t cap, PixelArrays px,
                     EntryArrays ent, uint32_t* cellCount, uint32_t* cellStart, unsigned long long* scan) {
    if (!cap) return;
    const uint32_t gb = min(blocks(cap, 256), kEntryBlocks);
    const uint32_t shift = sortShift(g, cap);
    k_entry_key<<<gb, 256, 0, s>>>(S, g, shift, st, cap, px, ent, cellCount);
    launchExclusiveScan(s, cellCount, cellStart, sortBuckets(g, cap), scan);
    k_entry_scatter<<<gb, 256, 0, s>>>(st, cap, cellStart, cellCount, ent);
}

void launchEntryGather(hipStream_t s, const DevScene& S, const DevGrid& G, DevState* st, uint32_t cap, const uint32_t* nGather,
                       EntryArrays ent, bool count) {
    if (!cap) return;
    if (count)
        k_entry_gather<true><<<blocks(cap, 256), 256, 0, s>>>(S, G, st, nGather, ent);
    else
        k_entry_gather<false><<<blocks(cap, 256), 256, 0, s>>>(S, G, st, nGather, ent);
}

void launchCamComposite(hipStream_t s, uint32_t npx, PixelArrays px, EntryArrays ent, float invSpp, float4* fb) {
    if (npx) k_cam_composite<<<blocks(npx, 256), 256, 0, s>>>(npx, nullptr, px, ent, invSpp, fb);
}

void launchPostprocess(hipStream_t s, const float4* fb, float4* ldr, uint32_t n) {
    if (n) k_post<<<blocks(n, 256), 256, 0, s>>>(fb, ldr, n);
}
void launchAdjRaygenBatch(hipStream_t s, BatchDesc b, uint32_t maxTiles, const float* dloss, RayQueue q,
                          PendingArrays pend, DevState* st, uint32_t* segFirst) {
    k_adj_raygen_batch<<<blocks(max(maxTiles, 1u), 4), 256, 0, s>>>(b, dloss, q, pend, st, segFirst);
}
void launchAdjNext(hipStream_t s, DevState* st, int bounce, uint32_t poolCap, TileStates ts, uint32_t rays,
                   uint32_t* segFirst, uint32_t* segEnd, uint32_t* segNext, uint32_t nSegs, uint4* groups,
                   uint32_t nGroups, const uint32_t* groupSegs) {
    k_adj_next<<<1, 256, 0, s>>>(st, bounce, poolCap, ts, tilesOf(rays), segFirst, segEnd, segNext, nSegs, groups,
                                 nGroups, groupSegs);
}
void launchAdjShade(hipStream_t s, const DevScene& S, DevState* st, uint32_t maxRays, uint32_t bounce, RayQueue in,
                    HitArrays hits, RayQueue out, uint32_t outCap, EventArrays pool, uint32_t poolCap,
                    PendingArrays pend, TraceParams tp, uint32_t* segNext, TileStates ts) {
    if (maxRays)
        k_adj_shade<<<tilesOf(maxRays), kTile, 0, s>>>(S, st, bounce, in, hits, out, outCap, pool, poolCap, pend,
                                                       maxRays, tp, segNext, ts);
}
void launchAdjRaygen(hipStream_t s, const DevCamera& cam, const float* dloss, RayQueue q, PendingArrays pend,
                     DevState* st, uint32_t seed) {
    const uint32_t npx = cam.W * cam.H;
    k_adj_raygen<<<blocks(npx > 0 ? npx : 1, 256), 256, 0, s>>>(cam, dloss, q, pend, st, seed);
}
void launchEventSort(hipStream_t s, const GridParams& g, DevState* st, uint32_t poolCap, EventArrays ev,
                     uint32_t* cell, uint32_t* sorted, uint32_t* cellCount, uint32_t* cellStart,
                     unsigned long long* scan) {
    if (!poolCap) return;
    k_event_key<<<min(blocks(poolCap, 256), kEntryBlocks), 256, 0, s>>>(g, sortShift(g, poolCap), st, poolCap, ev, cell,
                                                                          cellCount);
    launchExclusiveScan(s, cellCount, cellStart, sortBuckets(g, poolCap), scan);
    k_event_scatter<<<min(blocks(poolCap, 256), kEntryBlocks), 256, 0, s>>>(st, poolCap, cell, cellStart, cellCount, sorted);
}
void launchAdjTransport(hipStream_t s, const DevScene& S, const DevGrid& G, DevState* st, uint32_t poolCap,
                        EventArrays ev, const uint32_t* sorted, float* gradOpacity, float* gradFull, float* debugImg,
                        bool count) {
    if (!poolCap) return;
    if (count)
        k_adj_transport<true><<<blocks(poolCap, 256), 256, 0, s>>>(S, G, st, poolCap, ev, sorted, gradOpacity,
                                                                  gradFull, debugImg);
    else
        k_adj_transport<false><<<blocks(poolCap, 256), 256, 0, s>>>(S, G, st, poolCap, ev, sorted,
                                                                   gradOpacity, gradFull, debugImg);
}
void launchSplitGradients(hipStream_t s, const float* gradFull, uint32_t n, float* position, float* tangentU,
                          float* tangentV, float* scale, float* albedo, float* beta) {
    if (n) k_split_gradients<<<blocks(n, 256), 256, 0, s>>>(gradFull, n, position, tangentU, tangentV, scale, albedo,
                                                            beta);
}
void launchTraceRays(hipStream_t s, const DevScene& S, DevState* st, uint32_t n, const float* o, const float* d,
                     int32_t* inst, int32_t* prim, float* t, float* pos, float* alpha) {
    if (!n) return;
    launchFill(s, st->traceNext, kCursorWords, 0u);
    const size_t lds = stackBytes(S);
    const uint32_t g = min(traceGrid(reinterpret_cast<const void*>(&k_trace_rays), lds), blocks(n, kTraceBlock));
    k_trace_rays<<<g, kTraceBlock, lds, s>>>(S, st, n, o, d, inst, prim, t, pos, alpha);
}

void launchGatherPoints(hipStream_t s, const DevGrid& G, uint32_t n, const float* q, const float* nrm, float* out) {
    if (n) k_gather_points<<<blocks(n, 256), 256, 0, s>>>(G, n, q, nrm, out);
}

void launchQuadNodes(hipStream_t s, const WideNode* nodes, QuadNode* quads, uint32_t first, uint32_t count,
                     uint32_t levels) {
    if (count) k_quad_nodes<<<blocks(count, 256), 256, 0, s>>>(nodes, quads, first, count, levels);
}

void launchSetOpacity(hipStream_t s, SurfelShade* shade, const float* opacity, uint32_t n) {
    if (n) k_set_opacity<<<blocks(n, 256), 256, 0, s>>>(shade, opacity, n);
}

void launchApplyPoints(hipStream_t s, SurfelGeo* geo, SurfelShade* shade, float* raw, DevPointArrays a, uint32_t n) {
    if (n) k_apply_points<<<blocks(n, 256), 256, 0, s>>>(geo, shade, raw, a, n);
}

}  // namespace pale
