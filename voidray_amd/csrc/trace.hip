// Ray-query kernels: the batch form of SceneAcceleration::hit
// (voidray_renderer/src/core/scene.rs:182-185) over rays resident in HBM.
#include <mutex>
#include <string>

#include "internal.h"
#include "traverse.h"

namespace vr {

constexpr int kWave = 64;        // gfx950 wavefront size; one wave per block
// LDS stack entries per lane (8 B each).  The tree pushes one entry a level at
// most and is 9 to 10 levels deep on the million-triangle scenes, so next to
// nothing spills; 5 and 6 KB per wave allow the 7 waves per SIMD that the
// registers do.
constexpr int kLdsStack = 10;
constexpr int kLdsStackAny = 12;
constexpr int kSpillCap = 48;    // global spill entries per lane beyond the LDS part
// Idle lanes that trigger a wave-wide refill.  On 2^22 rays through 2^20
// triangles (closest hit) 32 idle lanes cost 2%, 48 gain 1% and cost 1% on the
// cornell frame; any hit over a million rays: 32 3% faster than 40, 48 4% slower.
constexpr int kRefill = 40;
constexpr int kRefillAny = 32;
// A record step runs once this share of the walking lanes waits for one
// (1 / n), else a node step.  Closest hit: a third (half: 4% slower, a
// quarter: 0.5%); any hit, whose rays end at their first hit: half (a third:
// 7% slower).
constexpr int kVote = 3;
constexpr int kVoteAny = 2;
// Up to this many rays per launched wave go eight lanes to a ray, two to a
// group (trace_groups).  64 rays: 45 -> 31 us; a 960 x 540 x 4 frame, whose late
// bounces hold a few thousand rays, 6.49 -> 5.80 ms; 16 requests of mixed sizes
// 57.7 -> 51.9 ms.  With 4, 8 and 32 rays a wave the reference-estimator frame
// (719p x 8) took 7.13, 6.93 and 7.17 ms instead of 6.93.
constexpr uint32_t kGroupRays = 16;

struct TraceArgs {
    SceneView sv;  // first (cold_args)
    const float* o;
    const float* d;
    uint32_t n;
    float tmin;
    int any;
    uint32_t* prim;
    float* t;
    float* u;
    float* v;
    uint8_t* hit;
    uint32_t* fb_list;
    uint32_t* fb_count;
    uint32_t* next;       // partition counters of the dynamic ray fetch (kFetchStride apart)
    u32x2* spill;         // [spill_cap][spill_lanes]
    uint32_t spill_lanes;
    const uint32_t* queue;  // optional: item k traces ray queue[k] (else ray k)
    const uint32_t* count;  // optional: device-side item count (else n)
    float tmax;             // any-hit: hits at t >= tmax do not count
    int spill_cap;          // global spill entries per lane; a deeper stack hands the ray to the exact engine
    u32x4* rec;             // optional: {prim, t, u, v} as one record (a path's hit)
    const float* add_src;   // optional, [ray][3]: a ray without a hit adds its entry to
    float* add_dst;         // its entry here (a path's next-event radiance)
};

// The kernel's arguments, for code outside the traversal loop (cold_scene).
__device__ __forceinline__ const TraceArgs& cold_args(const TraceArgs& a) {
    return *(const TraceArgs*)&cold_scene(a.sv);
}

__device__ __forceinline__ void write_out(const TraceArgs& a, uint32_t i, const HitOut& h) {
    if (a.rec) a.rec[i] = u32x4{h.prim, f2u(h.t), f2u(h.u), f2u(h.v)};
    if (a.add_dst && h.prim == 0xFFFFFFFFu) {
        const float* s = a.add_src + 3 * (size_t)i;
        float* d = a.add_dst + 3 * (size_t)i;
        const vf3 sum = mk3(d[0], d[1], d[2]) + mk3(s[0], s[1], s[2]);
        d[0] = sum.x;
        d[1] = sum.y;
        d[2] = sum.z;
    }
    if (a.prim) a.prim[i] = h.prim;
    if (a.t) a.t[i] = h.t;
    if (a.u) a.u[i] = h.u;
    if (a.v) a.v[i] = h.v;
    if (a.hit) a.hit[i] = h.prim != 0xFFFFFFFFu ? 1 : 0;
}

// Words of a scene's trace counter block.  The wide kernel appends to the
// fallback list and fetches rays through the partition counters; the
// cooperative exact kernel appends overflows, counts finished blocks, and its
// last block publishes the launch's counts and clears the working words, so
// every launch starts from zero without a reset launch (or a memset node in a
// captured graph).
enum : int {
    kCtrFallbacks = 0,      // rays handed from the wide engine to the exact engine
    kCtrOverflow = 2,       // rays whose frontier outgrew the cooperative LDS stack
    kCtrBlocksDone = 3,     // finished blocks of the cooperative exact kernel
    kCtrLastFallbacks = 8,  // published: fallbacks of the last launch
    kCtrLastOverflow = 9,   // published: overflows of the last launch
    kCtrFetch = 64,         // first ray-fetch partition counter
    kCtrWords = 1024,
};
// Ray fetch.  The rays are cut into blocks of 2^lb, dealt to kFetchParts parts
// in turn; each part has its own waves (blockIdx mod kFetchParts) and its own
// counter on its own 128-byte line.  Thousands of waves refilling through one
// counter serialise on that address (about 20 ns an atomic), so no wave ever
// draws from another part: dealing small blocks balances the parts instead (a
// part holds some of every stretch of the launch's rays).  Parts cut as
// stretches of the launch, with the waves of a finished part drawing from the
// others, were 22% slower on the 512 x 512 cornell frame and 20% on a million
// any-hit rays: at the end all waves meet on the counters that are left.
// Workgroups are dealt round-robin to the 8 XCDs, so a part's waves all run on
// one XCD and adjacent rays share its L2.
constexpr uint32_t kLogFetchParts = 4;
constexpr int kFetchParts = 1 << kLogFetchParts;
constexpr uint32_t kLogFetchChunks = 4;    // a counter hands out 1/16 of a wave's share at a time ...
constexpr uint32_t kMaxFetchChunk = 256;   // ... between 64 and 256 rays (64: the 2^27-path frame 1-6% slower)
// Blocks of 2^lb <= 4,096 rays, at least 32 of them a part (2 or 4 a part: 2-3% slower).
VR_HD uint32_t fetch_log_block(uint32_t n, uint32_t lparts) {
    const uint32_t lg = 31u - (uint32_t)__builtin_clz(n | 1u);
    const uint32_t lb = lg > lparts + 5u ? lg - lparts - 5u : 0u;
    return lb > 12u ? 12u : lb;
}
// Items of part `part` of n.
VR_HD uint32_t fetch_part_size(uint32_t n, uint32_t part, uint32_t lparts, uint32_t lb) {
    const uint32_t round = lb + lparts, rest = n & ((1u << round) - 1u), at = part << lb;
    const uint32_t tail = rest > at ? rest - at : 0u;
    return ((n >> round) << lb) + (tail < (1u << lb) ? tail : 1u << lb);
}
// Item k of part `part`.
VR_HD uint32_t fetch_item(uint32_t k, uint32_t part, uint32_t lparts, uint32_t lb) {
    return ((((k >> lb) << lparts) | part) << lb) | (k & ((1u << lb) - 1u));
}
constexpr int kFetchStride = 32;  // words between two partition counters
static_assert(kCtrFetch + kFetchParts * kFetchStride <= kCtrWords, "counter block too small");
static_assert(kFetchParts <= 64, "one lane clears each partition counter");

// ---- few rays: eight lanes a ray --------------------------------------------
// A launch with few rays takes as long as its longest ray's chain of steps, and
// a step of one lane is about 270 dependent-issue instructions besides its
// memory latency.  Eight lanes share a ray instead: each tests one child box of
// a node, or one record of the node's leaves (all of them, whichever leaf was
// hit: a superset of the candidates changes no answer), and the results meet
// in cross-lane reductions.  All lanes of a group hold the same state and make
// the same branches.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, CTRL, 0xF, 0xF, true);
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141;  // lane ^ 1, ^ 2, 7 - lane of each 8
// Minimum over the 8 lanes of a group.
__device__ __forceinline__ uint32_t min8_u(uint32_t x) {
    x = min(x, dpp_u<kDppXor1>(x));
    x = min(x, dpp_u<kDppXor2>(x));
    return min(x, dpp_u<kDppHalfMirror>(x));
}
__device__ __forceinline__ float min8_f(float x) {
    x = fminf(x, u2f(dpp_u<kDppXor1>(f2u(x))));
    x = fminf(x, u2f(dpp_u<kDppXor2>(f2u(x))));
    return fminf(x, u2f(dpp_u<kDppHalfMirror>(f2u(x))));
}

// Node step of a group (as wide_node_step and wide_node; `stk`: the group's
// stack in LDS, CAP entries; every lane writes the same entry).
template <int CAP, bool ANY, bool WT, bool INST, class WorldRay>
__device__ __forceinline__ uint32_t group_node_step(const SceneView& sv, WideState& st, lds_u32x2* stk, uint32_t c,
                                                    float tmin, float tmax_any, WorldRay world_ray) {
    while (st.cur == kNoNode) {
        if (st.sp == 0) return kStepDone;
        const u32x2 e = stk[st.sp - 1];
        if (INST && (e.x & kInstEntry)) {
            --st.sp;
            if (e.x == kInstExit) {
                vf3 wo, wd;
                world_ray(wo, wd);
                wide_instance_exit<WT>(st, wo, wd);
            } else if (ANY || !(u2f(e.y) > st.tbest * kCullSlack)) {
                if (st.sp >= CAP) return kStepFallback;
                const WideStack ws{stk, 1, nullptr, 0, 0};
                return (uint32_t)wide_instance_enter<CAP, WT>(sv, st, ws, e.x, tmin);
            }
            continue;
        }
        if (!ANY && u2f(e.y & 0xFFFF0000u) > st.tbest * kCullSlack) {
            --st.sp;
            continue;
        }
        const uint32_t hits = e.y & 0xFFu;
        const uint32_t slot = (e.x & kDescend) ? 31u - (uint32_t)__builtin_clz(hits) : (uint32_t)__builtin_ctz(hits);
        st.cur = (e.x & ~kDescend) + slot;
        if (hits & (hits - 1u)) stk[st.sp - 1] = u32x2{e.x, e.y & ~(1u << slot)};
        else --st.sp;
    }
    const QNode* q = sv.qnodes + st.cur;
    const u32x4 w0 = ((const u32x4*)q)[0], w1 = ((const u32x4*)q)[1];
    const uint8_t* lo = &q->qlo[0][0] + c;  // this lane's child; hi bytes 24 after lo
    const uint32_t lx = lo[0], ly = lo[8], lz = lo[16], hx = lo[24], hy = lo[32], hz = lo[40];
    const uint32_t e = w0.w;
    const float sx = u2f((e & 0xFFu) << 23) * st.idx;
    const float sy = u2f(((e >> 8) & 0xFFu) << 23) * st.idy;
    const float sz = u2f(((e >> 16) & 0xFFu) << 23) * st.idz;
    const uint32_t num_inner = e >> 24;
    const float bx = (u2f(w0.x) - st.o.x) * st.idx;
    const float by = (u2f(w0.y) - st.o.y) * st.idy;
    const float bz = (u2f(w0.z) - st.o.z) * st.idz;
    const bool negx = st.idx < 0.f, negy = st.idy < 0.f, negz = st.idz < 0.f;
    const float tcull = ANY ? tmax_any : st.tbest * kCullSlack;
    const float nx = fmaf((float)(negx ? hx : lx), sx, bx), fx = fmaf((float)(negx ? lx : hx), sx, bx);
    const float ny = fmaf((float)(negy ? hy : ly), sy, by), fy = fmaf((float)(negy ? ly : hy), sy, by);
    const float nz = fmaf((float)(negz ? hz : lz), sz, bz), fz = fmaf((float)(negz ? lz : hz), sz, bz);
    const float tnear = fmaxf(fmaxf(nx, ny), fmaxf(nz, tmin));
    const float tfar = fminf(fminf(fx, fy), fminf(fz, tcull));
    const bool hit = tnear <= tfar * kSlabSlack;
    uint32_t hits = (uint32_t)(__ballot(hit) >> (threadIdx.x & 56u)) & 0xFFu;
    const uint32_t inner = (1u << num_inner) - 1u;
    uint32_t leaves = hits & ~inner;
    leaves = (leaves | (leaves << 8)) & 0x00F00Fu;
    leaves = (leaves | (leaves << 4)) & 0x0C30C3u;
    leaves = (leaves | (leaves << 2)) & 0x249249u;
    st.tg_all = w1.z & 0xFFFFFFu;
    st.tg_mask = ((leaves << 3) - leaves) & st.tg_all;
    st.tg_base = w1.y;
    hits &= inner;
    st.cur = kNoNode;
    if (hits) {
        const uint32_t axis = (w1.z >> 24) & 3u;
        const bool neg = axis == 0u ? negx : axis == 1u ? negy : negz;
        uint32_t slot, bound = 0;
        if (ANY) {
            slot = neg ? 31u - (uint32_t)__builtin_clz(hits) : (uint32_t)__builtin_ctz(hits);
        } else {
            const uint32_t key = hit && c < num_inner ? (f2u(tnear) & ~7u) | c : 0xFFFFFFFFu;
            const uint32_t m1 = min8_u(key), m2 = min8_u(key == m1 ? 0xFFFFFFFFu : key);
            slot = m1 & 7u;
            bound = (m2 & 0xFFFF0000u) | (tmin < 0.0f ? 0xFFFF0000u : 0u);
        }
        st.cur = w1.x + slot;
        hits &= ~(1u << slot);
        if (hits) {
            if (st.sp >= CAP) return kStepFallback;
            stk[st.sp++] = u32x2{w1.x | (neg ? kDescend : 0u), bound | hits};
        }
    }
    return kStepContinue;
}

// Record step of a group: all records of the node's leaves, eight at a time.
template <int CAP, bool ANY, bool WT, bool INST>
__device__ __forceinline__ uint32_t group_tri_step(const SceneView& sv, WideState& st, lds_u32x2* stk, uint32_t c,
                                                   float tmin, float tmax_any) {
    const uint32_t gl = threadIdx.x & 56u, count = (uint32_t)__builtin_popcount(st.tg_all);
    const bool in_inst = INST && st.inst != kNoInstance;
    st.tg_mask = 0;
    for (uint32_t r0 = 0; r0 < count; r0 += 8) {
        float t = kInf, u = 0.f, v = 0.f;
        uint32_t prim = 0xFFFFFFFFu, slot = 0;
        bool enter = false, found = false, unconfirmed = false;
        u32x2 entry{};
        if (r0 + c < count) {
            const uint32_t rec = st.tg_base + r0 + c;
            slot = sv.tri_ref ? sv.tri_ref[rec] : rec;
            vf3 p0, p1, p2;
            load_tri_geom(sv.tris, slot, p0, p1, p2);
            if (INST && f2u(p2.x) == kInstanceMarker) {
                const float tcull = ANY ? tmax_any : st.tbest * kCullSlack;
                const float ax = (p0.x - st.o.x) * st.idx, bx = (p1.x - st.o.x) * st.idx;
                const float ay = (p0.y - st.o.y) * st.idy, by = (p1.y - st.o.y) * st.idy;
                const float az = (p0.z - st.o.z) * st.idz, bz = (p1.z - st.o.z) * st.idz;
                const float tnear = fmaxf(fmaxf(fminf(ax, bx), fminf(ay, by)), fmaxf(fminf(az, bz), tmin));
                const float tfar = fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fminf(fmaxf(az, bz), tcull));
                enter = tnear <= tfar * kSlabSlack;
                entry = u32x2{kInstEntry | f2u(p2.y), f2u(tnear)};
            } else {
                MTResult m;
                if (WT ? wt_hit(st.wt, st.o, p0, p1, p2, tmin, m)
                       : mt_hit(st.o, st.d, p0, p1, p2, tmin, m, in_inst ? st.inst_eps : -1.0f)) {
                    prim = (in_inst ? st.inst_base : 0u) + tri_word(sv.tris, slot, 9);
                    if (!ANY || m.t < tmax_any) {
                        found = !ANY || WT || in_inst ||
                                confirm_winner(cold_scene(sv), st.o, st.d, tmin, m.t, p0, p1, p2,
                                               tri_word(sv.tris, slot, 11), prim);
                        unconfirmed = !found;
                    }
                    t = m.t;
                    u = m.u;
                    v = m.v;
                }
            }
        }
        if (INST) {
            const uint32_t es = (uint32_t)(__ballot(enter) >> gl) & 0xFFu;
            if (es) {
                const int ne = __builtin_popcount(es);
                if (st.sp + ne > CAP) return kStepFallback;
                // (lane by lane, each entry written by all lanes, as every other push)
                for (uint32_t m = es; m; m &= m - 1u) {
                    const int from = (int)(gl + (uint32_t)__builtin_ctz(m));
                    stk[st.sp++] = u32x2{(uint32_t)__shfl((int)entry.x, from), (uint32_t)__shfl((int)entry.y, from)};
                }
            }
        }
        const uint32_t fs = (uint32_t)(__ballot(found) >> gl) & 0xFFu;
        if (ANY && ((uint32_t)(__ballot(unconfirmed) >> gl) & 0xFFu)) st.unconfirmed = 1u;
        if (fs == 0u) continue;
        // the winner: any hit the first lane's, closest hit the least (t, prim)
        uint32_t w;
        if (ANY) {
            w = (uint32_t)__builtin_ctz(fs);
        } else {
            const float tm = min8_f(found ? t : kInf);
            if (tm > st.tbest) continue;
            const bool tie = found && t == tm;
            const uint32_t pm = min8_u(tie ? prim : 0xFFFFFFFFu);
            if (!(tm < st.tbest || pm < st.best_prim)) continue;
            w = (uint32_t)__builtin_ctz((uint32_t)(__ballot(tie && prim == pm) >> gl) & 0xFFu);
        }
        const int from = (int)(gl + w);
        st.tbest = __shfl(t, from);
        st.bu = __shfl(u, from);
        st.bv = __shfl(v, from);
        st.best_prim = (uint32_t)__shfl((int)prim, from);
        st.best_slot = (uint32_t)__shfl((int)slot, from);
        if (INST) st.best_inst = st.inst;
        if (ANY) {
            st.found = 1u;
            return kStepDone;
        }
    }
    return kStepContinue;
}

template <bool ANY, bool WT, bool INST, int LDS>
__device__ __forceinline__ void trace_groups(const TraceArgs& a, uint32_t n, u32x2* lds) {
    constexpr int CAP = LDS * 8;
    const uint32_t lane = threadIdx.x, c = lane & 7u;
    lds_u32x2* stk = (lds_u32x2*)lds + (lane >> 3) * CAP;
    WideState st;
    uint32_t status = kStepDone, ray = 0xFFFFFFFFu;
    st.tg_mask = 0;
    // one ray a wave first, then a second one, ...
    for (uint32_t k = blockIdx.x + gridDim.x * (lane >> 3);;) {
        if (status != kStepContinue) {
            const TraceArgs& x = cold_args(a);
            if (ray != 0xFFFFFFFFu) {
                HitOut h;
                const int rc = status == kStepFallback ? kStepFallback : wide_finish<ANY, WT, INST>(x.sv, st, x.tmin, h);
                if (c == 0u) {
                    if (rc == kStepFallback) x.fb_list[atomicAdd(x.fb_count, 1u)] = ray;
                    else write_out(x, ray, h);
                }
                ray = 0xFFFFFFFFu;
            }
            if (k < n) {
                ray = x.queue ? x.queue[k] : k;
                k += gridDim.x * 8u;
                status = kStepContinue;
                const vf3 o = mk3(x.o[3 * ray], x.o[3 * ray + 1], x.o[3 * ray + 2]);
                const vf3 d = mk3(x.d[3 * ray], x.d[3 * ray + 1], x.d[3 * ray + 2]);
                wide_init<WT>(st, o, d, x.sv.num_qnodes > 0);
                if (x.sv.num_analytic) wide_seed_analytic<ANY, WT>(x.sv, st, x.tmin, x.tmax);
            }
        }
        const uint64_t walking = __ballot(status == kStepContinue);
        if (walking == 0ull) break;
        const uint64_t tri = __ballot(status == kStepContinue && st.tg_mask != 0u);
        if (2 * __popcll(tri) >= __popcll(walking)) {
            if (status == kStepContinue && st.tg_mask != 0u)
                status = group_tri_step<CAP, ANY, WT, INST>(a.sv, st, stk, c, a.tmin, a.tmax);
        } else if (status == kStepContinue && st.tg_mask == 0u) {
            status = group_node_step<CAP, ANY, WT, INST>(a.sv, st, stk, c, a.tmin, a.tmax, [&](vf3& wo, vf3& wd) {
                const TraceArgs& x = cold_args(a);
                wo = mk3(x.o[3 * ray], x.o[3 * ray + 1], x.o[3 * ray + 2]);
                wd = mk3(x.d[3 * ray], x.d[3 * ray + 1], x.d[3 * ray + 2]);
            });
        }
    }
}

// Persistent wide-engine kernel: every lane runs its own ray as a resumable
// state machine whose next step is a node or a triangle record.  In each
// iteration the wave votes: a record step runs if enough of the walking lanes
// wait for one (kVote), else a node step, so a good part of them takes part
// in every step, whatever their rays need.  A ray that has ended waits in its lane until kRefill lanes of
// the wave are idle; then all of them confirm and write their hits together
// and the wave fetches as many new rays with one atomic (dynamic ray fetch).
template <bool ANY, bool WT, bool INST>
__device__ __forceinline__ void trace_persist(const TraceArgs& a) {
    constexpr int LDS = ANY ? kLdsStackAny : kLdsStack;
    __shared__ u32x2 lds[LDS * kWave];
    const int lane = threadIdx.x;
    const uint32_t glane = blockIdx.x * kWave + lane;
    const WideStack ws{(lds_u32x2*)(lds + lane), kWave, a.spill + glane, (int)a.spill_lanes, a.spill_cap};
    const uint32_t n = a.count ? *a.count : a.n;
    if (n <= gridDim.x * kGroupRays) {
        trace_groups<ANY, WT, INST, LDS>(a, n, lds);
        return;
    }
    WideState st;
    uint32_t ray = 0;
    // The lane's state as one word.  (As bools they were lane masks in
    // scalar registers, which spilled: 3% slower.)
    enum : uint32_t { kWalk = 0, kDone = 1, kExact = 2, kIdle = 3 };
    uint32_t status = kIdle;
    st.tg_mask = 0;
    // Waves and blocks of 2^lb rays are dealt to the parts in turn.  A wave's
    // first rays are its own by position, as many as an equal share of a small
    // launch allows (at most 64): few rays are spread over all waves, where
    // they end soonest, and nothing is fetched for them.  What the first rays
    // of a part's waves leave of it is drawn from its counter in chunks.  (1 or
    // kFetchParts parts and shifts: nothing divides but once.)
    const uint32_t lparts = gridDim.x >= (uint32_t)kFetchParts ? kLogFetchParts : 0u, parts = 1u << lparts;
    const uint32_t part = blockIdx.x & (parts - 1u);
    const uint32_t waves = (gridDim.x - part + parts - 1u) >> lparts;  // of this part
    const uint32_t lb = fetch_log_block(n, lparts);
    const uint32_t size = fetch_part_size(n, part, lparts, lb);
    const uint32_t share = size ? (size - 1u) / waves + 1u : 0u;
    const uint32_t first = min(share, 64u), chunk = min(max(share >> kLogFetchChunks, 64u), kMaxFetchChunk);
    // the wave's rays at hand: the part's [base, end)
    uint32_t base = min(first * (blockIdx.x >> lparts), size), end = min(base + first, size);
    bool dry = first * waves >= size, exhausted = false;  // nothing left to draw; and no ray at hand
    for (;;) {
        const uint64_t walking = __ballot(status == kWalk);
        if (walking == 0ull || (!exhausted && 64 - __popcll(walking) >= (ANY ? kRefillAny : kRefill))) {
            const TraceArgs& c = cold_args(a);
            // finished rays: confirm and write, or hand over to the exact engine
            if (status == kDone || status == kExact) {
                HitOut h;
                int rc = status == kExact ? kStepFallback : wide_finish<ANY, WT, INST>(c.sv, st, c.tmin, h);
                if (rc == kStepFallback) {
                    uint32_t slot = atomicAdd(c.fb_count, 1u);
                    c.fb_list[slot] = ray;
                } else {
                    write_out(c, ray, h);
                }
                status = kIdle;
            }
            if (exhausted) break;  // (no lane walks)
            const uint64_t idle_mask = ~walking;
            const uint32_t nidle = (uint32_t)__popcll(idle_mask);
            // rays at hand, and if they do not suffice a new chunk [nbase, nend)
            const uint32_t avail = end - base;
            uint32_t nbase = 0, nend = 0;
            if (avail < nidle && !dry) {
                uint32_t got = 0;
                if (lane == 0) got = atomicAdd(c.next + part * kFetchStride, chunk);
                nbase = min(first * waves + __shfl(got, 0), size);
                nend = min(nbase + chunk, size);
                dry = nend == size;
            }
            const uint32_t rank = (uint32_t)__popcll(idle_mask & ((1ull << lane) - 1ull));
            const uint32_t k = rank < avail ? base + rank : nbase + (rank - avail);
            if (status == kIdle && (rank < avail || k < nend)) {
                const uint32_t item = fetch_item(k, part, lparts, lb);
                ray = c.queue ? c.queue[item] : item;
                status = kWalk;
                vf3 o = mk3(c.o[3 * ray], c.o[3 * ray + 1], c.o[3 * ray + 2]);
                vf3 d = mk3(c.d[3 * ray], c.d[3 * ray + 1], c.d[3 * ray + 2]);
                wide_init<WT>(st, o, d, c.sv.num_qnodes > 0);
                if (c.sv.num_analytic) wide_seed_analytic<ANY, WT>(c.sv, st, c.tmin, c.tmax);
            }
            if (avail < nidle) {
                base = min(nbase + (nidle - avail), nend);
                end = nend;
            } else {
                base += nidle;
            }
            exhausted = dry && base == end;
            continue;
        }
        const uint64_t tri = __ballot(status == kWalk && st.tg_mask != 0u);
        if ((ANY ? kVoteAny : kVote) * __popcll(tri) >= __popcll(walking)) {
            if (status == kWalk && st.tg_mask != 0u)
                status = (uint32_t)wide_tri_step<LDS, ANY, WT, INST>(a.sv, st, ws, a.tmin, a.tmax);
        } else {
            if (status == kWalk && st.tg_mask == 0u)
                status = (uint32_t)wide_node_step<LDS, ANY, WT, INST>(a.sv, st, ws, a.tmin, a.tmax, [&](vf3& wo, vf3& wd) {
                    const TraceArgs& c = cold_args(a);
                    wo = mk3(c.o[3 * ray], c.o[3 * ray + 1], c.o[3 * ray + 2]);
                    wd = mk3(c.d[3 * ray], c.d[3 * ray + 1], c.d[3 * ray + 2]);
                });
        }
    }
}

// Registers held to 7 waves per SIMD (72 VGPRs, no scratch).  The kernel waits
// for memory as much as it issues: at 3, 4, 5 and 6 waves the 2^27-path terrain
// frame took 30%, 16%, 8% and 1% longer; at 8 waves it spills.
template <bool ANY, bool WT = false, bool INST = false>
__global__ void k_trace_persist(TraceArgs a);
template <>
__global__ __launch_bounds__(kWave, 7) void k_trace_persist<false, false, false>(TraceArgs a) {
    trace_persist<false, false, false>(a);
}
template <>
__global__ __launch_bounds__(kWave, 7) void k_trace_persist<true, false, false>(TraceArgs a) {
    trace_persist<true, false, false>(a);
}
// watertight engine (extended estimator only)
template <>
__global__ __launch_bounds__(kWave, 7) void k_trace_persist<false, true, false>(TraceArgs a) {
    trace_persist<false, true, false>(a);
}
template <>
__global__ __launch_bounds__(kWave, 7) void k_trace_persist<true, true, false>(TraceArgs a) {
    trace_persist<true, true, false>(a);
}
// scenes with instances (the instance bookkeeping needs more registers): 5 waves
// per SIMD, 96 VGPRs, 4 of the watertight kernels' spilled.  Frames of 200
// instances with 4, 5 and 6 waves: 960 x 540 x 4 5.65, 5.51 and 5.64 ms
// (watertight 5.73, 5.64, 6.28), 1080p x 16 37.2, 34.9 and 34.6 ms (37.6, 35.7,
// 41.5); at 7 dozens of registers spill.
template <>
__global__ __launch_bounds__(kWave, 5) void k_trace_persist<false, false, true>(TraceArgs a) {
    trace_persist<false, false, true>(a);
}
template <>
__global__ __launch_bounds__(kWave, 5) void k_trace_persist<true, false, true>(TraceArgs a) {
    trace_persist<true, false, true>(a);
}
template <>
__global__ __launch_bounds__(kWave, 5) void k_trace_persist<false, true, true>(TraceArgs a) {
    trace_persist<false, true, true>(a);
}
template <>
__global__ __launch_bounds__(kWave, 5) void k_trace_persist<true, true, true>(TraceArgs a) {
    trace_persist<true, true, true>(a);
}

__device__ __forceinline__ uint32_t load_agent(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Serial exact engine for one ray, with its stacks in the caller's LDS.
template <bool WT>
__device__ __forceinline__ void exact_serial(const TraceArgs& a, uint32_t i, int32_t* tstack, int32_t* mstack, int stride) {
    vf3 o = mk3(a.o[3 * i], a.o[3 * i + 1], a.o[3 * i + 2]);
    vf3 d = mk3(a.d[3 * i], a.d[3 * i + 1], a.d[3 * i + 2]);
    HitOut h;
    trace_exact_stk<WT>(a.sv, o, d, a.tmin, h, tstack, mstack, stride);
    if (a.any && h.prim != 0xFFFFFFFFu && !(h.t < a.tmax)) h.prim = 0xFFFFFFFFu;
    write_out(a, i, h);
}

// Wave-cooperative exact engine: one wave per listed ray.  The reference
// traversal visits every node whose ancestors all pass the slab test, so the
// candidate set does not depend on visiting order; the wave pops up to 64
// pending nodes at once from an LDS stack, tests them in parallel and pushes
// the children of passing nodes.  The winner is the lexicographic minimum of
// (t, prim) over the wave, identical to trace_exact.  A ray whose frontier
// outgrows the LDS stack is listed for the serial engine, which the last block
// to finish runs over the list, one ray per lane.  `list` == nullptr: every
// ray (or every queued ray) is traced; otherwise the wide engine's fallbacks.
constexpr int kCoopStack = 6144;
static_assert(kCoopStack * 2 >= 2 * 64 * kWave, "the serial stacks reuse the cooperative stack");
enum : uint32_t { kCoopTop = 0u, kCoopMesh = 1u, kCoopTri = 2u };

template <bool WT>
__global__ __launch_bounds__(kWave) void k_trace_exact_wave(TraceArgs a, const uint32_t* list, uint32_t* ctr,
                                                            uint32_t* serial_list, uint64_t* accum) {
    __shared__ u32x2 stk[kCoopStack];
    const int lane = threadIdx.x;
    const SceneView& sv = a.sv;
    // (agent-scope loads: a select between a device count and the by-value
    // argument would otherwise be folded into one load through a pointer to a
    // private copy of the arguments)
    uint32_t n = a.n;
    if (list) n = load_agent(&ctr[kCtrFallbacks]);
    else if (a.count) n = load_agent(a.count);
    // Blocks without a ray leave at once; the others (at least block 0) take
    // part in the exit count.  A block that leaves may read the count after
    // the reset, but then it reads 0 and leaves all the same: the reset only
    // happens once every taking-part block has read the count.
    // (Without a ray, the usual case, there is no list to run and nobody to wait
    // for: block 0 resets without the fences and the count.  64 rays: 31.6 -> 30.7 us.)
    if (n == 0u) {
        if (blockIdx.x != 0u) return;
        if (lane == 0) ctr[kCtrLastFallbacks] = ctr[kCtrLastOverflow] = 0u;
        if (lane < kFetchParts) ctr[kCtrFetch + lane * kFetchStride] = 0u;
        return;
    }
    const uint32_t parts = n < gridDim.x ? (n > 1u ? n : 1u) : gridDim.x;
    if (blockIdx.x >= parts) return;
    for (uint32_t j = blockIdx.x; j < n; j += gridDim.x) {
        uint32_t ray = list ? list[j] : (a.queue ? a.queue[j] : j);
        vf3 o = mk3(a.o[3 * ray], a.o[3 * ray + 1], a.o[3 * ray + 2]);
        vf3 d = mk3(a.d[3 * ray], a.d[3 * ray + 1], a.d[3 * ray + 2]);
        float bt = kInf, bu = 0.f, bv = 0.f;
        uint32_t bprim = 0xFFFFFFFFu;
        WTRay wt{};
        if (WT) wt = wt_prepare(d);
        int sp = sv.top_root_valid ? 1 : 0;  // wave-uniform
        if (lane == 0) stk[0] = u32x2{kCoopTop << 30, 0u};
        bool overflow = false;
        __syncthreads();
        while (sp > 0) {
            int take = sp < kWave ? sp : kWave;
            u32x2 e = u32x2{0u, 0u};
            bool act = lane < take;
            if (act) e = stk[sp - take + lane];
            __syncthreads();
            sp -= take;
            // entries to push: two tree children (e0 = right, e1 = left), one
            // mesh root, or a run of np small-mesh triangles (e0.x + k)
            u32x2 e0 = u32x2{0u, 0u}, e1 = u32x2{0u, 0u};
            int np = 0;
            bool run = false;
            if (act) {
                uint32_t kind = e.x >> 30, idx = e.x & 0x3FFFFFFFu, surf = e.y;
                if (kind == kCoopTop) {
                    RefNode nd = sv.top_nodes[idx];
                    if (nd.obj >= 0) {
                        uint32_t s2 = (uint32_t)nd.obj;
                        const SurfaceInfo& si2 = sv.surfaces[s2];
                        if (si2.analytic >= 0) {  // analytic surface: its hit, in this lane
                            float t, u, v;
                            if (analytic_hit(sv.analytic[si2.analytic], o, d, a.tmin, t, u, v) &&
                                (t < bt || (t == bt && si2.prim_base < bprim))) {
                                bt = t;
                                bu = u;
                                bv = v;
                                bprim = si2.prim_base;
                            }
                        } else {
                            MeshInfo mi = sv.meshes[si2.mesh];
                            if (mi.root >= 0) {
                                e0 = u32x2{(kCoopMesh << 30) | (uint32_t)mi.root, s2};
                                np = 1;
                            } else {
                                e0 = u32x2{kCoopTri << 30, s2};
                                np = (int)(mi.num_tris < 4u ? mi.num_tris : 4u);
                                run = true;
                            }
                        }
                    } else {
                        Box3 b{mk3(nd.lo[0], nd.lo[1], nd.lo[2]), mk3(nd.hi[0], nd.hi[1], nd.hi[2])};
                        if (WT ? wt_slab_hit(b, o, d, a.tmin, kInf) : ref_slab_hit(b, o, d, a.tmin, kInf)) {
                            e0 = u32x2{(kCoopTop << 30) | (uint32_t)nd.right, 0u};
                            e1 = u32x2{(kCoopTop << 30) | (idx + 1), 0u};
                            np = 2;
                        }
                    }
                } else {
                    SurfaceInfo si = sv.surfaces[surf];
                    MeshInfo mi = sv.meshes[si.mesh];
                    // an instance's mesh is walked with the ray in its object space
                    vf3 mo = o, md = d;
                    WTRay mwt = wt;
                    float meps = -1.0f;
                    if (si.instance >= 0) {
                        instance_ray(sv.instances[si.instance], o, d, mo, md);
                        if (WT) mwt = wt_prepare(md);
                        meps = a.tmin * sv.instances[si.instance].det_inv;
                    }
                    int32_t tri = -1;
                    if (kind == kCoopMesh) {
                        RefNode nd = sv.ref_nodes[idx];
                        if (nd.obj >= 0) {
                            tri = nd.obj;
                        } else {
                            Box3 b{mk3(nd.lo[0], nd.lo[1], nd.lo[2]), mk3(nd.hi[0], nd.hi[1], nd.hi[2])};
                            if (WT ? wt_slab_hit(b, mo, md, a.tmin, kInf) : ref_slab_hit(b, mo, md, a.tmin, kInf)) {
                                e0 = u32x2{(kCoopMesh << 30) | (uint32_t)nd.right, surf};
                                e1 = u32x2{(kCoopMesh << 30) | (idx + 1), surf};
                                np = 2;
                            }
                        }
                    } else {
                        tri = (int32_t)idx;
                    }
                    if (tri >= 0) {
                        const uint32_t* ix = sv.mesh_idx + 3 * (size_t)(mi.tri_base + (uint32_t)tri);
                        const float* vp = sv.vpos + 3 * (size_t)mi.vert_base;
                        vf3 p0 = mk3(vp[3 * ix[0]], vp[3 * ix[0] + 1], vp[3 * ix[0] + 2]);
                        vf3 p1 = mk3(vp[3 * ix[1]], vp[3 * ix[1] + 1], vp[3 * ix[1] + 2]);
                        vf3 p2 = mk3(vp[3 * ix[2]], vp[3 * ix[2] + 1], vp[3 * ix[2] + 2]);
                        MTResult r;
                        if (WT ? wt_hit(mwt, mo, p0, p1, p2, a.tmin, r)
                               : mt_hit(mo, md, p0, p1, p2, a.tmin, r, meps)) {
                            const uint32_t prim = si.prim_base + (uint32_t)tri;
                            if (r.t < bt || (r.t == bt && prim < bprim)) {
                                bt = r.t;
                                bu = r.u;
                                bv = r.v;
                                bprim = prim;
                            }
                        }
                    }
                }
            }
            // wave exclusive scan of push counts
            int incl = np;
#pragma unroll
            for (int off = 1; off < kWave; off <<= 1) {
                int y = __shfl_up(incl, off);
                if (lane >= off) incl += y;
            }
            int total = __shfl(incl, kWave - 1);
            int base = sp + incl - np;
            if (sp + total > kCoopStack) {
                overflow = true;
                break;
            }
            for (int k = 0; k < np; ++k)
                stk[base + k] = run ? u32x2{e0.x + (uint32_t)k, e0.y} : (k == 0 ? e0 : e1);
            sp += total;
            __syncthreads();
        }
        __syncthreads();
        if (overflow) {
            if (lane == 0) {
                uint32_t slot = atomicAdd(&ctr[kCtrOverflow], 1u);
                serial_list[slot] = ray;
            }
            continue;
        }
        // wave argmin of (t, prim)
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            float ot = __shfl_xor(bt, off);
            float ou = __shfl_xor(bu, off), ov = __shfl_xor(bv, off);
            uint32_t oprim = __shfl_xor(bprim, off);
            bool take_other = oprim != 0xFFFFFFFFu &&
                              (bprim == 0xFFFFFFFFu || ot < bt || (ot == bt && oprim < bprim));
            if (take_other) {
                bt = ot;
                bu = ou;
                bv = ov;
                bprim = oprim;
            }
        }
        if (a.any && bprim != 0xFFFFFFFFu && !(bt < a.tmax)) bprim = 0xFFFFFFFFu;
        if (lane == 0) {
            HitOut h;
            h.prim = bprim;
            h.t = bprim == 0xFFFFFFFFu ? 0.f : bt;
            h.u = bprim == 0xFFFFFFFFu ? 0.f : bu;
            h.v = bprim == 0xFFFFFFFFu ? 0.f : bv;
            write_out(a, ray, h);
        }
    }
    // count this block out; the last one runs the overflow list and resets
    // (one same-address atomic per taking-part block, not per block)
    __threadfence();
    uint32_t ticket = 0;
    if (lane == 0) ticket = atomicAdd(&ctr[kCtrBlocksDone], 1u);
    ticket = __shfl(ticket, 0);
    if (ticket != parts - 1) return;
    __threadfence();
    const uint32_t ns = load_agent(&ctr[kCtrOverflow]);
    if (ns) {  // the cooperative stack is free now: 64 + 64 stack entries per lane
        int32_t* lds32 = (int32_t*)stk;
        for (uint32_t k = lane; k < ns; k += kWave)
            exact_serial<WT>(a, load_agent(&serial_list[k]), lds32 + lane, lds32 + 64 * kWave + lane, kWave);
    }
    if (lane == 0) {
        uint32_t fb = list ? load_agent(&ctr[kCtrFallbacks]) : 0u;
        if (accum) *accum += fb;
        ctr[kCtrLastFallbacks] = fb;
        ctr[kCtrLastOverflow] = ns;
        ctr[kCtrFallbacks] = 0u;
        ctr[kCtrOverflow] = 0u;
        ctr[kCtrBlocksDone] = 0u;
    }
    if (lane < kFetchParts) ctr[kCtrFetch + lane * kFetchStride] = 0u;
}

// The persistent kernel for a query: [any + 2 * watertight + 4 * instances].
static void (*const kPersistKernels[8])(TraceArgs) = {
    k_trace_persist<false, false, false>, k_trace_persist<true, false, false>, k_trace_persist<false, true, false>,
    k_trace_persist<true, true, false>,   k_trace_persist<false, false, true>, k_trace_persist<true, false, true>,
    k_trace_persist<false, true, true>,   k_trace_persist<true, true, true>};

static int persist_grid(vr_scene* s, bool any, bool wt, uint32_t& blocks) {
    const bool inst = s->view.num_instances > 0;
    const int k = (any ? 1 : 0) + (wt ? 2 : 0) + (inst ? 4 : 0);
    if (s->persist_blocks[k] == 0) {
        int dev = 0, cus = 0, per_cu = 0;
        VR_HIP_CHECK(hipGetDevice(&dev));
        VR_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        void (*const* kern)(TraceArgs) = kPersistKernels;
        VR_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern[k], kWave, 0));
        s->persist_blocks[k] = (uint32_t)std::max(1, cus * std::max(1, per_cu));
    }
    blocks = s->persist_blocks[k];
    return 0;
}

int ensure_trace_scratch(vr_scene* s, uint32_t n) {
    if (!s->spill) {
        uint32_t b[4] = {0, 0, 0, 0};
        for (int k = 0; k < 4; ++k) {
            int rc = persist_grid(s, k & 1, k & 2, b[k]);
            if (rc) return rc;
        }
        s->spill_lanes = std::max(std::max(b[0], b[1]), std::max(b[2], b[3])) * kWave;
        size_t bytes = (size_t)kSpillCap * s->spill_lanes * sizeof(u32x2);
        if (hipMalloc((void**)&s->spill, bytes) != hipSuccess) return fail(VR_ERR_OOM, "spill stack allocation failed");
    }
    if (!s->counters) {
        VR_HIP_CHECK(hipMalloc((void**)&s->counters, kCtrWords * sizeof(uint32_t)));
        VR_HIP_CHECK(hipHostMalloc((void**)&s->host_counters, 64 * sizeof(uint32_t), hipHostMallocDefault));
        for (int k = 0; k < 64; ++k) s->host_counters[k] = 0;
        // starts at zero; from then on every launch leaves it at zero
        std::vector<uint32_t> zeros(kCtrWords, 0u);
        VR_HIP_CHECK(hipMemcpy(s->counters, zeros.data(), kCtrWords * sizeof(uint32_t), hipMemcpyHostToDevice));
    }
    // two lists of n entries: wide-engine fallbacks, then the serial-exact overflow list
    if (s->fallback_cap < 2 * n) {
        if (s->fallback_list) VR_HIP_CHECK(hipFree(s->fallback_list));
        s->fallback_list = nullptr;
        if (hipMalloc((void**)&s->fallback_list, 2 * (size_t)n * sizeof(uint32_t)) != hipSuccess)
            return fail(VR_ERR_OOM, "fallback list allocation failed");
        s->fallback_cap = 2 * n;
    }
    return 0;
}

// Device scratch of one trace launch: the counter block (kCtrWords), the
// wide engine's fallback list and the exact engine's overflow list (one entry
// per ray each), and the per-lane spill stacks of the persistent kernels.
struct TraceScratch {
    uint32_t* counters;
    uint32_t* fb_list;
    uint32_t* serial_list;
    u32x2* spill;
    uint32_t spill_lanes;   // lanes the spill stacks cover (the grid may use fewer)
    int spill_cap;
};

static int launch_trace_with(vr_scene* s, const TraceJob& j, const TraceScratch& sc, hipStream_t stream) {
    TraceArgs a{s->view, j.o, j.d, j.n_max, j.tmin, j.any ? 1 : 0, j.prim, j.t, j.u, j.v, j.hit,
                sc.fb_list, sc.counters, sc.counters + kCtrFetch, sc.spill, sc.spill_lanes, j.queue, j.count, j.tmax,
                sc.spill_cap, j.rec, j.add_src, j.add_dst};
    const bool wt = j.engine == VR_ENGINE_WATERTIGHT;
    uint64_t* accum = j.engine != VR_ENGINE_REFERENCE ? j.fallback_accum : nullptr;
    if (j.engine != VR_ENGINE_REFERENCE) {
        uint32_t blocks = 0;
        int rc = persist_grid(s, j.any, wt, blocks);
        if (rc) return rc;
        blocks = std::min<uint32_t>(blocks, sc.spill_lanes / kWave);
        blocks = std::min<uint32_t>(blocks, j.n_max);
        void (*persist)(TraceArgs) =
            kPersistKernels[(j.any ? 1 : 0) + (wt ? 2 : 0) + (s->view.num_instances > 0 ? 4 : 0)];
        void (*exact)(TraceArgs, const uint32_t*, uint32_t*, uint32_t*, uint64_t*) =
            wt ? k_trace_exact_wave<true> : k_trace_exact_wave<false>;
        if (j.timed) VR_HIP_CHECK(hipEventRecord(s->trace_ev[0], stream));
        hipLaunchKernelGGL(persist, dim3(blocks), dim3(kWave), 0, stream, a);
        if (j.timed) VR_HIP_CHECK(hipEventRecord(s->trace_ev[1], stream));
        // fallbacks: one wave per ray; the grid reads the device-side count (no host sync)
        hipLaunchKernelGGL(exact, dim3(1024), dim3(kWave), 0, stream, a, (const uint32_t*)sc.fb_list, sc.counters,
                           sc.serial_list, accum);
    } else {
        uint32_t blocks = std::min<uint32_t>(j.n_max, 65535u);
        void (*exact)(TraceArgs, const uint32_t*, uint32_t*, uint32_t*, uint64_t*) = k_trace_exact_wave<false>;
        hipLaunchKernelGGL(exact, dim3(blocks), dim3(kWave), 0, stream, a, (const uint32_t*)nullptr, sc.counters,
                           sc.serial_list, accum);
    }
    VR_HIP_CHECK(hipGetLastError());
    return 0;
}

int launch_trace(vr_scene* s, const TraceJob& j, hipStream_t stream) {
    if (j.n_max == 0) return 0;
    int rc = ensure_trace_scratch(s, j.n_max);
    if (rc) return rc;
    TraceScratch sc{s->counters, s->fallback_list, s->fallback_list + s->fallback_cap / 2, s->spill, s->spill_lanes,
                    kSpillCap};
    return launch_trace_with(s, j, sc, stream);
}

static int check_trace_desc(const vr_trace_desc* desc, const float* d_o, const float* d_d) {
    if (!d_o || !d_d) return fail(VR_ERR_INVALID, "null ray buffers");
    const int32_t m = desc->mode & ~VR_TRACE_TIMING;
    if (m != VR_TRACE_CLOSEST && m != VR_TRACE_ANY) return fail(VR_ERR_INVALID, "bad trace mode");
    if (desc->engine != VR_ENGINE_WIDE && desc->engine != VR_ENGINE_REFERENCE && desc->engine != VR_ENGINE_WATERTIGHT)
        return fail(VR_ERR_INVALID, "bad engine");
    return 0;
}

int trace_device(vr_scene* s, const vr_trace_desc* desc, const float* d_o, const float* d_d, uint32_t* d_prim,
                 float* d_t, float* d_u, float* d_v, uint8_t* d_hit, hipStream_t stream) {
    uint32_t n = desc->num_rays;
    if (n == 0) return 0;
    int rc = check_trace_desc(desc, d_o, d_d);
    if (rc) return rc;
    TraceJob j;
    j.o = d_o;
    j.d = d_d;
    j.n_max = n;
    j.tmin = desc->t_min;
    j.tmax = kInf;
    j.any = (desc->mode & ~VR_TRACE_TIMING) == VR_TRACE_ANY;
    j.engine = desc->engine;
    j.prim = d_prim;
    j.t = d_t;
    j.u = d_u;
    j.v = d_v;
    j.hit = d_hit;
    j.timed = (desc->mode & VR_TRACE_TIMING) && desc->engine != VR_ENGINE_REFERENCE;
    if (j.timed && !s->trace_ev[0]) {
        VR_HIP_CHECK(hipEventCreate(&s->trace_ev[0]));
        VR_HIP_CHECK(hipEventCreate(&s->trace_ev[1]));
    }
    s->trace_timed = j.timed;
    rc = launch_trace(s, j, stream);
    if (rc) return rc;
    VR_HIP_CHECK(hipMemcpyAsync(s->host_counters, s->counters + kCtrLastFallbacks, 2 * sizeof(uint32_t),
                                hipMemcpyDeviceToHost, stream));
    return 0;
}

// ---- ray queries without allocation --------------------------------------
// vr_trace_device_noalloc_async keeps all of its device scratch in one
// file-scope array per GPU, laid out as
//   [counter block: kCtrWords u32][fallback list: kNoAllocMaxRays u32]
//   [overflow list: kNoAllocMaxRays u32][spill stacks: kNoAllocSpill x kNoAllocLanes x 8 B]
// The persistent grid is capped at kNoAllocMaxBlocks one-wave blocks (32 per
// CU on 256 CUs: every resident wave), and a lane's traversal stack may spill
// kNoAllocSpill entries past its LDS ring; a deeper stack sends the ray to the
// exact engine, which gives the same answer.
constexpr uint32_t kNoAllocMaxRays = VR_NOALLOC_MAX_RAYS;
constexpr uint32_t kNoAllocMaxBlocks = 8192;
constexpr uint32_t kNoAllocLanes = kNoAllocMaxBlocks * kWave;
constexpr int kNoAllocSpill = 16;
constexpr size_t kNoAllocCtrBytes = (size_t)kCtrWords * sizeof(uint32_t);
constexpr size_t kNoAllocListBytes = (size_t)kNoAllocMaxRays * sizeof(uint32_t);
constexpr size_t kNoAllocSpillBytes = (size_t)kNoAllocSpill * kNoAllocLanes * sizeof(u32x2);
constexpr size_t kNoAllocBytes = kNoAllocCtrBytes + 2 * kNoAllocListBytes + kNoAllocSpillBytes;
static_assert(kNoAllocBytes == VR_NOALLOC_SCRATCH_BYTES, "scratch size differs from the header's");
static_assert(kNoAllocCtrBytes % 256 == 0 && kNoAllocListBytes % 256 == 0, "scratch parts stay 256-byte aligned");

static __device__ __align__(256) uint8_t scratch[kNoAllocBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

__global__ void k_clear_words(uint32_t* p, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

// Device address of `scratch` on `device`, looked up once per device (with
// that device current) and kept: in host code the array's name is only a
// host-side stand-in, never a device address.
int noalloc_scratch(int device, void** out) {
    if (device < 0 || device >= kMaxDevices) return fail(VR_ERR_INVALID, "device index out of range for the trace scratch");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        int cur = 0;
        VR_HIP_CHECK(hipGetDevice(&cur));
        if (cur != device) VR_HIP_CHECK(hipSetDevice(device));
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e == hipSuccess && p) {
            // the counter block must start at zero; every launch leaves it so
            hipLaunchKernelGGL(k_clear_words, dim3(4), dim3(256), 0, nullptr, (uint32_t*)p, (uint32_t)kCtrWords);
            e = hipGetLastError();
            if (e == hipSuccess) e = hipDeviceSynchronize();
        }
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess || !p)
            return fail(VR_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch_ptr[device] = p;
    }
    *out = g_scratch_ptr[device];
    return 0;
}

int trace_device_noalloc(vr_scene* s, const vr_trace_desc* desc, const float* d_o, const float* d_d,
                         uint32_t* d_prim, float* d_t, float* d_u, float* d_v, uint8_t* d_hit, hipStream_t stream) {
    const uint32_t n = desc->num_rays;
    if (n > kNoAllocMaxRays)
        return fail(VR_ERR_INVALID, "vr_trace_device_noalloc_async traces at most VR_NOALLOC_MAX_RAYS (1,048,576) "
                                    "rays per call; split the batch");
    if (n == 0) return 0;
    int rc = check_trace_desc(desc, d_o, d_d);
    if (rc) return rc;
    void* base = nullptr;
    rc = noalloc_scratch(s->ctx->device, &base);
    if (rc) return rc;
    uint8_t* b = (uint8_t*)base;
    TraceScratch sc{(uint32_t*)b, (uint32_t*)(b + kNoAllocCtrBytes),
                    (uint32_t*)(b + kNoAllocCtrBytes + kNoAllocListBytes),
                    (u32x2*)(b + kNoAllocCtrBytes + 2 * kNoAllocListBytes), kNoAllocLanes, kNoAllocSpill};
    // whatever an earlier call on this GPU left, this call starts from zero
    hipLaunchKernelGGL(k_clear_words, dim3(4), dim3(256), 0, stream, sc.counters, (uint32_t)kCtrWords);
    TraceJob j;
    j.o = d_o;
    j.d = d_d;
    j.n_max = n;
    j.tmin = desc->t_min;
    j.tmax = kInf;
    j.any = (desc->mode & ~VR_TRACE_TIMING) == VR_TRACE_ANY;
    j.engine = desc->engine;
    j.prim = d_prim;
    j.t = d_t;
    j.u = d_u;
    j.v = d_v;
    j.hit = d_hit;
    j.timed = false;
    return launch_trace_with(s, j, sc, stream);
}

}  // namespace vr
