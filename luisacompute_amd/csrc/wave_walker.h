// wave_walker.h -- BVH8 traversal of one ray per lane with the triangle tests of a wave shared by
// its lanes (the persistent trace kernel, trace.hip). Same semantics and node format as Walker
// (traverse.h); every member is called by all 64 lanes of a wave together.
//
// A node step visits one node per lane that has one. The triangles of the leaf slots it hits go
// into a queue of (triangle record, lane) pairs that the wave keeps in LDS. Once the queue holds
// enough pairs, or no lane has a node left, a triangle step tests up to 64 pairs, one per lane,
// whichever lanes' rays they belong to: the ray's data come from its lane by ds_bpermute, and the
// nearest hit per ray is settled by a 64-bit minimum in LDS over (distance, primitive).
// Tested by the lanes that own them instead, the triangles of a step filled 20-30% of a wave (soup
// of 16.7M triangles: 11.1M triangle steps for 213M tests) while the other lanes idled in a kernel
// that VALU issue bounds. With the queue 3.16 G instructions per 8.4M rays on that soup instead of 4.03,
// 5.0 ms instead of 6.0 (618 G/s, 4.1 TB/s behind the L2s); 2.1M rays on 1M triangles 1,463 -> 1,215 us.
// Two levels issue 440-460 G/s and wait for half of the waves' cycles at 5 waves per SIMD: 1,024 instances
// 1,502 -> 919 us with the sort rule, the 1080p room of four samples 16.5 -> 15.1 ms.
#pragma once

#include "lc_hip_internal.h"
#include "traverse.h"

namespace lchip {
namespace trav {

constexpr uint32_t kTriQueue = 128; // pairs a wave's queue holds (a power of two)

// Inclusive prefix sum over the 64 lanes through DPP row shifts and broadcasts (no LDS).
template<int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_add(uint32_t v) {
    return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
}
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
    v = dpp_add<0x111, 0xF>(v); // row_shr:1
    v = dpp_add<0x112, 0xF>(v);
    v = dpp_add<0x114, 0xF>(v);
    v = dpp_add<0x118, 0xF>(v);
    v = dpp_add<0x142, 0xA>(v); // row_bcast:15 into rows 1 and 3
    return dpp_add<0x143, 0xC>(v); // row_bcast:31 into rows 2 and 3
}

// Orders the LDS accesses of one wave: they complete in order, this keeps the compiler from moving
// them across the point.
__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float from_lane(uint32_t lane4, float v) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute((int)lane4, __float_as_int(v)));
}
__device__ __forceinline__ uint32_t from_lane(uint32_t lane4, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)lane4, (int)v);
}

// Distances as unsigned integers in the same order; -0 and +0 are one value.
__device__ __forceinline__ uint32_t t_order(float t) {
    const uint32_t u = __float_as_uint(t + 0.0f);
    return u ^ ((uint32_t)((int)u >> 31) | 0x80000000u);
}
__device__ __forceinline__ float t_value(uint32_t k) {
    return __uint_as_float(k ^ ((k & 0x80000000u) ? 0x80000000u : 0xFFFFFFFFu));
}

constexpr uint32_t kKeyInf = 0xFF800000u; // t_order(+inf)
constexpr uint32_t kNegZero = 0x80000000u; // in a hit's record word: its distance is -0

template<bool ANY, int BLOCK, int SLDS>
struct WaveShared {
    uint2 stk[SLDS][BLOCK];                          // traversal stacks, one column per lane
    uint2 queue[BLOCK / 64][kTriQueue];              // (triangle record, lane)
    unsigned long long key[ANY ? BLOCK / 64 : BLOCK]; // nearest hit per lane; ANY: mask of lanes with a hit
    float u[ANY ? 1 : BLOCK], v[ANY ? 1 : BLOCK];    // barycentrics and record of the nearest hit
    uint32_t rec[ANY ? 1 : BLOCK];
};

// What is traced and where its rays and results are: plain traces over ray batches. (query.hip has the
// other mode: nearest-commit ray queries, whose candidates go through callbacks.)
struct TraceMode {
    using Params = TraceParams;
    static constexpr bool kQuery = false;
    __device__ __forceinline__ static void locate(const Params &P, uint32_t q, uint32_t &batch, uint32_t &ray) {
        batch = find_batch(P.batches, q);
        ray = q - P.batches.b[batch].start;
    }
    __device__ __forceinline__ static const float4 *rays(const Params &P, uint32_t batch) { return P.batches.b[batch].rays; }
    __device__ __forceinline__ static uint32_t mask(const Params &P, uint32_t batch) { return P.batches.b[batch].mask; }
    __device__ __forceinline__ static char *out(const Params &P, uint32_t batch) { return static_cast<char *>(P.batches.b[batch].out); }
};

template<bool ANY, bool TWO, bool COUNT, int BLOCK, int SLDS, class Mode = TraceMode>
struct WaveWalker {
    using Shared = WaveShared<ANY, BLOCK, SLDS>;
    using Params = typename Mode::Params;
    static constexpr bool kQuery = Mode::kQuery;
    static_assert(!kQuery || (TWO && !ANY && !COUNT), "queries: nearest commit over instances");
    Shared *sh;
    uint2 *queue;          // this wave's queue
    uint32_t tid, lane;
    uint32_t head, tail;   // wave-uniform: pairs taken from and put into the queue so far
    uint32_t last;         // `tail` after this lane's latest pair
    int sp;
    RaySetup R;            // current (object space when inside an instance)
    float tmin, tmax;
    uint32_t batch, ray;   // which ray this is: its batch and the index there
    float t_best;          // nearest hit so far (inside an instance: or the limit it was entered with)
    bool any_hit;          // some hit so far (two-level closest hit: in an instance left before)
    uint32_t g_base, g_mask, t_base, t_mask;
    int floor;             // stack height of the current level: 0, or where the instance was entered
    uint32_t cur_inst;     // instance this lane is in (two-level; kWorld: in the TLAS)
    uint32_t cur_flags;    // queries: its InstanceRecord flags
    const WideNode *nodes;
    const TriRecord *tris;
    uint64_t n_nodes, n_tris, n_live, n_wave; // counting form only: node visits, triangle tests, lane and wave steps (account)

    static constexpr uint32_t kWorld = 0xFFFFFFFFu;
    __device__ __forceinline__ bool in_blas() const { return !TWO || cur_inst != kWorld; }

    __device__ __forceinline__ void init(const Params &P, Shared *shared, uint32_t t) {
        sh = shared; tid = t; lane = t & 63u; queue = shared->queue[t >> 6];
        head = tail = last = 0u;
        sp = floor = 0; g_mask = t_mask = 0u; any_hit = false;
        n_nodes = 0; n_tris = 0; n_live = 0; n_wave = 0;
        if constexpr (TWO) {
            nodes = P.geo.tlas_nodes;
            tris = nullptr;
            cur_inst = kWorld;
        } else {
            nodes = P.geo.blas_nodes;
            tris = P.geo.blas_tris;
            cur_inst = 0u;
        }
        cur_flags = 0u;
        batch = ray = 0u;
    }

    // This lane's spill entry k (TraceGrid::spill_areas; traces that count nothing take 64 rays per wave,
    // or eight lanes per ray). As in Walker the host sizes spill_depth from the built depths; the checks
    // only guard memory.
    __device__ __forceinline__ uint2 *spill_at(const Params &P, int k) const {
        uint64_t area = (uint64_t)blockIdx.x * BLOCK + tid;
        if ((kQuery || COUNT) && P.lanes != 0u)
            area = ((uint64_t)blockIdx.x * (BLOCK / 64) + (tid >> 6)) * P.lanes + lane;
        return P.spill + area * P.spill_depth + k;
    }
    __device__ __forceinline__ void push(const Params &P, uint2 e) {
        if (sp < SLDS) sh->stk[sp][tid] = e;
        else if ((uint32_t)(sp - SLDS) < P.spill_depth) *spill_at(P, sp - SLDS) = e;
        else atomicOr(P.error, 1u);
        sp++;
    }
    __device__ __forceinline__ uint2 pop(const Params &P) {
        sp--;
        if (sp < SLDS) return sh->stk[sp][tid];
        if ((uint32_t)(sp - SLDS) < P.spill_depth) return *spill_at(P, sp - SLDS);
        return make_uint2(0u, 0u);
    }

    __device__ __forceinline__ void reset_key(float limit) {
        if (!ANY) sh->key[tid] = ((unsigned long long)t_order(limit) << 32) | 0xFFFFFFFFu;
    }

    // Ray `r` of batch `b` as the launch was given it.
    __device__ __forceinline__ void load_ray(const Params &P, float o[3], float d[3], float &lo, float &hi) const {
        const float4 *rays = Mode::rays(P, batch);
        const float4 r0 = rays[2 * (uint64_t)ray], r1 = rays[2 * (uint64_t)ray + 1];
        o[0] = r0.x; o[1] = r0.y; o[2] = r0.z; lo = r0.w;
        d[0] = r1.x; d[1] = r1.y; d[2] = r1.z; hi = r1.w;
    }
    __device__ __forceinline__ uint2 *out_hit(const Params &P) const {
        return reinterpret_cast<uint2 *>(Mode::out(P, batch) + 24ull * ray);
    }

    // A new ray for this lane (called by the lanes that take one).
    __device__ __forceinline__ void start(const Params &P, uint32_t b, uint32_t r) {
        const auto &G = P.geo;
        batch = b;
        ray = r;
        t_best = FLT_MAX * 2.0f; // +inf
        any_hit = false;
        sp = floor = 0;
        t_mask = 0;
        g_base = 0;
        last = head;
        float o[3], d[3];
        load_ray(P, o, d, tmin, tmax);
        reset_key(t_best);
        if constexpr (TWO) {
            for (int k = 0; k < 3; k++) { R.o[k] = o[k]; R.d[k] = d[k]; }
            cur_inst = kWorld;
            nodes = G.tlas_nodes;
            ray_setup(R);
            g_mask = G.empty ? 0u : ((1u << R.oct) | (1u << 8));
            if constexpr (kQuery) {
                if (!G.two) { // one instance and no TLAS: instance 0 is entered next
                    g_mask = 0u;
                    t_base = 0u;
                    t_mask = G.empty ? 0u : 1u;
                }
            }
        } else {
            xform_point(G.inst_inv, o, R.o);
            xform_vector(G.inst_inv, d, R.d);
            ray_setup(R);
            g_mask = (G.empty || (G.inst_mask & Mode::mask(P, b) & 0xFFu) == 0u) ? 0u : ((1u << R.oct) | (1u << 8));
        }
    }

    __device__ __forceinline__ bool pending() const { return (int)(last - head) > 0; }
    __device__ __forceinline__ bool node_work() const { return t_mask == 0u && ((g_mask & 0xFFu) != 0u || sp > floor); }
    // instance work: an instance to enter, or one whose nodes and pairs are used up
    __device__ __forceinline__ bool inst_work() const {
        return TWO && (in_blas() ? (t_mask == 0u && (g_mask & 0xFFu) == 0u && sp == floor && !pending()) : t_mask != 0u);
    }
    // nothing left to do for this lane's ray
    __device__ __forceinline__ bool finished() const {
        return t_mask == 0u && (g_mask & 0xFFu) == 0u && sp == 0 && !pending() && (!TWO || !in_blas());
    }

    // Puts the triangles a lane holds (t_base, t_mask) into the queue, as far as it has room; what
    // does not fit stays with its lane, which visits no node until it is in.
    __device__ __forceinline__ void queue_triangles(bool active) {
        uint32_t m = active && in_blas() ? t_mask : 0u;
        if (__ballot(m != 0u) == 0ull) return;
        const uint32_t c = (uint32_t)__popc(m);
        const uint32_t upto = wave_scan(c);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)upto, 63);
        const uint32_t room = kTriQueue - (tail - head);
        uint32_t pos = upto - c;
        while (m != 0u && pos < room) {
            queue[(tail + pos) & (kTriQueue - 1u)] = make_uint2(t_base + (uint32_t)__builtin_ctz(m), lane);
            m &= m - 1u;
            pos++;
            last = tail + pos;
        }
        if (active && in_blas()) t_mask = m;
        tail += min(total, room);
        lds_order();
    }

    // Tests up to 64 pairs of the queue, one per lane.
    __device__ __forceinline__ void triangle_step(const Params &P) {
        const uint32_t n = min(64u, tail - head);
        const bool on = lane < n;
        const uint2 e = queue[(head + lane) & (kTriQueue - 1u)];
        const uint32_t owner = on ? e.y : lane, from = owner << 2;
        RaySetup r;
        r.o[0] = from_lane(from, R.o[0]); r.o[1] = from_lane(from, R.o[1]); r.o[2] = from_lane(from, R.o[2]);
        r.Sx = from_lane(from, R.Sx); r.Sy = from_lane(from, R.Sy); r.Sz = from_lane(from, R.Sz);
        r.kxyz = from_lane(from, R.kxyz);
        const float lo = from_lane(from, tmin), hi = from_lane(from, tmax);
        const TriRecord *base = tris;
        if (TWO) {
            const uint64_t p = reinterpret_cast<uint64_t>(tris);
            base = reinterpret_cast<const TriRecord *>((uint64_t)from_lane(from, (uint32_t)p) |
                                                       ((uint64_t)from_lane(from, (uint32_t)(p >> 32)) << 32));
        }
        bool hit = false;
        float t = 0.0f, u = 0.0f, v = 0.0f;
        uint32_t prim = 0u, procedural = 0u;
        if constexpr (kQuery) {
            const uint32_t inst = from_lane(from, cur_inst), flags = from_lane(from, cur_flags);
            procedural = on && (flags & kInstProcedural) ? 1u : 0u;
            if (__ballot(procedural != 0u) != 0ull) { // the callback takes the object-space ray
                r.d[0] = from_lane(from, R.d[0]); r.d[1] = from_lane(from, R.d[1]); r.d[2] = from_lane(from, R.d[2]);
                if (procedural) {
                    const float4 *pr = reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(base) + 32ull * e.x);
                    const float4 b0 = pr[0], b1 = pr[1];
                    prim = __float_as_uint(b0.w);
                    hit = Mode::procedural(P, inst, prim, r.o, r.d, b0, b1, t) && t >= lo && t < hi;
                }
            }
            if (on && !procedural) {
                const float4 *tr = reinterpret_cast<const float4 *>(base + e.x);
                const float4 a = tr[0], b = tr[1], c = tr[2];
                prim = __float_as_uint(a.w);
                hit = wt_intersect(r, a, b, c, lo, hi, t, u, v) &&
                      ((flags & kInstOpaque) || Mode::surface(P, inst, prim, u, v, t));
            }
        } else if (on) {
            const float4 *tr = reinterpret_cast<const float4 *>(base + e.x);
            const float4 a = tr[0], b = tr[1], c = tr[2];
            if (COUNT) n_tris++;
            hit = wt_intersect(r, a, b, c, lo, hi, t, u, v);
            prim = __float_as_uint(a.w);
        }
        head += n;
        if (__ballot(hit) == 0ull) return;
        if (ANY) {
            unsigned long long *word = sh->key + (tid >> 6);
            if (lane == 0u) *word = 0ull;
            lds_order();
            if (hit) atomicOr(word, 1ull << owner);
            lds_order();
            if ((*word >> lane) & 1ull) { // occluded: nothing left to visit (pairs still queued may be tested)
                any_hit = true;
                g_mask = 0u;
                t_mask = 0u;
                sp = 0;
                if (TWO) { floor = 0; cur_inst = kWorld; }
            }
            lds_order();
        } else {
            unsigned long long *slot = sh->key + (tid & ~63u) + owner;
            const unsigned long long k = ((unsigned long long)t_order(t) << 32) | prim;
            if (hit) atomicMin(slot, k);
            lds_order();
            if (hit && *slot == k) { // the nearest of its ray so far
                const uint32_t w = (tid & ~63u) + owner;
                sh->u[w] = u;
                sh->v[w] = v;
                sh->rec[w] = (kQuery ? procedural : e.x) | (__float_as_uint(t) == 0x80000000u ? kNegZero : 0u);
            }
            lds_order();
            t_best = t_value((uint32_t)(sh->key[tid] >> 32));
        }
    }

    // Leaves the current instance and / or enters the next one (called by the lanes with inst_work()).
    __device__ __forceinline__ void instance_step(const Params &P) {
        const auto &G = P.geo;
        float o[3], d[3], lo, hi;
        load_ray(P, o, d, lo, hi);
        bool world = false; // the world-space ray is needed again
        if (in_blas()) {
            if (!ANY) {
                // the nearest hit of the instances left before is in the ray's output record
                const unsigned long long k = sh->key[tid];
                const uint32_t prim = (uint32_t)k;
                if (prim != 0xFFFFFFFFu) {
                    if (COUNT) {
                        t_best = t_value((uint32_t)(k >> 32));
                    } else {
                        const float t = t_value((uint32_t)(k >> 32));
                        bool better = !any_hit;
                        if (any_hit) {
                            const uint2 *h = out_hit(P);
                            const uint2 h0 = h[0];
                            better = nearer(t, cur_inst, prim, __uint_as_float(kQuery ? h[2].y : h[2].x), h0.x, h0.y);
                        }
                        if (better) store_hit(P, k, cur_inst);
                        any_hit = true;
                        t_best = t;
                    }
                }
            }
            cur_inst = kWorld;
            floor = 0;
            if (sp > 0) {
                const uint2 e = pop(P);
                if (e.y & kInstGroup) { // more instances of the same TLAS leaf
                    t_base = e.x;
                    t_mask = e.y & ~kInstGroup;
                } else {
                    g_base = e.x;
                    g_mask = e.y;
                }
                world = true;
            }
        }
        while (t_mask != 0u) {
            const uint32_t b = (uint32_t)__builtin_ctz(t_mask);
            t_mask &= t_mask - 1u;
            uint32_t id = 0u;
            if constexpr (kQuery) id = G.two ? G.tlas_prims[t_base + b] : 0u;
            else id = G.tlas_prims[t_base + b];
            const InstanceRecord *ir = G.instances + id;
            const uint32_t imask = ir->vis_mask;
            const uint64_t bn = ir->blas_nodes;
            // procedural primitives report only to ray queries (plain traces run without
            // intersection functions, cpu/accel.rs:476-484)
            const uint32_t iflags = ir->flags;
            if (bn == 0u || (imask & Mode::mask(P, batch) & 0xFFu) == 0u || (!kQuery && (iflags & kInstProcedural))) continue;
            cur_flags = iflags;
            if ((g_mask & 0xFFu) != 0u) push(P, make_uint2(g_base, g_mask));
            if (t_mask != 0u) push(P, make_uint2(t_base, t_mask | kInstGroup));
            t_mask = 0u;
            float inv[12];
            const float4 *m = reinterpret_cast<const float4 *>(ir->inv);
            const float4 m0 = m[0], m1 = m[1], m2 = m[2];
            inv[0] = m0.x; inv[1] = m0.y; inv[2] = m0.z; inv[3] = m0.w;
            inv[4] = m1.x; inv[5] = m1.y; inv[6] = m1.z; inv[7] = m1.w;
            inv[8] = m2.x; inv[9] = m2.y; inv[10] = m2.z; inv[11] = m2.w;
            xform_point(inv, o, R.o);
            xform_vector(inv, d, R.d);
            nodes = reinterpret_cast<const WideNode *>(bn);
            tris = reinterpret_cast<const TriRecord *>(ir->blas_tris);
            cur_inst = id;
            floor = sp;
            reset_key(t_best);
        }
        if (in_blas()) {
            ray_setup(R);
            g_base = 0;
            g_mask = (1u << R.oct) | (1u << 8);
        } else if (world) { // back to the TLAS
            for (int k = 0; k < 3; k++) { R.o[k] = o[k]; R.d[k] = d[k]; }
            ray_setup(R);
            nodes = G.tlas_nodes;
        }
    }

    // Visits the next node of this lane (called by the lanes with node_work()).
    __device__ __forceinline__ void visit(const Params &P) {
        if ((g_mask & 0xFFu) == 0u) {
            const uint2 e = pop(P);
            if (TWO && (e.y & kInstGroup)) {
                t_base = e.x;
                t_mask = e.y & ~kInstGroup;
                return;
            }
            g_base = e.x;
            g_mask = e.y;
        }
        const float tcull = ANY ? tmax : fminf(tmax, t_best);
        uint32_t hm = g_mask & 0xFFu;
        const uint32_t im = (g_mask >> 8) & 0xFFu;
        const uint32_t i = (uint32_t)__builtin_ctz(hm);
        hm &= hm - 1u;
        const uint32_t slot = i ^ R.oct;
        const uint32_t node = g_base + (uint32_t)__popc(im & ((1u << slot) - 1u));
        if (hm != 0u) push(P, make_uint2(g_base, hm | (im << 8)));
        uint4 w0, w1, w2, w3, w4;
        load_node(nodes, node, w0, w1, w2, w3, w4);
        if (COUNT) n_nodes++;
        const uint32_t hits = intersect_node(R, w0, w1, w2, w3, w4, tmin, tcull);
        const uint32_t nim = w0.w >> 24;
        g_base = w1.x;
        g_mask = permute8(hits & nim, R.oct) | (nim << 8);
        uint32_t leaf = hits & ~nim;
        uint32_t nt = 0u;
        while (leaf) {
            const uint32_t s = (uint32_t)__builtin_ctz(leaf);
            leaf &= leaf - 1u;
            const uint32_t m = ((s < 4 ? w1.z : w1.w) >> (8 * (s & 3))) & 0xFFu;
            nt |= ((1u << (m >> 5)) - 1u) << (m & 31u);
        }
        t_base = w1.y;
        t_mask = nt;
    }

    // Counting form: a step of the wave, in which this lane is busy or not.
    __device__ __forceinline__ void account(bool busy) {
        if (busy) n_live++;
        if (lane == 0u) n_wave++;
    }

    // Runs up to P.steps steps of the wave's rays (`active` lanes hold one), each of the kind that
    // the most lanes can take: a triangle step tests one queued pair per lane, an instance step
    // moves lanes into and out of instances, a node step visits a node per lane. A queue that fills
    // P.tri_quarters quarters of a wave goes first, so that distances found cull later boxes.
    // (Against fixed quarters for both kinds 6% on a path-traced room, 3% on a soup of 1M triangles.)
    // Returns when no lane has work left, or, with P.refill_below > 0 and rays to hand out
    // (can_refill), once fewer lanes than that are busy.
    __device__ __forceinline__ void run(const Params &P, bool active, bool can_refill) {
        const uint32_t full = 16u * P.tri_quarters; // 1..4 (set_step_policy)
        const uint32_t refill_below = can_refill ? P.refill_below : 0u;
        for (int it = 0; it < P.steps; it++) {
            const bool work = active && node_work();
            const uint64_t wm = __ballot(work);
            const uint32_t queued = tail - head;
            if ((uint32_t)__popcll(wm) < refill_below &&
                (uint32_t)__popcll(__ballot(active && !finished())) < refill_below)
                return;
            bool tri = queued >= full || (queued != 0u && queued >= (uint32_t)__popcll(wm));
            if (TWO && !tri) {
                const uint64_t im = __ballot(active && inst_work());
                if (im != 0ull && (wm == 0ull || (uint32_t)__popcll(im) >= (uint32_t)__popcll(wm))) {
                    if (COUNT) account(active && !finished());
                    if (active && inst_work()) instance_step(P);
                    continue;
                }
            }
            if (!tri && wm == 0ull) { // no node to visit: test what is queued
                if (queued == 0u) return; // every ray is done
                tri = true;
            }
            if (COUNT) account((active && !finished()) || (tri && lane < queued));
            if (tri) triangle_step(P);
            else if (work) visit(P);
            queue_triangles(active);
        }
    }

    static constexpr unsigned long long kMissKey = 0xFFFFFFFFull;
    // Writes the ray's closest-hit record (24-B SurfaceHit) for the nearest hit `k` of instance `inst`;
    // the padding word carries the leaf record with P.hit_record (queues of the path tracer).
    __device__ __forceinline__ void store_hit(const Params &P, unsigned long long k, uint32_t inst) const {
        uint2 *h = out_hit(P);
        const uint32_t prim = (uint32_t)k;
        const bool hit = prim != 0xFFFFFFFFu;
        const uint32_t rec = hit ? sh->rec[tid] : 0u;
        const uint32_t t = !hit ? __float_as_uint(tmax)
                                : ((rec & kNegZero) ? kNegZero : __float_as_uint(t_value((uint32_t)(k >> 32))));
        h[0] = make_uint2(hit ? inst : 0xFFFFFFFFu, prim);
        h[1] = hit ? make_uint2(__float_as_uint(sh->u[tid]), __float_as_uint(sh->v[tid])) : make_uint2(0u, 0u);
        if constexpr (kQuery) h[2] = make_uint2(!hit ? Mode::kMiss : ((rec & 1u) ? Mode::kProcedural : Mode::kSurface), t);
        else h[2] = make_uint2(t, hit && P.hit_record ? (rec & ~kNegZero) : 0u);
    }

    // The result of a finished ray (two-level closest hits were written as instances were left).
    __device__ __forceinline__ void write(const Params &P) const {
        if (ANY) reinterpret_cast<uint8_t *>(Mode::out(P, batch))[ray] = any_hit ? 1u : 0u;
        else if (!TWO) store_hit(P, sh->key[tid], 0u);
        else if (!any_hit) store_hit(P, kMissKey, 0u);
    }

    // Traces the first `count` rays of the launch's queue with this wave and the launch's others;
    // returns the rounds of handing out rays.
    __device__ __forceinline__ uint64_t trace_queue(const Params &P, uint32_t count) {
        uint64_t rounds = 0;
        // Fetching: the queue is split into kFetchSegments contiguous segments, one per XCD
        // (workgroups are dealt to the XCDs round-robin, so block b runs on XCD b mod 8), each with a
        // slot counter on its own cache line. A wave claims `chunk` slots of its segment per atomic
        // and hands them to its idle lanes from that pool; when the segment is used up it takes
        // slots from the others. One counter address serialises its atomics (about 85M/s), so a
        // per-round atomic on one counter would cap the launch; a segment per XCD also keeps each
        // XCD's L2 on one region of a sorted queue.
        // fetch_chunk 0 claims exactly the slots the idle lanes need (the narrowest window of the
        // queue in flight, one atomic per refill round); fetch_segments 1 or kFetchSegments.
        const uint32_t waves = gridDim.x * (BLOCK / 64);
        const uint32_t chunk = P.fetch_chunk ? max(64u, min(P.fetch_chunk, (count / max(1u, waves * 4u)) & ~63u)) : 0u;
        const uint32_t nseg = P.fetch_segments > 1 ? kFetchSegments : 1u;
        const uint32_t seg0 = blockIdx.x % nseg;
        const bool simple = chunk == 0u && nseg == 1u;
        uint32_t pool = 0, pool_end = 0; // wave-uniform: unclaimed slots [pool, pool_end)
        bool drained = false;            // wave-uniform: every segment is used up
        bool active = false, exhausted = false;
        if (P.lanes != 0u) {
            // every ray has a lane: wave w takes the slots [w lanes, w lanes + lanes) of the queue, with
            // w counted XCD by XCD (block b runs on XCD b mod 8), so that each XCD has its own part
            const uint32_t per_xcd = gridDim.x / kFetchSegments;
            const uint32_t b = (blockIdx.x % kFetchSegments) * per_xcd + blockIdx.x / kFetchSegments;
            const uint64_t w = (uint64_t)b * (BLOCK / 64) + (tid >> 6);
            const uint64_t my = w * P.lanes + lane;
            drained = exhausted = true;
            if (lane < P.lanes && my < count) {
                uint32_t bt, r;
                Mode::locate(P, P.order ? P.order[my] : (uint32_t)my, bt, r);
                start(P, bt, r);
                active = true;
            }
        }
        for (;;) {
            const uint64_t need = __ballot(!active && !exhausted);
            if (need) {
                const uint32_t n_need = (uint32_t)__popcll(need);
                const uint32_t rank = (uint32_t)__popcll(need & ((1ull << lane) - 1ull));
                const uint32_t avail = pool_end - pool;
                uint32_t my = rank < avail ? pool + rank : 0xFFFFFFFFu; // lanes served by the pool
                if (simple) {
                    // one counter, exactly the slots the idle lanes need
                    const uint32_t leader = (uint32_t)__ffsll((long long)need) - 1u;
                    uint32_t b = 0;
                    if (lane == leader) b = atomicAdd(P.ray_counter, n_need);
                    b = __builtin_amdgcn_readlane(b, (int)leader);
                    my = b + rank;
                    drained = b + n_need >= count;
                } else if (avail >= n_need) {
                    pool += n_need;
                } else if (drained) {
                    pool = pool_end;
                } else {
                    // refill: the leader claims a chunk of this XCD's segment, else of another one
                    const uint32_t leader = (uint32_t)__ffsll((long long)need) - 1u;
                    uint32_t nb = 0, ne = 0;
                    if (lane == leader) {
                        const uint32_t claim = chunk ? chunk : n_need - avail;
                        for (uint32_t k = 0; k < nseg; k++) {
                            const uint32_t s = (seg0 + k) % nseg;
                            const uint32_t lo = (uint32_t)((uint64_t)count * s / nseg);
                            const uint32_t hi = (uint32_t)((uint64_t)count * (s + 1) / nseg);
                            if (lo == hi) continue;
                            const uint32_t b = atomicAdd(P.ray_counter + s * kCounterStride, claim);
                            if (b < hi - lo) {
                                nb = lo + b;
                                ne = lo + min(b + claim, hi - lo);
                                break;
                            }
                        }
                    }
                    nb = __builtin_amdgcn_readlane(nb, (int)leader); // wave-uniform from here on
                    ne = __builtin_amdgcn_readlane(ne, (int)leader);
                    drained = nb == ne;
                    if (rank >= avail && rank - avail < ne - nb) my = nb + (rank - avail);
                    pool = nb + min(n_need - avail, ne - nb);
                    pool_end = ne;
                }
                if (!active && !exhausted) {
                    if (my < count) {
                        uint32_t b, r;
                        Mode::locate(P, P.order ? P.order[my] : my, b, r); // sorted queue: fetch in key order
                        start(P, b, r);
                        active = true;
                    } else if (drained) {
                        exhausted = true; // no slot left in any segment (else: retry next round)
                    }
                }
            }
            if (!__any(active)) break;
            if (COUNT && lane == (uint32_t)__ffsll((long long)__ballot(1)) - 1u) rounds++;
            run(P, active, !drained);
            if (active && finished()) {
                if (!COUNT) write(P); // the counting form has no output buffers (out is null)
                active = false;
            }
        }
        return rounds;
    }
};

} // namespace trav
} // namespace lchip
