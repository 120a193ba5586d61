// oct_walker.h -- BVH8 traversal with eight lanes per ray, for launches of so few rays that a wave runs
// alone on its SIMD and a ray's chain of steps is all the time there is (trace.hip). Same semantics
// and node format as Walker (traverse.h).
//
// The eight lanes of a ray hold the same state and take the same steps. In a node, lane k tests child
// k and, if that is a leaf slot the ray reaches, its triangles; the masks and the nearest hit are
// settled across the eight by a ballot and DPP moves. A lone wave issues one VALU instruction per
// 8 cycles, whatever its lanes do, so the ~320 instructions of a node step of one ray per lane cost
// more than its memory latency; here a node step takes ~110 and its triangles follow at once.
#pragma once

#include "wave_walker.h"

namespace lchip {
namespace trav {

constexpr int kOctStack = 24; // stack entries in LDS per ray

// Moves within groups of eight lanes: pairs, quads, then the half-row mirror (lane i and 7 - i).
template<int CTRL>
__device__ __forceinline__ uint32_t oct_move(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t oct_or(uint32_t v) {
    v |= oct_move<0xB1>(v);
    v |= oct_move<0x4E>(v);
    return v | oct_move<0x141>(v);
}
template<int CTRL>
__device__ __forceinline__ unsigned long long oct_min_step(unsigned long long v) {
    const unsigned long long w = ((unsigned long long)oct_move<CTRL>((uint32_t)(v >> 32)) << 32) | oct_move<CTRL>((uint32_t)v);
    return w < v ? w : v;
}
__device__ __forceinline__ unsigned long long oct_min(unsigned long long v) {
    return oct_min_step<0x141>(oct_min_step<0x4E>(oct_min_step<0xB1>(v)));
}

template<bool ANY, bool TWO>
struct OctWalker {
    uint2 (*stk)[8];      // [kOctStack][ray of the wave]
    uint32_t k, group;    // child of this lane, ray of the wave
    int sp, floor;
    RaySetup R;
    float tmin, tmax, t_best, bu, bv;
    uint32_t b_prim, b_inst, b_rec, batch, ray, cur_inst;
    bool any_hit;
    uint32_t g_base, g_mask, t_base, t_mask;
    const WideNode *nodes;
    const TriRecord *tris;

    static constexpr uint32_t kWorld = 0xFFFFFFFFu;

    // As Walker: the host sizes spill_depth (from at most 24 LDS entries) by the built depths. One area
    // per ray (TraceGrid::spill_areas); queues counted on the device have the areas of 64 lanes per wave.
    __device__ __forceinline__ uint2 *spill_at(const TraceParams &P, int e) const {
        return P.spill + ((uint64_t)blockIdx.x * (P.octets ? P.lanes : 8u) + group) * P.spill_depth + e;
    }
    __device__ __forceinline__ void push(const TraceParams &P, uint2 e) {
        if (sp < kOctStack) stk[sp][group] = e; // the eight lanes store the same value
        else if ((uint32_t)(sp - kOctStack) < P.spill_depth) *spill_at(P, sp - kOctStack) = e;
        else atomicOr(P.error, 1u);
        sp++;
    }
    __device__ __forceinline__ uint2 pop(const TraceParams &P) {
        sp--;
        if (sp < kOctStack) return stk[sp][group];
        if ((uint32_t)(sp - kOctStack) < P.spill_depth) return *spill_at(P, sp - kOctStack);
        return make_uint2(0u, 0u);
    }
    __device__ __forceinline__ void load_ray(const TraceParams &P, float o[3], float d[3]) {
        const float4 *rays = P.batches.b[batch].rays;
        const float4 r0 = rays[2 * (uint64_t)ray], r1 = rays[2 * (uint64_t)ray + 1];
        o[0] = r0.x; o[1] = r0.y; o[2] = r0.z; tmin = r0.w;
        d[0] = r1.x; d[1] = r1.y; d[2] = r1.z; tmax = r1.w;
    }

    __device__ __forceinline__ void start(const TraceParams &P, uint32_t q) {
        const Geometry &G = P.geo;
        batch = find_batch(P.batches, q);
        ray = q - P.batches.b[batch].start;
        t_best = FLT_MAX * 2.0f; // +inf
        bu = bv = 0.0f;
        b_prim = b_inst = 0xFFFFFFFFu;
        b_rec = 0u;
        any_hit = false;
        sp = floor = 0;
        t_base = t_mask = g_base = 0u;
        float o[3], d[3];
        load_ray(P, o, d);
        bool misses = G.empty != 0u;
        if (TWO) {
            cur_inst = kWorld;
            nodes = G.tlas_nodes;
            tris = nullptr;
            for (int a = 0; a < 3; a++) { R.o[a] = o[a]; R.d[a] = d[a]; }
        } else {
            cur_inst = 0u;
            nodes = G.blas_nodes;
            tris = G.blas_tris;
            xform_point(G.inst_inv, o, R.o);
            xform_vector(G.inst_inv, d, R.d);
            misses = misses || (G.inst_mask & P.batches.b[batch].mask & 0xFFu) == 0u;
        }
        ray_setup(R);
        g_mask = misses ? 0u : ((1u << R.oct) | (1u << 8));
    }

    // Enters the next instance of the TLAS leaf that takes part; false when none is left.
    __device__ __forceinline__ bool enter(const TraceParams &P) {
        const Geometry &G = P.geo;
        while (t_mask != 0u) {
            const uint32_t id = G.tlas_prims[t_base + (uint32_t)__builtin_ctz(t_mask)];
            t_mask &= t_mask - 1u;
            const InstanceRecord *ir = G.instances + id;
            const uint64_t bn = ir->blas_nodes;
            if (bn == 0u || (ir->vis_mask & P.batches.b[batch].mask & 0xFFu) == 0u || (ir->flags & kInstProcedural)) continue;
            if ((g_mask & 0xFFu) != 0u) push(P, make_uint2(g_base, g_mask));
            if (t_mask != 0u) push(P, make_uint2(t_base, t_mask | kInstGroup));
            t_mask = 0u;
            float o[3], d[3];
            load_ray(P, o, d);
            xform_point(ir->inv, o, R.o);
            xform_vector(ir->inv, d, R.d);
            ray_setup(R);
            nodes = reinterpret_cast<const WideNode *>(bn);
            tris = reinterpret_cast<const TriRecord *>(ir->blas_tris);
            cur_inst = id;
            floor = sp;
            g_base = 0u;
            g_mask = (1u << R.oct) | (1u << 8);
            return true;
        }
        return false;
    }

    // Brings a node group into (g_base, g_mask); false when the ray is finished.
    __device__ __forceinline__ bool next_group(const TraceParams &P) {
        bool world = !TWO || cur_inst == kWorld; // R and nodes are those of the TLAS
        for (;;) {
            if (TWO && t_mask != 0u) { // instances of the TLAS leaf just visited or popped
                if (enter(P)) return true;
                if (world && (g_mask & 0xFFu) != 0u) return true;
            }
            if (TWO && cur_inst != kWorld && sp == floor) { // the instance's nodes are used up
                cur_inst = kWorld;
                floor = 0;
            }
            if (sp == floor) return false;
            const uint2 e = pop(P);
            if (TWO && (e.y & kInstGroup)) {
                g_mask = 0u;
                t_base = e.x;
                t_mask = e.y & ~kInstGroup;
                continue;
            }
            g_base = e.x;
            g_mask = e.y;
            if (TWO && cur_inst == kWorld && !world) { // back in the TLAS
                float o[3], d[3];
                load_ray(P, o, d);
                for (int a = 0; a < 3; a++) { R.o[a] = o[a]; R.d[a] = d[a]; }
                ray_setup(R);
                nodes = P.geo.tlas_nodes;
            }
            return true;
        }
    }

    // Visits the next node of the group and tests the triangles of the leaf slots the ray reaches.
    __device__ __forceinline__ void visit(const TraceParams &P) {
        uint32_t hm = g_mask & 0xFFu;
        const uint32_t im = (g_mask >> 8) & 0xFFu;
        const uint32_t i = (uint32_t)__builtin_ctz(hm);
        hm &= hm - 1u;
        const uint32_t slot = i ^ R.oct;
        const WideNode *node = nodes + (g_base + (uint32_t)__popc(im & ((1u << slot) - 1u)));
        const uint4 w0 = reinterpret_cast<const uint4 *>(node)[0], w1 = reinterpret_cast<const uint4 *>(node)[1];
        const unsigned char *plane = reinterpret_cast<const unsigned char *>(node) + 32 + k; // lo x y z, hi x y z, 8 B apart
        const float q[6] = {(float)plane[0], (float)plane[8], (float)plane[16], (float)plane[24], (float)plane[32], (float)plane[40]};
        if (hm != 0u) push(P, make_uint2(g_base, hm | (im << 8)));
        const float tcull = ANY ? tmax : fminf(tmax, t_best);
        const float p[3] = {__uint_as_float(w0.x), __uint_as_float(w0.y), __uint_as_float(w0.z)};
        float tn = tmin, tf = tcull;
        for (int a = 0; a < 3; a++) {
            const float s = __uint_as_float(((w0.w >> (8 * a)) & 0xFFu) << 23) * R.inv[a];
            const float b = (p[a] - R.o[a]) * R.inv[a];
            // a plane's distance q s + b: the errors of s, b and the FMA stay below 8 units of 2^-24
            // (256|s| + |b|); the slack of 16 such units keeps the test conservative (intersect_node)
            const float e = 0x1p-20f * (256.0f * fabsf(s) + fabsf(b));
            const bool neg = R.inv[a] < 0.0f;
            tn = fmaxf(tn, __builtin_fmaf(neg ? q[3 + a] : q[a], s, b - e));
            tf = fminf(tf, __builtin_fmaf(neg ? q[a] : q[3 + a], s, b + e));
        }
        const bool reached = tn <= tf;
        const uint32_t hits = (uint32_t)(__ballot(reached) >> (8u * group)) & 0xFFu;
        const uint32_t nim = w0.w >> 24;
        g_base = w1.x;
        g_mask = permute8(hits & nim, R.oct) | (nim << 8);
        if ((hits & ~nim) == 0u) return;
        const uint32_t meta = ((k < 4u ? w1.z : w1.w) >> (8u * (k & 3u))) & 0xFFu;
        const uint32_t cnt = reached && !((nim >> k) & 1u) ? meta >> 5 : 0u, first = meta & 31u;
        if (TWO && cur_inst == kWorld) { // instances: entered one after another
            t_base = w1.y;
            t_mask = oct_or(((1u << cnt) - 1u) << first);
            return;
        }
        unsigned long long key = ~0ull;
        float ht = 0.0f, hu = 0.0f, hv = 0.0f;
        uint32_t hrec = 0u;
        for (uint32_t j = 0; j < cnt; j++) {
            const uint32_t rec = w1.y + first + j;
            const float4 *tr = reinterpret_cast<const float4 *>(tris + rec);
            const float4 v0 = tr[0], v1 = tr[1], v2 = tr[2];
            float t, u, v;
            if (wt_intersect(R, v0, v1, v2, tmin, tmax, t, u, v)) {
                const unsigned long long kk = ((unsigned long long)t_order(t) << 32) | __float_as_uint(v0.w);
                if (kk < key) {
                    key = kk;
                    ht = t; hu = u; hv = v;
                    hrec = rec;
                }
            }
        }
        // the nearest of the eight lanes' hits (this is uniform over the ray's lanes)
        if (((__ballot(key != ~0ull) >> (8u * group)) & 0xFFull) == 0ull) return;
        if (ANY) {
            any_hit = true;
            g_mask = 0u;
            sp = floor = 0;
            if (TWO) cur_inst = kWorld;
            return;
        }
        const unsigned long long low = oct_min(key);
        const uint32_t win = (uint32_t)__builtin_ctz((uint32_t)(__ballot(key == low) >> (8u * group)) & 0xFFu);
        const uint32_t from = (8u * group + win) << 2;
        const float t = from_lane(from, ht), u = from_lane(from, hu), v = from_lane(from, hv);
        const uint32_t rec = from_lane(from, hrec), prim = (uint32_t)low;
        if (nearer(t, cur_inst, prim, t_best, b_inst, b_prim)) {
            t_best = t; bu = u; bv = v;
            b_prim = prim; b_inst = cur_inst; b_rec = rec;
        }
    }

    __device__ __forceinline__ void write(const TraceParams &P) const {
        char *out = static_cast<char *>(P.batches.b[batch].out);
        if (ANY) {
            reinterpret_cast<uint8_t *>(out)[ray] = any_hit ? 1u : 0u;
            return;
        }
        uint2 *h = reinterpret_cast<uint2 *>(out + 24ull * ray);
        const bool hit = b_prim != 0xFFFFFFFFu;
        h[0] = make_uint2(hit ? b_inst : 0xFFFFFFFFu, b_prim);
        h[1] = make_uint2(hit ? __float_as_uint(bu) : 0u, hit ? __float_as_uint(bv) : 0u);
        h[2] = make_uint2(__float_as_uint(hit ? t_best : tmax), hit && P.hit_record ? b_rec : 0u);
    }
};

// Wave w of the launch traces the `rays` queue slots from w x rays on.
template<bool ANY, bool TWO>
__device__ __forceinline__ void trace_octets(const TraceParams &P, uint2 (*stk)[8], uint32_t w, uint32_t rays, uint32_t count) {
    OctWalker<ANY, TWO> W;
    W.stk = stk;
    W.k = threadIdx.x & 7u;
    W.group = threadIdx.x >> 3;
    const uint64_t my = (uint64_t)w * rays + W.group;
    if (W.group >= rays || my >= count) return;
    W.start(P, P.order ? P.order[my] : (uint32_t)my);
    for (;;) {
        if (((W.g_mask & 0xFFu) == 0u || (TWO && W.t_mask != 0u)) && !W.next_group(P)) break;
        W.visit(P);
    }
    if (W.k == 0u) W.write(P);
}

} // namespace trav
} // namespace lchip
