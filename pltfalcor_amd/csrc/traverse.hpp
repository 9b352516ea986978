// Software ray traversal for CDNA4: BVH4 with the four child boxes in the parent as SoA rows (one
// 128 B node = eight independent 16 B loads tests four boxes, so a level costs one memory latency),
// triangles re-ordered into leaf order as 48 B records (v0 + triangle id, v1, v2), two of which are
// tested per trip, and a per-lane traversal stack: its first kTraversalStackDepth
// entries in LDS laid out [depth][lane] (a wave's pushes/pops hit 64 distinct banks), the rest in
// private memory (scratch), touched only by rays deep in very deep trees.
//
// Hit results are independent of the tree: the watertight test (Woop, Benthin, Wald 2013,
// "Watertight Ray/Triangle Intersection", JCGT 2(1)) runs with FP contraction off and a double
// fallback on zero edge functions, box tests are conservative (far distance widened by
// 1 + 2*gamma(3), Ize 2013 "Robust BVH Ray Traversal"), and equal distances resolve to the
// smallest triangle id. The CPU oracle uses the same arithmetic, so hit ids are bit-exact.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace plt {

struct Ray {
    float ox, oy, oz, dx, dy, dz, tmin, tmax;
};
struct Hit {
    uint32_t tri;  // 0xFFFFFFFF = miss
    float b1, b2, t;
};

struct TraceScene {
    const float4* __restrict__ nodes;  // 8 per node (BvhNode)
    const float4* __restrict__ tris;   // 3 per triangle in leaf order
    uint32_t n_nodes;
};

constexpr uint32_t kNoHit = 0xFFFFFFFFu;

// Watertight ray/triangle state: axis permutation and shear constants.
struct RayPrep {
    int kx, ky, kz;
    float Sx, Sy, Sz;
    float o[3];
};

__device__ __forceinline__ float pick3(float x, float y, float z, int k) { return k == 0 ? x : (k == 1 ? y : z); }

__device__ __forceinline__ RayPrep prep_ray(const Ray& r) {
#pragma clang fp contract(off)
    RayPrep p;
    const float ax = fabsf(r.dx), ay = fabsf(r.dy), az = fabsf(r.dz);
    p.kz = ax > ay ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    p.kx = p.kz == 2 ? 0 : p.kz + 1;
    p.ky = p.kx == 2 ? 0 : p.kx + 1;
    const float dkz = pick3(r.dx, r.dy, r.dz, p.kz);
    if (dkz < 0.f) { const int t = p.kx; p.kx = p.ky; p.ky = t; }
    p.Sx = pick3(r.dx, r.dy, r.dz, p.kx) / dkz;
    p.Sy = pick3(r.dx, r.dy, r.dz, p.ky) / dkz;
    p.Sz = 1.f / dkz;
    p.o[0] = r.ox; p.o[1] = r.oy; p.o[2] = r.oz;
    return p;
}

// Returns true and (t, b1, b2) when the ray hits the triangle with tmin <= t <= tmax.
__device__ __forceinline__ bool intersect_tri(const RayPrep& p, float4 v0, float4 v1, float4 v2, float tmin, float tmax, float& t_out, float& b1,
                                              float& b2) {
#pragma clang fp contract(off)
    const float Ak = pick3(v0.x, v0.y, v0.z, p.kx) - pick3(p.o[0], p.o[1], p.o[2], p.kx);
    const float Al = pick3(v0.x, v0.y, v0.z, p.ky) - pick3(p.o[0], p.o[1], p.o[2], p.ky);
    const float Az0 = pick3(v0.x, v0.y, v0.z, p.kz) - pick3(p.o[0], p.o[1], p.o[2], p.kz);
    const float Bk = pick3(v1.x, v1.y, v1.z, p.kx) - pick3(p.o[0], p.o[1], p.o[2], p.kx);
    const float Bl = pick3(v1.x, v1.y, v1.z, p.ky) - pick3(p.o[0], p.o[1], p.o[2], p.ky);
    const float Bz0 = pick3(v1.x, v1.y, v1.z, p.kz) - pick3(p.o[0], p.o[1], p.o[2], p.kz);
    const float Ck = pick3(v2.x, v2.y, v2.z, p.kx) - pick3(p.o[0], p.o[1], p.o[2], p.kx);
    const float Cl = pick3(v2.x, v2.y, v2.z, p.ky) - pick3(p.o[0], p.o[1], p.o[2], p.ky);
    const float Cz0 = pick3(v2.x, v2.y, v2.z, p.kz) - pick3(p.o[0], p.o[1], p.o[2], p.kz);
    const float Ax = Ak - p.Sx * Az0, Ay = Al - p.Sy * Az0;
    const float Bx = Bk - p.Sx * Bz0, By = Bl - p.Sy * Bz0;
    const float Cx = Ck - p.Sx * Cz0, Cy = Cl - p.Sy * Cz0;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.f || V == 0.f || W == 0.f) {
        U = float(double(Cx) * double(By) - double(Cy) * double(Bx));
        V = float(double(Ax) * double(Cy) - double(Ay) * double(Cx));
        W = float(double(Bx) * double(Ay) - double(By) * double(Ax));
    }
    if ((U < 0.f || V < 0.f || W < 0.f) && (U > 0.f || V > 0.f || W > 0.f)) return false;
    const float det = U + V + W;
    if (det == 0.f) return false;
    const float Az = p.Sz * Az0, Bz = p.Sz * Bz0, Cz = p.Sz * Cz0;
    const float T = U * Az + V * Bz + W * Cz;
    const float t = T / det;
    if (!(t >= tmin && t <= tmax)) return false;
    t_out = t;
    b1 = V / det;
    b2 = W / det;
    return true;
}

// Levels of 4-wide nodes that a scene's tree may have: the device builder and the upload of a host tree
// refuse more. Every node on the way down pushes at most three children.
constexpr int kMaxTreeLevels = 33;
// Traversal stack entries kept in LDS per lane (32 slots x 4 B x 64 lanes = 8 KB per one-wave block, which
// leaves LDS room for 20 blocks per CU), and the entries beyond them, in private memory.
constexpr int kTraversalStackDepth = 32;
constexpr int kTraversalSpill = 68;
static_assert(3 * kMaxTreeLevels <= kTraversalStackDepth + kTraversalSpill, "the traversal stack holds the deepest tree");

// Sorts four keys ascending (five compare-exchanges).
__device__ __forceinline__ void sort4(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) {
    uint32_t t;
    t = min(a, b); b = max(a, b); a = t;
    t = min(c, d); d = max(c, d); c = t;
    t = min(a, c); c = max(a, c); a = t;
    t = min(b, d); d = max(b, d); b = t;
    t = min(b, c); c = max(b, c); b = t;
}

// What all of a ray's box and triangle tests share.
struct RayConst {
    RayPrep p;
    float ix, iy, iz, oix, oiy, oiz, tmin;
    uint32_t sx, sy, sz;  // byte offset of each axis's near row within its two slab rows (0: lo, 16: hi)
};
__device__ __forceinline__ RayConst ray_const(const Ray& r) {
    RayConst c;
    c.p = prep_ray(r);
    const float dx = fabsf(r.dx) > 1e-30f ? r.dx : copysignf(1e-30f, r.dx);
    const float dy = fabsf(r.dy) > 1e-30f ? r.dy : copysignf(1e-30f, r.dy);
    const float dz = fabsf(r.dz) > 1e-30f ? r.dz : copysignf(1e-30f, r.dz);
    c.ix = 1.f / dx; c.iy = 1.f / dy; c.iz = 1.f / dz;
    c.oix = r.ox * c.ix; c.oiy = r.oy * c.iy; c.oiz = r.oz * c.iz;
    c.tmin = r.tmin;
    c.sx = c.ix < 0.f ? 16u : 0u; c.sy = c.iy < 0.f ? 16u : 0u; c.sz = c.iz < 0.f ? 16u : 0u;
    return c;
}
// Conservative slab test of one child box given its near and far planes (fma rounds monotonically, so
// the plane picked by the direction's sign is the one a min or max would pick): the entry distance,
// +inf on a miss. An unused slot's box [+inf, +inf] is missed whatever tmax is.
__device__ __forceinline__ float box_entry(const RayConst& c, float nx, float fx, float ny, float fy, float nz, float fz, float tmax) {
    const float tn = fmaxf(fmaxf(fmaf(nx, c.ix, -c.oix), fmaf(ny, c.iy, -c.oiy)), fmaxf(fmaf(nz, c.iz, -c.oiz), c.tmin));
    const float tf = fminf(fminf(fmaf(fx, c.ix, -c.oix), fmaf(fy, c.iy, -c.oiy)), fminf(fmaf(fz, c.iz, -c.oiz), tmax));
    return tn <= tf * 1.0000005f ? tn : __builtin_inff();
}
// Sort key of a child: the entry distance's bits (non-negative floats order as integers) with the slot
// in the low two bits; a missed box sorts last.
__device__ __forceinline__ uint32_t box_key(float entry, uint32_t slot) {
    return entry != __builtin_inff() ? ((__float_as_uint(entry) & ~3u) | slot) : 0xFFFFFFFFu;
}

// Traverses the BVH. anyHit: stop at the first hit in [tmin, tmax] (visibility rays); a per-lane
// value lets one call serve a wave whose lanes cast both kinds (whether a ray hits anything in
// [tmin, tmax] does not depend on it). `stack` points at this lane's first LDS slot; consecutive
// slots are `stride` ints apart. Children are visited nearest entry first (ties and order only
// change the speed: the closest hit is the smallest (t, triangle id) over every triangle tested,
// and boxes are conservative).
//
// A wave issues the instructions of its slowest lanes: 9 to 14 of 64 lanes are active on average in
// the frame's kernels, which are bound by VALU issue (70-84 % busy). So a trip is kept short and
// fits every lane: each lane reads 112 B, the boxes of its node or two triangles of its leaf, with
// one wait for both kinds (a leaf of four takes two trips, during which the other lanes advance,
// instead of the wave waiting for its longest leaf), and the hit children are pushed without
// branches. Against one node or one whole leaf per trip: 1,048,576 incoherent closest-hit rays over
// 1.31 M triangles 0.421 -> 0.380 ms; per 1080p frame of 5.24 M triangles sample kernel 2.78 -> 2.63,
// light sampling 2.72 -> 2.63 ms. (The two loads apart, with one triangle per trip: 0.46 ms.) The ray's
// constants and the slab test stand in the function itself: taken from RayConst and box_entry, as
// traverse_quad does, the compiler moved the loads into the branches (0.48 ms).
template <int kDepth>
__device__ __forceinline__ Hit traverse_rays(const TraceScene& sc, const Ray& r, int* stack, int stride, bool anyHit) {
    Hit h{kNoHit, 0.f, 0.f, r.tmax};
    const RayPrep p = prep_ray(r);
    const float dx = fabsf(r.dx) > 1e-30f ? r.dx : copysignf(1e-30f, r.dx);
    const float dy = fabsf(r.dy) > 1e-30f ? r.dy : copysignf(1e-30f, r.dy);
    const float dz = fabsf(r.dz) > 1e-30f ? r.dz : copysignf(1e-30f, r.dz);
    const float ix = 1.f / dx, iy = 1.f / dy, iz = 1.f / dz;
    const float oix = r.ox * ix, oiy = r.oy * iy, oiz = r.oz * iz;
    const uint32_t sx = ix < 0.f ? 16u : 0u, sy = iy < 0.f ? 16u : 0u, sz = iz < 0.f ? 16u : 0u;
    int spill[kTraversalSpill];
    int sp = 0;
    int node = 0;
    float best = r.tmax;
    const char* nodes = reinterpret_cast<const char*>(sc.nodes);
    const char* tris = reinterpret_cast<const char*>(sc.tris);
    auto ld = [](const char* q) { return *reinterpret_cast<const float4*>(q); };
    auto push = [&](int x) {
        if (sp < kDepth) stack[sp * stride] = x;
        else if (sp < kDepth + kTraversalSpill) spill[sp - kDepth] = x;
        ++sp;
    };
    auto pop = [&]() {
        --sp;
        node = sp < kDepth ? stack[sp * stride] : spill[sp - kDepth];
    };
    auto entry = [&](float nx, float fx, float ny, float fy, float nz, float fz) {
        const float ax = fmaf(nx, ix, -oix), bx = fmaf(fx, ix, -oix);
        const float ay = fmaf(ny, iy, -oiy), by = fmaf(fy, iy, -oiy);
        const float az = fmaf(nz, iz, -oiz), bz = fmaf(fz, iz, -oiz);
        const float tn = fmaxf(fmaxf(ax, ay), fmaxf(az, r.tmin));
        const float tf = fminf(fminf(bx, by), fminf(bz, best));
        return tn <= tf * 1.0000005f ? tn : __builtin_inff();
    };
    // the boxes of a node's children: pushes the hit ones but the nearest, which goes next
    auto boxes = [&](float4 nx, float4 fx, float4 ny, float4 fy, float4 nz, float4 fz, float4 cf) {
        const float e0 = entry(nx.x, fx.x, ny.x, fy.x, nz.x, fz.x);
        const float e1 = entry(nx.y, fx.y, ny.y, fy.y, nz.y, fz.y);
        const float e2 = entry(nx.z, fx.z, ny.z, fy.z, nz.z, fz.z);
        const float e3 = entry(nx.w, fx.w, ny.w, fy.w, nz.w, fz.w);
        // sort keys: the entry distance's bits (non-negative floats order as integers) with the
        // slot in the low two bits; a missed box sorts last
        constexpr float kInf = __builtin_inff();
        uint32_t k0 = e0 != kInf ? (__float_as_uint(e0) & ~3u) : 0xFFFFFFFFu;
        uint32_t k1 = e1 != kInf ? ((__float_as_uint(e1) & ~3u) | 1u) : 0xFFFFFFFFu;
        uint32_t k2 = e2 != kInf ? ((__float_as_uint(e2) & ~3u) | 2u) : 0xFFFFFFFFu;
        uint32_t k3 = e3 != kInf ? ((__float_as_uint(e3) & ~3u) | 3u) : 0xFFFFFFFFu;
        sort4(k0, k1, k2, k3);
        // The child references are used only when a box is hit; left to itself the compiler
        // issues their load there, after the box tests, which costs every node visit a second
        // dependent memory round trip. Requiring them in registers here keeps the load with
        // the boxes' (the empty asm emits nothing).
        asm volatile("" : : "v"(cf.x), "v"(cf.y), "v"(cf.z), "v"(cf.w));
        const int c0 = __float_as_int(cf.x), c1 = __float_as_int(cf.y), c2 = __float_as_int(cf.z), c3 = __float_as_int(cf.w);
        auto child = [&](uint32_t k) {  // selects, no branches
            const int lo = (k & 1u) ? c1 : c0, hi = (k & 1u) ? c3 : c2;
            return (k & 2u) ? hi : lo;
        };
        // the farther hit children on the stack, farthest first; the nearest next
        if (sp + 3 <= kDepth) {  // each slot is written and kept only if its child was hit
            int* top = stack + sp * stride;
            *top = child(k3);
            int n = k3 != 0xFFFFFFFFu ? 1 : 0;
            top += k3 != 0xFFFFFFFFu ? stride : 0;
            *top = child(k2);
            n += k2 != 0xFFFFFFFFu ? 1 : 0;
            top += k2 != 0xFFFFFFFFu ? stride : 0;
            *top = child(k1);
            n += k1 != 0xFFFFFFFFu ? 1 : 0;
            sp += n;
        } else {
            if (k3 != 0xFFFFFFFFu) push(child(k3));
            if (k2 != 0xFFFFFFFFu) push(child(k2));
            if (k1 != 0xFFFFFFFFu) push(child(k1));
        }
        node = child(k0);
        return k0 != 0xFFFFFFFFu;
    };
    auto tri = [&](float4 v0, float4 v1, float4 v2) {
        float tt, b1, b2;
        if (intersect_tri(p, v0, v1, v2, r.tmin, best, tt, b1, b2)) {
            const uint32_t id = __float_as_uint(v0.w);
            if (tt < best || id < h.tri) {
                best = tt;
                h.tri = id; h.b1 = b1; h.b2 = b2; h.t = tt;
            }
        }
    };
    while (true) {
        bool next = false;  // node holds the next thing to visit; otherwise it comes off the stack
        const bool inner = node >= 0;
        const uint32_t leaf = uint32_t(~node);
        const bool two = (leaf & 7u) != 0u;
        // a node's slab rows by the direction's signs, or triangles 0 and 1 (0 again if there is one)
        const char* A = inner ? nodes + 128 * size_t(uint32_t(node)) : tris + 48 * size_t(leaf >> 3);
        const uint32_t ox = inner ? sx : 0u, oy = inner ? sy : 0u, oz = inner ? sz : 0u;
        const char* B = (inner || two) ? A : A - 48;
        const float4 q0 = ld(A + ox), q1 = ld(A + (16u - ox)), q2 = ld(A + (32u + oy));
        const float4 q3 = ld(B + (48u - oy)), q4 = ld(B + (64u + oz)), q5 = ld(B + (80u - oz));
        const float4 q6 = ld(inner ? A + 96 : A);
        if (inner) {
            next = boxes(q0, q1, q2, q3, q4, q5, q6);
        } else {
            tri(q0, q1, q2);
            if (two && !(anyHit && h.tri != kNoHit)) tri(q3, q4, q5);
            if (anyHit && h.tri != kNoHit) return h;
            if ((leaf & 7u) > 1u) {  // the rest of the leaf: two triangles on, two fewer
                node = ~int(leaf + 14u);
                next = true;
            }
        }
        if (!next) {
            if (sp == 0) break;
            pop();
        }
    }
    return h;
}
// The same slab test without the direction's signs.
__device__ __forceinline__ float box_entry_minmax(float lox, float hix, float loy, float hiy, float loz, float hiz, float ix,
                                           float iy, float iz, float oix, float oiy, float oiz, float tmin, float tmax) {
    const float tx0 = fmaf(lox, ix, -oix), tx1 = fmaf(hix, ix, -oix);
    const float ty0 = fmaf(loy, iy, -oiy), ty1 = fmaf(hiy, iy, -oiy);
    const float tz0 = fmaf(loz, iz, -oiz), tz1 = fmaf(hiz, iz, -oiz);
    const float tn = fmaxf(fmaxf(fminf(tx0, tx1), fminf(ty0, ty1)), fmaxf(fminf(tz0, tz1), tmin));
    const float tf = fminf(fminf(fmaxf(tx0, tx1), fmaxf(ty0, ty1)), fminf(fmaxf(tz0, tz1), tmax));
    return tn <= tf * 1.0000005f ? tn : __builtin_inff();
}

// The same traversal with one node or one whole leaf per trip, for small trees and for kernels that spill
// registers: it holds fewer of them across a trip. The solve megakernel (128 VGPRs and 1.2-1.5 KB of scratch
// per lane) takes 2.82 ms with it and 2.92 ms with traverse_rays (512 x 512, depth 6, 1.31 M triangles).
template <int kDepth>
__device__ __forceinline__ Hit traverse_rays_lean(const TraceScene& sc, const Ray& r, int* stack, int stride, bool anyHit) {
    Hit h{kNoHit, 0.f, 0.f, r.tmax};
    const RayPrep p = prep_ray(r);
    const float dx = fabsf(r.dx) > 1e-30f ? r.dx : copysignf(1e-30f, r.dx);
    const float dy = fabsf(r.dy) > 1e-30f ? r.dy : copysignf(1e-30f, r.dy);
    const float dz = fabsf(r.dz) > 1e-30f ? r.dz : copysignf(1e-30f, r.dz);
    const float ix = 1.f / dx, iy = 1.f / dy, iz = 1.f / dz;
    const float oix = r.ox * ix, oiy = r.oy * iy, oiz = r.oz * iz;
    int spill[kTraversalSpill];
    int sp = 0;
    int node = 0;
    float best = r.tmax;
    auto push = [&](int x) {
        if (sp < kDepth) stack[sp * stride] = x;
        else if (sp < kDepth + kTraversalSpill) spill[sp - kDepth] = x;
        ++sp;
    };
    while (true) {
        if (node >= 0) {
            const float4* q = sc.nodes + 8 * node;
            const float4 lox = q[0], hix = q[1], loy = q[2], hiy = q[3], loz = q[4], hiz = q[5], cf = q[6];
            const float e0 = box_entry_minmax(lox.x, hix.x, loy.x, hiy.x, loz.x, hiz.x, ix, iy, iz, oix, oiy, oiz, r.tmin, best);
            const float e1 = box_entry_minmax(lox.y, hix.y, loy.y, hiy.y, loz.y, hiz.y, ix, iy, iz, oix, oiy, oiz, r.tmin, best);
            const float e2 = box_entry_minmax(lox.z, hix.z, loy.z, hiy.z, loz.z, hiz.z, ix, iy, iz, oix, oiy, oiz, r.tmin, best);
            const float e3 = box_entry_minmax(lox.w, hix.w, loy.w, hiy.w, loz.w, hiz.w, ix, iy, iz, oix, oiy, oiz, r.tmin, best);
            // sort keys: the entry distance's bits (non-negative floats order as integers) with the
            // slot in the low two bits; a missed box sorts last
            constexpr float kInf = __builtin_inff();
            uint32_t k0 = e0 != kInf ? (__float_as_uint(e0) & ~3u) : 0xFFFFFFFFu;
            uint32_t k1 = e1 != kInf ? ((__float_as_uint(e1) & ~3u) | 1u) : 0xFFFFFFFFu;
            uint32_t k2 = e2 != kInf ? ((__float_as_uint(e2) & ~3u) | 2u) : 0xFFFFFFFFu;
            uint32_t k3 = e3 != kInf ? ((__float_as_uint(e3) & ~3u) | 3u) : 0xFFFFFFFFu;
            sort4(k0, k1, k2, k3);
            asm volatile("" : : "v"(cf.x), "v"(cf.y), "v"(cf.z), "v"(cf.w));
            if (k0 != 0xFFFFFFFFu) {
                const int c0 = __float_as_int(cf.x), c1 = __float_as_int(cf.y), c2 = __float_as_int(cf.z), c3 = __float_as_int(cf.w);
                auto child = [&](uint32_t k) {  // selects, no branches
                    const int lo = (k & 1u) ? c1 : c0, hi = (k & 1u) ? c3 : c2;
                    return (k & 2u) ? hi : lo;
                };
                // the farther hit children on the stack, farthest first; the nearest next
                if (k3 != 0xFFFFFFFFu) push(child(k3));
                if (k2 != 0xFFFFFFFFu) push(child(k2));
                if (k1 != 0xFFFFFFFFu) push(child(k1));
                node = child(k0);
                continue;
            }
        } else {
            const uint32_t leaf = uint32_t(~node);
            const uint32_t start = leaf >> 3, cnt = (leaf & 7u) + 1u;
            const float4* t = sc.tris + 3 * size_t(start);
            float4 v0 = t[0], v1 = t[1], v2 = t[2];
            for (uint32_t i = 0; i < cnt; ++i) {
                float4 w0 = v0, w1 = v1, w2 = v2;
                if (i + 1 < cnt) {  // the next triangle's fetch overlaps this test
                    w0 = t[3 * (i + 1) + 0];
                    w1 = t[3 * (i + 1) + 1];
                    w2 = t[3 * (i + 1) + 2];
                }
                float tt, b1, b2;
                if (intersect_tri(p, v0, v1, v2, r.tmin, best, tt, b1, b2)) {
                    const uint32_t id = __float_as_uint(v0.w);
                    if (tt < best || id < h.tri) {
                        best = tt;
                        h.tri = id; h.b1 = b1; h.b2 = b2; h.t = tt;
                        if (anyHit) return h;
                    }
                }
                v0 = w0; v1 = w1; v2 = w2;
            }
        }
        if (sp == 0) break;
        --sp;
        node = sp < kDepth ? stack[sp * stride] : spill[sp - kDepth];
    }
    return h;
}
// Closest hits in a tree of few nodes, whose memory round trips the caches shorten and whose paths have
// few trips to share, are faster with the leaner loop; any-hit rays are not. The sample kernel at 569 x 512
// (traverse_rays, lean): 100 nodes 0.215, 0.197 ms; 1,153: 0.309, 0.291; 3,234: 0.429, 0.419; 5,108: 0.495,
// 0.488; 7,062: 0.524, 0.526; 10,126: 0.537, 0.545; 212,000: 0.700, 0.791. 1,048,576 rays: 1,153 nodes 167,
// 156 us; 3,234: 233, 231; 5,108: 268, 273. The tree is the launch's, so a wave takes one loop.
constexpr uint32_t kSmallTree = 4096;
template <bool kAnyHit, int kDepth, bool kLean = false>
__device__ __forceinline__ Hit traverse(const TraceScene& sc, const Ray& r, int* stack, int stride) {
    if (kLean || (!kAnyHit && sc.n_nodes < kSmallTree)) return traverse_rays_lean<kDepth>(sc, r, stack, stride, kAnyHit);
    return traverse_rays<kDepth>(sc, r, stack, stride, kAnyHit);
}

// ---------------------------------------------------------------------------------------
// One ray per quad of lanes: lane i of the quad tests child i of a node and triangles i and i + 4 of a
// leaf (the host builder's have up to eight).
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t quad_xor1(uint32_t v) { return uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0xB1, 0xF, 0xF, true)); }
__device__ __forceinline__ uint32_t quad_xor2(uint32_t v) { return uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x4E, 0xF, 0xF, true)); }
__device__ __forceinline__ uint32_t quad_xor3(uint32_t v) { return uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x1B, 0xF, 0xF, true)); }
__device__ __forceinline__ uint32_t quad_first(uint32_t v) { return uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x00, 0xF, 0xF, true)); }
// Stack entries of a quad's traversal, all in LDS, interleaved over the wave's 16 quads ([entry][quad]).
// Its pushes are not checked.
constexpr int kQuadStack = 3 * kMaxTreeLevels;
constexpr int kQuads = 16;

// The hit traverse_rays finds for the same ray, cast by the four lanes of a quad together (the ray is
// the same in all four, and so is the control flow; the result is too). `stack` points at the quad's
// first slot; its lanes read what the others wrote, in one wave's program order, so the accesses are
// wavefront-scope atomics (plain LDS instructions that the compiler neither merges nor moves).
__device__ __forceinline__ Hit traverse_quad(const TraceScene& sc, const Ray& r, int* stack, bool anyHit) {
    const RayConst c = ray_const(r);
    const uint32_t sub = __lane_id() & 3u, shift = __lane_id() & 60u;
    const uint32_t onx = (c.sx >> 2) + sub, ofx = 4u - (c.sx >> 2) + sub;
    const uint32_t ony = 8u + (c.sy >> 2) + sub, ofy = 12u - (c.sy >> 2) + sub;
    const uint32_t onz = 16u + (c.sz >> 2) + sub, ofz = 20u - (c.sz >> 2) + sub;
    const float* nodes = reinterpret_cast<const float*>(sc.nodes);
    Hit h{kNoHit, 0.f, 0.f, r.tmax};
    int node = 0, sp = 0;
    for (;;) {
        bool next = false;
        if (node >= 0) {
            const float* q = nodes + 32 * size_t(uint32_t(node));
            const float nx = q[onx], fx = q[ofx], ny = q[ony], fy = q[ofy], nz = q[onz], fz = q[ofz];
            const uint32_t child = __float_as_uint(q[24u + sub]);
            const uint32_t key = box_key(box_entry(c, nx, fx, ny, fy, nz, fz, h.t), sub);
            const bool in = key != 0xFFFFFFFFu;
            // how many children are nearer: 0 goes next, the others on the stack, farthest first
            const uint32_t rank = (quad_xor1(key) < key ? 1u : 0u) + (quad_xor2(key) < key ? 1u : 0u) + (quad_xor3(key) < key ? 1u : 0u);
            const int hits = __popc(uint32_t(__ballot(in) >> shift) & 15u);
            if (in && rank != 0u)
                __hip_atomic_store(stack + (sp + hits - 1 - int(rank)) * kQuads, int(child), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            uint32_t sel = in && rank == 0u ? child : 0u;
            sel |= quad_xor1(sel);
            sel |= quad_xor2(sel);
            if (hits > 0) {
                node = int(sel);
                sp += hits - 1;
                next = true;
            }
        } else {
            const uint32_t leaf = uint32_t(~node), cnt = (leaf & 7u) + 1u;
            const float4* t = sc.tris + 3 * size_t((leaf >> 3) + min(sub, cnt - 1u));
            const float4 v0 = t[0], v1 = t[1], v2 = t[2];
            Hit x{kNoHit, 0.f, 0.f, h.t};
            float tt, b1, b2;
            const bool ok = intersect_tri(c.p, v0, v1, v2, c.tmin, h.t, tt, b1, b2);
            if (ok && sub < cnt) x = Hit{__float_as_uint(v0.w), b1, b2, tt};
            if ((uint32_t(__ballot(x.tri != kNoHit) >> shift) & 15u) != 0u) {
                // the quad's smallest (t, id), against the closest hit so far
                auto better = [](Hit& a, const Hit& b) {
                    if (b.t < a.t || (b.t == a.t && b.tri < a.tri)) a = b;
                };
                auto other = [](const Hit& a, auto f) {
                    return Hit{f(a.tri), __uint_as_float(f(__float_as_uint(a.b1))), __uint_as_float(f(__float_as_uint(a.b2))),
                               __uint_as_float(f(__float_as_uint(a.t)))};
                };
                better(x, other(x, quad_xor1));
                better(x, other(x, quad_xor2));
                better(h, x);
                if (anyHit) return h;
            }
            next = (leaf & 4u) != 0u;  // more than four: the rest of the leaf is four triangles on, four fewer
            node -= 28;                // = ~(leaf + 28)
        }
        if (!next) {
            if (sp == 0) break;
            --sp;
            node = __hip_atomic_load(stack + sp * kQuads, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        }
    }
    return h;
}

}  // namespace plt
