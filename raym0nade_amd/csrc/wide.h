// The wide walk: closest and any hits of the reference's traversal, bit for
// bit, found on a compact four-wide tree in any order.
//
// The reference's result depends on its binary tree only through which leaves
// it visits.  With L(leaf) the entry distance rayInBox computes for a leaf's
// box and G(leaf) whether that box is entered at all (both independent of the
// running t_max), the reference visits a leaf for certain when G holds and L
// lies below its running t_max: the boxes of the leaf's ancestors contain the
// leaf's, and every operation of the slab test is monotone, so theirs pass
// too.  Let a walk end with closest hit t* in one leaf, t2 being the next t
// that it accepted, and let no triangle that it did not test have a
// computed t below lim(t*), somewhat more than t*.  Then
//     G(leaf)  and  t* < t2  and  L(leaf) < min(t2, lim(t*))
// proves that the reference ends with the same triangle: its t_max stays
// >= min(t2, lim(t*)) until it reaches that leaf, and > t* then, and later
// hits are no closer.  Where a triangle of one other leaf has the same t
// (doubled triangles), first_of says which leaf comes first.  The walk here tests a superset of the
// reference's boxes with cheap arithmetic (fused multiply-adds on 16-bit
// boxes, rounded outward, with margins that cover every rounding) and checks
// this certificate once per ray, on the reference's own box.  Where it fails
// -- hits of different leaves within a rounding error of each other -- the ray is walked
// again in the reference's order, by the same lane (RefWalker).  A shadow ray
// is blocked for certain when an accepted t < aim lies in a leaf with G and
// L < aim.
//
// What the walk leaves out lies beyond the closest hit so far by its box.  But
// the computed t of a triangle that the ray grazes can lie far before the box
// that holds the triangle, so boxes are grown by a bound of that error
// (WIDE_ERR) from the largest edge among the triangles below a node.  A
// triangle much larger than those around it would grow every box up to the
// root by its own edge.  A few such triangles (a ground, the walls of a room)
// are tested before the walk and left out of the growth; where there are more,
// they leave the others' bounds as they are, and the children on the way to
// them are flagged and always entered.
//
// Node, 64 B (a cache line), four children: origin on a 16-bit grid, child
// boxes as offsets from it in fp16, so a box plane costs one mixed-precision
// fused multiply-add.  Coordinates are scaled by a power of two to a scene of
// at most 30000 units.  The children of a node are
// consecutive, so a node and a two-bit number name any of them; below the
// reference's leaves one more level splits a leaf's at most 10 triangles into
// four runs with boxes of their own, which leaves two triangle tests where
// the whole leaf took eight.
//
// Why: the binary walk ran at the limit of two units at once.  On the
// incoherent 1M-triangle batch it spent 8.1 ms with the vector ALUs issuing
// 87% of the time and the texture data path busy 97% of it: every 16 bytes a
// lane loads occupies that path for a cycle of its compute unit, and a ray
// loaded 511 of them (88 nodes of 64 B, 61 triangles of 48 B).  Here, before
// boxes were grown, it loaded 287 (46 nodes, 18 runs), and 44 of a wave's 64
// lanes took part in a node's step instead of 30.  Before and after (us,
// launches included): 8M incoherent rays 8550 -> 5050, 8M camera rays 3280 ->
// 2930, 100k incoherent rays among 200k triangles 587 -> 338, 1M shadow rays
// 1027 -> 714; 1080p frame of 2M triangles at 16 spp 106 -> 82 ms.  (The growth
// takes 4 to 8% of these batches: up to 4% more nodes, and some 20 instructions a
// node.)  What bounds it now: the same data path (94% busy), then the vector ALUs.
#pragma once
#include "traverse.h"

namespace rm {

constexpr int WALK_WIDE = 6;     // walk kind of the render's inlined walks (beside 0, 1, 2, 4 triangles per step)
constexpr int WALK_FLAT = 7;     // walk kind: every triangle of a flat scene, else the reference-order walk
constexpr uint32_t WIDE_NONE = 0xffffffffu;

// A group of up to four sibling children still to visit, two words: x = the
// reference of the node's child 0; y = their number (bits 8-10), their child
// numbers in visiting order (bits 0-7) and a lower bound of their entry
// distances (the upper 21 bits of the float); y = 0: no group.  A walk has
// at most one group per level of the tree, and keeps its newest in registers.
constexpr uint32_t GROUP_T = 0xfffff800u;

// The walk's older groups, in the block's dynamic LDS (blocks of WALK_BLOCK
// lanes; the launch provides wide_lds_bytes), so that a wave's accesses to one
// entry are contiguous.
struct WideLds {
    uint2 *col;
    __device__ __forceinline__ void bind() {
        extern __shared__ uint32_t walk_lds[];
        col = reinterpret_cast<uint2 *>(walk_lds) + threadIdx.x;
    }
    __device__ __forceinline__ void put(int i, uint32_t x, uint32_t y) { col[i * WALK_BLOCK] = make_uint2(x, y); }
    __device__ __forceinline__ uint2 get(int i) const { return col[i * WALK_BLOCK]; }
};
// Entries and bytes of dynamic LDS per block for the walk of a tree of
// `depth` binary levels (leaves included).
inline int wide_lds_entries(int depth) { return depth > 1 ? depth / 2 : 1; }
inline size_t wide_lds_bytes(int depth) { return (size_t)wide_lds_entries(depth) * WALK_BLOCK * 8; }

// A ray in the wide tree's scaled coordinates.  A box plane p of axis i is
// crossed at p * inv[i] + nr[i] or later (as an entry) and at
// p * inv[i] + fr[i] or earlier (as an exit).
struct WideRay {
    V3 o, d;         // as given: the triangle tests use these
    float inv[3];
    float nr[3], fr[3];
    float err;       // WIDE_ERR |d| / scale: a box grows by err E distance; negative for a ray with parallel axes

    // For RefWalker, which needs the wide tree's values no more.
    __device__ __forceinline__ void reciprocals(V3 dir) {
        inv[0] = 1.0f / dir.x;
        inv[1] = 1.0f / dir.y;
        inv[2] = 1.0f / dir.z;
    }
};

// How far from a triangle the test accepts a ray: with the computed a, u, v
// and t of an accepted test, eps = 2^-24 and s = o - v0,
//     R = s - u e1 - v e2 + t d
//     a R = da s - du e1 - dv e2 + dt d
// where da..dt are the errors of the computed e1.h, s.h, d.q and e2.q (Cramer:
// without them the right side is 0).  A cross product is off by at most (2 /
// sqrt 3 + 1) eps times its factors' lengths and a dot product by 3 eps more,
// so each of the four terms is at most 5.16 eps |d| |e1| |e2| |s|; and a test
// with |a| < 1e-4 |e1| is rejected.  So o + t d, the point where the reference
// has the hit, lies within |R| <= 4 * 5.16 eps / 1e-4 |d| |e2| |s| = 0.01231
// |d| |e2| |s| of v0 + u e1 + v e2, a point of the triangle.  (Rounding s, e1
// and e2 moves it by parts of 1e-7 of the coordinates, which wide_ray's margins
// cover.)  A box that holds the triangle, grown by that much, is entered no
// later than at the computed t.
//
// The bound grows with the square of a scene's size, and grown boxes are
// entered more often, so the tree serves scenes and rays of moderate size
// only, others walk the binary tree.  WIDE_SCENE bounds the growth relative to
// |e2| over the size of a scene for |d| = 1: over 10 / 30 / 100 units, closest
// hits among a million triangles take 0.57 / 0.73 / 1.33 of the binary walk's
// time, 5000 take 0.65 / 0.88 / 1.75, 300 take 0.70 / 1.04 / 1.64.  WIDE_FAR
// bounds it for a ray over its distance from the scene's middle, or half the
// scene's size; RefWalker serves others.  Among spheres over 8 units that bound
// is 1.0 for |d| = 20: 0.6 to 1.25 of the binary walk's time; over 240 units,
// from outside, 3: 4 to 6 times, with RefWalker 1.3.
constexpr float WIDE_ERR = 0.0126f;
constexpr float WIDE_SCENE = 0.4f, WIDE_FAR = 1.5f;
// The entry distances' slack below the running t_max: 3 eps_zero of rayInBox,
// rounding and a margin.
__device__ __forceinline__ float wide_limit(float t) { return __builtin_fmaf(fabsf(t), 0x1p-16f, t) + 4.2e-4f; }

// Sets up the ray; false when it is outside the margins' range (origin far
// outside the scene, non-finite or extreme values, a negative tmin) or
// WIDE_FAR: such rays are walked in the reference's order.
__device__ __forceinline__ bool wide_ray(const SceneView &S, V3 o, V3 d, float tmin, WideRay &r) {
    r.o = o;
    r.d = d;
    const float p[3] = {(o.x - S.wide_lo[0]) * S.wide_scale, (o.y - S.wide_lo[1]) * S.wide_scale,
                        (o.z - S.wide_lo[2]) * S.wide_scale};
    const float dv[3] = {d.x, d.y, d.z};
    const float far = fmaxf(fmaxf(fabsf(p[0]), fabsf(p[1])), fabsf(p[2]));
    const float off = fmaxf(fmaxf(fabsf(p[0] - S.wide_mid[0]), fabsf(p[1] - S.wide_mid[1])), fabsf(p[2] - S.wide_mid[2]));
    const float dmax = fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
    // fmax drops NaNs, so they are looked for in the sums
    const float sum = ((p[0] + p[1]) + p[2]) + ((d.x + d.y) + d.z);
    r.err = length(d) * S.wide_rscale * WIDE_ERR;
    const bool ok = tmin >= 0.0f && far < 4e6f && dmax > 1e-3f && dmax < 1e9f && sum == sum &&
                    r.err * fmaxf(off, 0.5f * S.wide_reach) < WIDE_FAR;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const bool par = fabsf(dv[k]) < T_EPS;
        // a parallel axis asks only for lo <= o <= hi; its planes lie
        // (almost) infinitely far ahead or behind
        const float iv = par ? 0x1p60f : (1.0f / dv[k]) * S.wide_rscale;
        // the slab test's roundings, here and in the reference, stay below
        // 8 eps (|o| + extent) / |d|; twice that is allowed
        const float g = (fabsf(p[k]) + 32768.0f) * 0x1p-20f;
        if (par) r.err = -fabsf(r.err);
        const float m = fabsf(iv) * g, c = p[k] * iv;
        r.inv[k] = iv;
        r.nr[k] = -c - m;
        r.fr[k] = -c + m + 3.2e-4f;
    }
    return ok;
}

// The number of a triangle's leaf in the implicit heap.
__device__ __forceinline__ uint32_t leaf_of(const TriRec *tris, int32_t slot) { return __float_as_uint(tris[slot].e2[3]); }

// G(leaf) and L(leaf) < limit for the leaf that holds triangle `slot`.
__device__ __forceinline__ bool leaf_certain(const PairNode *nodes, const TriRec *tris, int32_t slot, V3 o, V3 d,
                                             float tmin, float limit) {
    const uint32_t c = leaf_of(tris, slot);
    const float4 *P = reinterpret_cast<const float4 *>(nodes + (c >> 1));
    const float4 A = P[0], B = P[1], C = P[2];
    float tL = tmin, tR = INFINITY;
    if (c & 1u)
        box_test(ray_pre(o, d), B.z, B.w, C.x, C.y, C.z, C.w, tL, tR);
    else
        box_test(ray_pre(o, d), A.x, A.y, A.z, A.w, B.x, B.y, tL, tR);
    return tL < tR && tL < limit;
}

// Of two triangles of different leaves, the one whose leaf the reference comes
// to first if it visits both: it enters first the child of their leaves'
// common ancestor whose box the ray enters first, child 1 of equal ones.
__device__ __forceinline__ int32_t first_of(const PairNode *nodes, const TriRec *tris, int32_t x, int32_t y, V3 o, V3 d,
                                            float tmin) {
    uint32_t a = leaf_of(tris, x), b = leaf_of(tris, y);
    const int up = (int)__clz(a) - (int)__clz(b);
    a >>= up < 0 ? -up : 0;
    b >>= up > 0 ? up : 0;
    const int k = 32 - (int)__clz(a ^ b);
    const float4 *P = reinterpret_cast<const float4 *>(nodes + (a >> k));
    const float4 A = P[0], B = P[1], C = P[2];
    const RayPre r = ray_pre(o, d);
    float tL0 = tmin, tR0 = INFINITY, tL1 = tmin, tR1 = INFINITY;
    box_test(r, A.x, A.y, A.z, A.w, B.x, B.y, tL0, tR0);
    box_test(r, B.z, B.w, C.x, C.y, C.z, C.w, tL1, tR1);
    return ((a >> (k - 1)) & 1u) == (tL0 < tL1 ? 0u : 1u) ? x : y;
}

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float half_lo(uint32_t w) { return (float)__builtin_bit_cast(half2_t, w)[0]; }
__device__ __forceinline__ float half_hi(uint32_t w) { return (float)__builtin_bit_cast(half2_t, w)[1]; }
// mask ? a : b per bit (v_bfi)
__device__ __forceinline__ uint32_t bit_select(uint32_t mask, uint32_t a, uint32_t b) { return (a & mask) | (b & ~mask); }

// A node reference: an index into the nodes, or with bit 31 one of the four
// runs of a leaf's triangles, first << 6 | count << 2 | run.
//
// A walk visits nodes (cur) and runs (the group l) independently: a leaf's
// runs wait in l while the lane goes on to its next nodes, until a second
// leaf's runs come up.  So a wave can take steps of one kind with most of its
// lanes, whichever kind its lanes came to first.
struct WideWalker {
    WideLds stk;
    int sp;             // groups in stk
    uint32_t cur;       // the node to visit next, or WIDE_NONE
    uint32_t gx, gy;    // newest group
    uint32_t lx, ly;    // a leaf's runs still to test
    int32_t best;
    float tmax, t2;     // the closest accepted t, and the next one (both start at the search limit)

    __device__ __forceinline__ void init(float tmax0) {
        sp = 0;
        cur = 0u;
        gy = ly = 0u;
        best = -1;
        tmax = t2 = tmax0;
    }
    __device__ __forceinline__ void stop() {
        sp = 0;
        cur = WIDE_NONE;
        gy = ly = 0u;
    }
    __device__ __forceinline__ bool has_node() const { return cur != WIDE_NONE; }
    __device__ __forceinline__ bool has_run() const { return ly != 0u; }

    // Finds the next node: the first child of the newest group that may hold
    // a closer hit.  A leaf's runs move to l if that is free, else cur stays
    // WIDE_NONE until they can.
    __device__ __forceinline__ void next(float lim) {
        cur = WIDE_NONE;
        while (true) {
            if (gy == 0u) {
                if (sp == 0) return;
                const uint2 e = stk.get(--sp);
                gx = e.x;
                gy = e.y;
            }
            if (!(__uint_as_float(gy & GROUP_T) <= lim)) {
                gy = 0u;
            } else if (gx & 0x80000000u) {
                if (ly) return;
                lx = gx;
                ly = gy;
                gy = 0u;
            } else {
                cur = gx | (gy & 3u);
                drop_first(gy);
                return;
            }
        }
    }
    static __device__ __forceinline__ void drop_first(uint32_t &y) {
        const uint32_t rest = (y & GROUP_T) | ((y & 0x700u) - 0x100u) | ((y & 0xffu) >> 2);
        y = (y & 0x600u) ? rest : 0u;
    }

    // pad for a ray with parallel axes, whose planes lie at 2^60 times their
    // distance.  Over a leaf's runs, which are smaller than the leaf, the ray
    // also drifts by its small component.
    static __device__ __forceinline__ float par_pad(const WideRay &r, float scale, const float (&cn)[3], uint4 M) {
        const float d[3] = {fabsf(r.d.x), fabsf(r.d.y), fabsf(r.d.z)};
        float dist = half_lo(M.z), drift = 0.0f;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const bool par = d[a] < T_EPS;
            dist = __builtin_fmaf(fabsf(cn[a]), par ? 0x1p-60f : d[a] * scale, dist);
            drift = par ? fmaxf(drift, d[a]) : drift;
        }
        const float pad = -r.err * half_hi(M.y) * dist;
        return M.w & 0x80000000u ? __builtin_fmaf(drift / fmaxf(fmaxf(d[0], d[1]), d[2]), dist, pad) : pad;
    }

    // Visits cur.
    __device__ __forceinline__ void step_node(const WideNode *nodes, float scale, const WideRay &r, float tmin) {
        const float lim = wide_limit(tmax);
        const uint4 *P = reinterpret_cast<const uint4 *>(nodes + cur);
        const uint4 X = P[0], Y = P[1], Z = P[2], M = P[3];
        const float org[3] = {(float)(M.x & 0xffffu), (float)(M.x >> 16), (float)(M.y & 0xffffu)};
        float cn[3], cf[3];
        uint32_t sg[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            cn[a] = __builtin_fmaf(org[a], r.inv[a], r.nr[a]);
            cf[a] = __builtin_fmaf(org[a], r.inv[a], r.fr[a]);
            sg[a] = (uint32_t)((int32_t)__float_as_uint(r.inv[a]) >> 31);
        }
        // how far from a triangle below the ray may pass where the test
        // accepts it (WIDE_ERR): at this distance, at most that to the node's
        // origin along the axes, plus D.  Entries are that much earlier; over
        // a leaf's runs, which the reference does not test, exits later too.
        const float dx = fabsf(cn[0] * r.d.x), dy = fabsf(cn[1] * r.d.y), dz = fabsf(cn[2] * r.d.z);
        // (a 2-norm is at most 0.415 times the sum and 0.585 times the largest)
        const float dist = __builtin_fmaf(__builtin_fmaf(0.585f, fmaxf(fmaxf(dx, dy), dz), 0.415f * (dx + dy + dz)), scale, half_lo(M.z));
        float pad = r.err * half_hi(M.y) * dist;
        if (r.err < 0.0f) pad = par_pad(r, scale, cn, M);
        pad = fminf(pad, 1e9f);  // an infinite E: beyond every coordinate
        const float padf = __uint_as_float(__float_as_uint(pad) & (uint32_t)((int32_t)M.w >> 31));
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            cn[a] = __builtin_fmaf(-pad, fabsf(r.inv[a]), cn[a]);
            cf[a] = __builtin_fmaf(padf, fabsf(r.inv[a]), cf[a]);
        }
        const uint32_t nx[2] = {bit_select(sg[0], X.z, X.x), bit_select(sg[0], X.w, X.y)};
        const uint32_t fx[2] = {bit_select(sg[0], X.x, X.z), bit_select(sg[0], X.y, X.w)};
        const uint32_t ny[2] = {bit_select(sg[1], Y.z, Y.x), bit_select(sg[1], Y.w, Y.y)};
        const uint32_t fy[2] = {bit_select(sg[1], Y.x, Y.z), bit_select(sg[1], Y.y, Y.w)};
        const uint32_t nz[2] = {bit_select(sg[2], Z.z, Z.x), bit_select(sg[2], Z.w, Z.y)};
        const uint32_t fz[2] = {bit_select(sg[2], Z.x, Z.z), bit_select(sg[2], Z.y, Z.w)};
        int key[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int w = k >> 1;
            const float ax = __builtin_fmaf(k & 1 ? half_hi(nx[w]) : half_lo(nx[w]), r.inv[0], cn[0]);
            const float ay = __builtin_fmaf(k & 1 ? half_hi(ny[w]) : half_lo(ny[w]), r.inv[1], cn[1]);
            const float az = __builtin_fmaf(k & 1 ? half_hi(nz[w]) : half_lo(nz[w]), r.inv[2], cn[2]);
            const float bx = __builtin_fmaf(k & 1 ? half_hi(fx[w]) : half_lo(fx[w]), r.inv[0], cf[0]);
            const float by = __builtin_fmaf(k & 1 ? half_hi(fy[w]) : half_lo(fy[w]), r.inv[1], cf[1]);
            const float bz = __builtin_fmaf(k & 1 ? half_hi(fz[w]) : half_lo(fz[w]), r.inv[2], cf[2]);
            const float en = fmaxf(fmaxf(fmaxf(ax, ay), az), tmin);
            const float ex = fminf(fminf(fminf(bx, by), bz), lim);
            // entry distance with the child's number in the low bits; as
            // integers, non-negative floats order like their values
            const uint32_t e = en <= ex ? __float_as_uint(en) : 0x7f800000u;
            key[k] = (int)((e & ~3u) | (uint32_t)k);
        }
        // children with larger triangles are entered whatever E says, after
        // the others where their boxes say no
        const uint32_t flags = M.z >> 28;
        if (flags) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (flags & (1u << k)) key[k] = key[k] < 0x7f7ffffc ? key[k] : 0x7f7ffffc | k;
        }
        // sort the four, nearest first
#define RM_CSWAP(a, b)                                  \
    {                                                   \
        const int lo_ = key[a] < key[b] ? key[a] : key[b]; \
        const int hi_ = key[a] < key[b] ? key[b] : key[a]; \
        key[a] = lo_;                                   \
        key[b] = hi_;                                   \
    }
        RM_CSWAP(0, 1)
        RM_CSWAP(2, 3)
        RM_CSWAP(0, 2)
        RM_CSWAP(1, 3)
        RM_CSWAP(1, 2)
#undef RM_CSWAP
        const uint32_t n = (key[0] < 0x7f800000 ? 0x100u : 0u) + (key[1] < 0x7f800000 ? 0x100u : 0u) +
                           (key[2] < 0x7f800000 ? 0x100u : 0u) + (key[3] < 0x7f800000 ? 0x100u : 0u);
        if (n) {
            if (gy) stk.put(sp++, gx, gy);
            gx = M.w;
            gy = (flags ? 0u : (uint32_t)key[0] & GROUP_T) | n | ((uint32_t)key[0] & 3u) | ((uint32_t)key[1] & 3u) << 2 |
                 ((uint32_t)key[2] & 3u) << 4 | ((uint32_t)key[3] & 3u) << 6;
        }
        next(lim);
    }

    // Tests a triangle (twice is as good as once).  Of equal t in one leaf the
    // first triangle stands, as in the reference; an equal t of another leaf
    // is kept in tie, or -1 there for two such leaves.  tie is memory, touched
    // only then: another register would cost every walk 4%.
    __device__ __forceinline__ void test(const TriRec *tris, uint32_t i, const TriRec &T, V3 o, V3 d, float tmin,
                                         volatile int32_t &tie) {
        const float t = tri_test_flat(o, d, V3{T.p[0], T.p[1], T.p[2]}, T.p[3], V3{T.e1[0], T.e1[1], T.e1[2]},
                                      V3{T.e2[0], T.e2[1], T.e2[2]});
        if (tmin < t && t <= t2) {
            if (t < tmax) {
                t2 = tmax;
                tmax = t;
                best = (int32_t)i;
            } else if (t > tmax) {
                t2 = t;
            } else if (best >= 0 && best != (int32_t)i) {
                const uint32_t leaf = leaf_of(tris, (int32_t)i);
                const int32_t was = t2 > tmax ? -1 : tie;
                if (leaf == leaf_of(tris, best)) {
                    best = min(best, (int32_t)i);
                } else if (t2 > tmax) {
                    tie = (int32_t)i;
                    t2 = tmax;
                } else {
                    tie = was >= 0 && leaf == leaf_of(tris, was) ? min(was, (int32_t)i) : -1;
                }
            }
        }
    }
    // After the walk (of the tree: only its tests write tie): with t2 == tmax,
    // tie is the one other leaf's triangle with that t, or -1.  Every other is
    // beyond it, so the least t2 that says so will do.
    __device__ __forceinline__ void settle(const SceneView &S, V3 o, V3 d, float tmin, const volatile int32_t &tie) {
        if (best < 0 || t2 != tmax) return;
        const int32_t other = tie;
        if (other >= 0) {
            best = first_of(S.nodes, S.tris, best, other, o, d, tmin);
            t2 = __uint_as_float(__float_as_uint(tmax) + 1u);
        }
    }
    // Those that the boxes' growth leaves out, by scalar loads where a wave's
    // lanes share the scene.
    __device__ __forceinline__ void test_big(const SceneView &S, V3 o, V3 d, float tmin, volatile int32_t &tie) {
        typedef const __attribute__((address_space(4))) uint32_t scalar_uint;
        typedef const __attribute__((address_space(4))) float scalar_float;
        scalar_uint *slots = (scalar_uint *)(uint64_t)S.big;
        for (int k = 0; k < S.n_big; ++k) {
            const uint32_t i = slots[k];
            scalar_float *p = (scalar_float *)(uint64_t)(S.tris + i);
            const TriRec T{{p[0], p[1], p[2], p[3]}, {p[4], p[5], p[6], p[7]}, {p[8], p[9], p[10], p[11]}};
            test(S.tris, i, T, o, d, tmin, tie);
        }
    }

    // Tests the first run of l.
    __device__ __forceinline__ void step_run(const TriRec *tris, const WideRay &r, float tmin, volatile int32_t &tie) {
        const uint32_t first = (lx >> 6) & 0x1ffffffu, c = (lx >> 2) & 15u, k = ly & 3u;
        const uint32_t end = first + (c * (k + 1u) >> 2);
        for (uint32_t i = first + (c * k >> 2); i < end; ++i) {
            TriRec T = load_tri(tris, i);
            // the whole record at once: v0 loaded past the first rejection
            // would cost a second memory latency
            asm volatile("" : "+v"(T.p[0]), "+v"(T.p[1]), "+v"(T.p[2]));
            test(tris, i, T, r.o, r.d, tmin, tie);
        }
        drop_first(ly);
        const float lim = wide_limit(tmax);
        if (!(__uint_as_float(ly & GROUP_T) <= lim)) ly = 0u;
        if (!has_node() && !ly) next(lim);
    }
};

// The reference's walk for one ray (Walker, whole leaves), a node at a time;
// its pending entries in per-lane scratch.
struct RefWalker {
    uint2 e[MAX_STACK];
    int sp;
    uint32_t cur;

    // the wide walk's tie, while this one is not under way
    __device__ __forceinline__ volatile int32_t &tie() { return *reinterpret_cast<volatile int32_t *>(&e[0].x); }
    __device__ __forceinline__ void init(uint32_t root_leaf) {
        sp = 0;
        cur = root_leaf ? root_leaf | 0x80000000u : 1u;
    }
    // True when the walk has finished (or tmax < aim).  inv: 1 / d.
    __device__ __forceinline__ bool step(const PairNode *bin, const TriRec *tris, V3 o, V3 d, const float (&inv)[3], float tmin,
                                         float aim, float &tmax, int32_t &best) {
        if (cur & 0x80000000u) {
            const uint32_t first = (cur & 0x7fffffffu) >> LEAF_SHIFT, cnt = cur & LEAF_MASK;
            for (uint32_t i = first; i < first + cnt; ++i) {
                const float t = tri_test(o, d, load_tri(tris, i));
                if (tmin < t && t < tmax) {
                    tmax = t;
                    best = (int32_t)i;
                }
            }
            cur = 0u;
            if (tmax < aim) return true;
        } else {
            const float4 *P = reinterpret_cast<const float4 *>(bin + cur);
            const float4 A = P[0], B = P[1], C = P[2];
            const uint2 L = *reinterpret_cast<const uint2 *>(&P[3]);
            const RayPre r{o, d, {inv[0], inv[1], inv[2]}, {fabsf(d.x) < T_EPS, fabsf(d.y) < T_EPS, fabsf(d.z) < T_EPS}};
            float tL0 = tmin, tR0 = tmax, tL1 = tmin, tR1 = tmax;
            if (r.par[0] || r.par[1] || r.par[2]) {
                box_test(r, A.x, A.y, A.z, A.w, B.x, B.y, tL0, tR0);
                box_test(r, B.z, B.w, C.x, C.y, C.z, C.w, tL1, tR1);
            } else {
                box_test_fast(r, A.x, A.y, A.z, A.w, B.x, B.y, tL0, tR0);
                box_test_fast(r, B.z, B.w, C.x, C.y, C.z, C.w, tL1, tR1);
            }
            const uint32_t ref0 = L.x ? (L.x | 0x80000000u) : (cur << 1);
            const uint32_t ref1 = L.y ? (L.y | 0x80000000u) : (cur << 1 | 1u);
            const bool f0 = tL0 < tL1;
            const float tLs = f0 ? tL1 : tL0, tRs = f0 ? tR1 : tR0;
            if (tLs < tRs) {
                e[sp++] = make_uint2(f0 ? ref1 : ref0, __float_as_uint(tLs));
            }
            cur = ((f0 ? tL0 : tL1) < (f0 ? tR0 : tR1)) ? (f0 ? ref0 : ref1) : 0u;
        }
        while (cur == 0u) {
            if (sp == 0) return true;
            const uint2 p = e[--sp];
            if (__uint_as_float(p.y) < tmax) cur = p.x;
        }
        return false;
    }

};

// Scenes of at most FLAT_MAX triangles are not walked.  Every lane passes over
// every triangle, whose rejection record the wave loads once into scalar
// registers, and keeps those its line may pass through as a bit mask; then
// each lane tests its own few with the reference's arithmetic, in order.  No
// lane waits for lanes at other nodes.  With the certificate of the wide walk
// the result is the reference's; a scene of one leaf is tested in the
// reference's own order.
//
// The rejection works on the unscaled values a, u a and v a from the line's
// moment (25 instructions a triangle, the exact test takes 66).  With eps =
// 2^-24: u a and v a are off here by at most 8 eps |d| |e| |o| + 7 eps |d| |e|
// |v0|, e being e2 or e1, and in the exact test, whose accepted u and v may lie
// outside [0, 1] by that, by 5.2 eps |d| |e| (|o| + |v0|); a by 4 and 5.2 eps |d|
// |e1| |e2|, and rounding u, v and their sum by 5 more.  Together at most 13.2 eps
// |d| (|e1| + |e2|) (|o| + |v0|) + 14.2 eps |d| |e1| |e2|.  With coordinates of at
// most m, |v0| is at most 1.74 m and |e1| |e2| at most 1.74 m (|e1| + |e2|), so this
// is below eps |d| (|e1| + |e2|) (13.2 |o| + 48 m); 64 |o| + 192 m are allowed
// (FLAT_ERR, flat_b = 3 m).
//
// FLAT_MAX is the masks' width.  Closest hits of 2M rays among 12 / 36 / 64
// triangles take 41 / 80 / 125 us, in the binary walk 616 / 645 / 681, of 20k
// rays 14 / 14 / 19 and 78 / 97 / 118; 100 triangles in the four-wide tree
// 439 and 39.  Extension rays of a 512 x 512 Cornell render (36 triangles, 16
// launches) took 2.99 ms with every triangle tested exactly, 1.00 with the
// masks and wide_per_wave's shares.
constexpr int FLAT_MAX = 64;
constexpr double FLAT_ERR = 64.0 / 16777216.0;

template <bool ANY>
__device__ __forceinline__ void flat_tris(const SceneView &S, V3 o, V3 d, float tmin, float aim, float &tmax, float &t2,
                                          int32_t &best) {
    typedef const __attribute__((address_space(4))) float scalar_float;
    const V3 m{__builtin_fmaf(o.y, d.z, -(o.z * d.y)), __builtin_fmaf(o.z, d.x, -(o.x * d.z)),
               __builtin_fmaf(o.x, d.y, -(o.y * d.x))};
    const float d1 = (fabsf(d.x) + fabsf(d.y)) + fabsf(d.z);
    float rho = -d1 * (((fabsf(o.x) + fabsf(o.y)) + fabsf(o.z)) + S.flat_b);
    // lines whose products could leave the normal numbers keep every triangle
    if (!(d1 > 1e-5f && rho > -1e18f)) rho = -INFINITY;
    uint32_t mask[2] = {0u, 0u};
    // one scene at a time: the lanes of a batch may hold several
    const uint64_t p = (uint64_t)S.flat_tris;
    uint64_t pending = __ballot(true);
    while (pending) {
        const int lead = (int)__ffsll((unsigned long long)pending) - 1;
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)p, lead);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(p >> 32), lead);
        const uint32_t n = (uint32_t)__builtin_amdgcn_readlane(S.flat, lead);
        const uint64_t q = (uint64_t)hi << 32 | lo;
        const bool mine = p == q;
        if (mine) {
            scalar_float *T = (scalar_float *)q;
            for (uint32_t i = 0; i < n; ++i, T += sizeof(FlatTri) / 4) {
                // -a, u a and -v a of the line; a's sign makes them comparable
                const float a = __builtin_fmaf(T[12], d.x, __builtin_fmaf(T[13], d.y, T[14] * d.z));
                const float u = __builtin_fmaf(T[3], m.x, __builtin_fmaf(T[4], m.y, __builtin_fmaf(T[5], m.z,
                                __builtin_fmaf(T[9], d.x, __builtin_fmaf(T[10], d.y, T[11] * d.z)))));
                const float v = __builtin_fmaf(T[0], m.x, __builtin_fmaf(T[1], m.y, __builtin_fmaf(T[2], m.z,
                                __builtin_fmaf(T[6], d.x, __builtin_fmaf(T[7], d.y, T[8] * d.z)))));
                const uint32_t sg = __float_as_uint(a) & 0x80000000u;
                const float x = __uint_as_float(__float_as_uint(u) ^ sg ^ 0x80000000u);
                const float y = __uint_as_float(__float_as_uint(v) ^ sg);
                const float z = fabsf(a) - (x + y);
                const bool out = fminf(fminf(x, y), z) < rho * T[15];
                mask[i >> 5] |= out ? 0u : 1u << (i & 31u);
            }
        }
        pending &= ~__ballot(mine);
    }
    int32_t tie = -1;                    // a triangle of another leaf with best's t
    uint32_t leaf = 0u, tie_leaf = 0u;   // best's and tie's
    while (mask[0] | mask[1]) {
        uint32_t i;
        if (mask[0]) {
            i = (uint32_t)__ffs((int)mask[0]) - 1u;
            mask[0] &= mask[0] - 1u;
        } else {
            i = 31u + (uint32_t)__ffs((int)mask[1]);
            mask[1] &= mask[1] - 1u;
        }
        const TriRec T = load_tri(S.tris, i);
        const float t = tri_test_flat(o, d, V3{T.p[0], T.p[1], T.p[2]}, T.p[3], V3{T.e1[0], T.e1[1], T.e1[2]},
                                      V3{T.e2[0], T.e2[1], T.e2[2]});
        const uint32_t l = __float_as_uint(T.e2[3]);
        const bool in = tmin < t && t < t2, first = t < tmax, other = l != leaf;
        const bool tied = in && other && t == tmax && (tie < 0 || l == tie_leaf);
        t2 = in && (first ? other || tie >= 0 : other && !tied) ? (first ? tmax : t) : t2;
        tie = in && first ? -1 : tied && tie < 0 ? (int32_t)i : tie;
        tie_leaf = tied ? l : tie_leaf;
        leaf = in && first ? l : leaf;
        best = in && first ? (int32_t)i : best;
        tmax = in && first ? t : tmax;
        if (ANY && tmax < aim) break;
    }
    if (tie >= 0) best = first_of(S.nodes, S.tris, best, tie, o, d, tmin);
}

// Whether the result of flat_tris or of a finished wide walk stands.
template <bool ANY>
__device__ __forceinline__ bool hit_sure(const SceneView &S, V3 o, V3 d, float tmin, float aim, float tmax, float t2,
                                         int32_t best) {
    if (S.root_leaf) return true;
    if (ANY && aim > -INFINITY) return !(tmax < aim) || leaf_certain(S.nodes, S.tris, best, o, d, tmin, aim);
    return best < 0 || (tmax < t2 && leaf_certain(S.nodes, S.tris, best, o, d, tmin, fminf(t2, wide_limit(tmax))));
}

// The whole wide walk of one ray, for kernels that do more than traversal.
// Same contract as trace_walk; the kernel provides wide_lds_bytes.
template <bool ANY>
__device__ __forceinline__ int32_t wide_walk(const SceneView &S, V3 o, V3 d, float tmin, float &tmax, float aim) {
    WideWalker w;
    WideRay r;
    RefWalker ref;
    w.stk.bind();
    w.init(tmax);
    bool sure = true;
    if (S.flat) {
        flat_tris<ANY>(S, o, d, tmin, aim, w.tmax, w.t2, w.best);
    } else if (S.wide && wide_ray(S, o, d, tmin, r)) {
        w.test_big(S, o, d, tmin, ref.tie());
        while (!(ANY && w.tmax < aim)) {
            if (w.has_run()) {
                w.step_run(S.tris, r, tmin, ref.tie());
                if (ANY && w.tmax < aim) break;
            } else if (w.has_node()) {
                w.step_node(S.wide, S.wide_scale, r, tmin);
            } else {
                break;
            }
        }
        w.settle(S, o, d, tmin, ref.tie());
    } else {
        sure = false;
    }
    if (!sure || !hit_sure<ANY>(S, o, d, tmin, aim, w.tmax, w.t2, w.best)) {
        ref.init((uint32_t)S.root_leaf);
        r.reciprocals(d);
        w.tmax = tmax;
        w.best = -1;
        while (!ref.step(S.nodes, S.tris, o, d, r.inv, tmin, aim, w.tmax, w.best)) {
        }
    }
    tmax = w.tmax;
    return w.best;
}

// Rays a wave takes at a time from n in a launch of `waves` waves.  Many: an
// eighth of its share, up to 512.  Few: over a fifth of the waves, between 8
// and 64 each; the walks of a wave wait for each other, and those of many
// waves compete (closest hits among 1M triangles, 8 / 16 / 32 / 64 rays a
// wave: 10k rays 223 / 241 / 258 / 278 us, 100k rays 571 / 377 / 344 / 339 us).
// The rays of a flat scene cost the same, so a wave takes whole batches, its
// whole share at the start where that is at most 512: claims are atomic adds
// to one address, 12 ns each on the traces' 64-bit counter, and 64 rays a claim
// held 2M closest hits among 36 triangles to 392 us (80 so, and 302 for 8M).
__host__ __device__ inline uint32_t wide_per_wave(uint32_t n, uint32_t waves, bool flat) {
    if (flat) {
        const uint32_t p = ((n - 1u) / 64u + waves) / waves * 64u;
        return p > 512u ? 512u : p;
    }
    if (n / 64u < waves) {
        const uint32_t p = (uint32_t)(((uint64_t)n * 5u + waves - 1u) / waves);
        return p < 8u ? 8u : p > 64u ? 64u : p;
    }
    const uint32_t p = n / (8u * waves) & ~63u;
    return p < 64u ? 64u : p > 512u ? 512u : p;
}

// The loop of a persistent wide walk.  Src: the kernel's rays,
//   n()                     how many
//   load(i, o, d, tmax, aim) takes ray i and its scene (i may become another
//                           name of the ray, which store() gets)
//   scene()                 the SceneView of the ray taken last
//   store(i, tmax, best, aim) writes ray i's result
// A wave starts with the `per` rays at its own number, takes `per` more at a
// time from *work (0 at the start) while there are any, and hands them to
// lanes whose rays are done once `fetch_min` lanes are without one; those
// lanes then check and store their results together.  Each iteration takes
// one kind of step: runs when at least phases / 64 of the walking lanes have
// one, else nodes.  Every wave leaves when its rays are used up and its lanes
// are done.  (Waves that all begin with an atomic on one address wait 6 ns for
// each other on the renders' 32-bit counters: 50 us for a launch of 8192 with
// little or nothing to do.)
template <bool ANY, class Src, class Count>
__device__ __forceinline__ void wide_loop(Src &src, Count *work, uint32_t per, float tmin, int fetch_min, int phases) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t n = src.n();
    const uint32_t wave = blockIdx.x * (WALK_BLOCK / 64u) + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t begun = gridDim.x * (WALK_BLOCK / 64u) * per;  // the rays that waves start with
    uint32_t at = wave * per;                                     // the wave's rays in hand
    if (at >= n) return;
    uint32_t end = at + per < n ? at + per : n;
    bool more = begun < n;
    WideWalker w;
    RefWalker ref;
    WideRay r;
    w.stk.bind();
    w.stop();
    float aim = -INFINITY, tmax0 = 0.0f;
    uint32_t ray = WIDE_NONE;   // this lane's ray
    bool in_ref = false;        // it is walked in the reference's order
    while (true) {
        const bool walking = in_ref || w.has_node() || w.has_run();
        const uint32_t nwalk = (uint32_t)__popcll(__ballot(walking));
        if (nwalk == 0u || ((more || at < end) && 64u - nwalk >= (uint32_t)fetch_min)) {
            // results of the lanes that finished
            if (ray != WIDE_NONE && !walking) {
                const SceneView &S = src.scene();
                if (!S.flat) w.settle(S, r.o, r.d, tmin, ref.tie());  // (flat_tris has its own)
                if (hit_sure<ANY>(S, r.o, r.d, tmin, aim, w.tmax, w.t2, w.best)) {
                    src.store(ray, w.tmax, w.best, aim);
                    ray = WIDE_NONE;
                } else {
                    in_ref = true;
                    ref.init((uint32_t)S.root_leaf);
                    r.reciprocals(r.d);
                    w.tmax = tmax0;
                    w.best = -1;
                }
            }
            if (at >= end && more) {
                uint32_t b = 0;
                if (lane == 0) b = (uint32_t)atomicAdd(work, (Count)per);
                at = begun + (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
                end = at + per < n ? at + per : n;
                if (at >= n) {
                    end = at;
                    more = false;
                }
            }
            const uint64_t idle = __ballot(ray == WIDE_NONE);
            if (at >= end && ~idle == 0ull && !more) break;
            if (at < end && ray == WIDE_NONE) {
                const uint32_t i = at + (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
                if (i < end) {
                    ray = i;
                    V3 o, d;
                    src.load(ray, o, d, tmax0, aim);
                    w.init(tmax0);
                    const SceneView &S = src.scene();
                    const bool ok = wide_ray(S, o, d, tmin, r) && S.wide;
                    if (S.flat) {
                        w.stop();
                        flat_tris<ANY>(S, o, d, tmin, aim, w.tmax, w.t2, w.best);
                    } else if (!ok) {
                        in_ref = true;
                        ref.init((uint32_t)S.root_leaf);
                        r.reciprocals(d);
                        w.stop();
                    } else {
                        w.test_big(S, o, d, tmin, ref.tie());
                        if (ANY && w.tmax < aim) w.stop();
                    }
                }
            }
            if (at < end) at += (uint32_t)__popcll(idle);
        }
        if (__ballot(in_ref)) {
            if (walk_turn(ref.cur, phases, in_ref) && in_ref) {
                const SceneView &S = src.scene();
                if (ref.step(S.nodes, S.tris, r.o, r.d, r.inv, tmin, aim, w.tmax, w.best)) {
                    src.store(ray, w.tmax, w.best, aim);
                    ray = WIDE_NONE;
                    in_ref = false;
                }
            }
        }
        const uint64_t nodes = __ballot(w.has_node()), runs = __ballot(w.has_run());
        const uint32_t nr = (uint32_t)__popcll(runs), nw = (uint32_t)__popcll(nodes | runs);
        if (nr && (!nodes || 64u * nr >= (uint32_t)phases * nw)) {
            if (w.has_run()) {
                w.step_run(src.scene().tris, r, tmin, ref.tie());
                if (ANY && w.tmax < aim) w.stop();
            }
        } else if (w.has_node()) {
            const SceneView &S = src.scene();
            w.step_node(S.wide, S.wide_scale, r, tmin);
        }
    }
}

// One ray's walk of kind TPS: WALK_WIDE, WALK_FLAT, or the reference-order walk
// with TPS triangles per step.
template <bool ANY, bool LDSW = true, int TPS = 0>
__device__ __forceinline__ int32_t scene_walk(const SceneView &S, const RayPre &r, float tmin, float &tmax, float aim) {
    static_assert(TPS != WALK_WIDE || LDSW, "the wide walk's groups are in LDS");
    if constexpr (TPS == WALK_WIDE)
        return wide_walk<ANY>(S, r.o, r.d, tmin, tmax, aim);
    else if constexpr (TPS == WALK_FLAT) {
        if (S.flat) {
            float tm = tmax, t2 = tmax;
            int32_t best = -1;
            flat_tris<ANY>(S, r.o, r.d, tmin, aim, tm, t2, best);
            if (hit_sure<ANY>(S, r.o, r.d, tmin, aim, tm, t2, best)) {
                tmax = tm;
                return best;
            }
        }
        return trace_walk<ANY, LDSW, 0>(S, r, tmin, tmax, aim);
    } else
        return trace_walk<ANY, LDSW, TPS>(S, r, tmin, tmax, aim);
}

}  // namespace rm
