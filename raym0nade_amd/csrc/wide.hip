// Builds the four-wide tree (wide.h) of an uploaded scene on the GPU, from
// the binary tree and the triangles that rm_scene_create put there.
//
// Levels of the binary heap are taken two at a time, such that the deepest
// leaves' level is one of those kept; an odd rest goes to the root.  Slot
// (level l, position j) of a kept level is the child of one node only, so a
// node's children sit side by side and every slot is filled by one thread
// without looking at any other.  A leaf one level above a kept level takes the
// slot of its first would-be descendant.
#include <cstring>

#include "rm_internal.h"
#include "wide.h"

namespace rm {

// fp16 bits of v >= 0 rounded down or up (up: at most 65504).
__device__ __forceinline__ uint32_t half_down(double v) {
    if (!(v > 0.0)) return 0u;
    const _Float16 h = (_Float16)v;
    uint32_t b = __builtin_bit_cast(unsigned short, h);
    if (b > 0x7bffu) b = 0x7bffu;
    return (double)__builtin_bit_cast(_Float16, (unsigned short)b) > v ? b - 1u : b;
}
__device__ __forceinline__ uint32_t half_up(double v) {
    if (!(v > 0.0)) return 0u;
    const _Float16 h = (_Float16)v;
    uint32_t b = __builtin_bit_cast(unsigned short, h);
    if (b >= 0x7bffu) return 0x7bffu;
    return (double)__builtin_bit_cast(_Float16, (unsigned short)b) < v ? b + 1u : b;
}

// Child boxes of a node in scene coordinates, then its record.
struct WideBoxes {
    float lo[4][3], hi[4][3];
    bool used[4];
};
__device__ void set_child(WideBoxes &B, int k, const PairNode &P, int side) {
    const float v[12] = {P.a[0], P.a[1], P.a[2], P.a[3], P.b[0], P.b[1], P.b[2], P.b[3], P.c[0], P.c[1], P.c[2], P.c[3]};
    for (int a = 0; a < 3; ++a) {
        B.lo[k][a] = v[6 * side + a];
        B.hi[k][a] = v[6 * side + 3 + a];
    }
    B.used[k] = true;
}

__global__ __launch_bounds__(256) void k_wide_build(const PairNode *__restrict__ bin, TriRec *__restrict__ tris,
                                                    const TriShade *__restrict__ shade, WideNode *__restrict__ out,
                                                    uint32_t off, int level, int step, uint32_t child_off, float lx,
                                                    float ly, float lz, double scale) {
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    if (j >= (1u << level)) return;
    // what heap node w = 2^level + j is: follow its bits from the root
    const uint32_t w = (1u << level) + j;
    uint32_t u = 1u, leaf = 0u;
    int b = level;
    while (b > 0) {
        --b;
        leaf = bin[u].leaf[(w >> b) & 1u];
        u = w >> b;
        if (leaf) break;
    }
    // b bits are left below a leaf: w itself, or its parent when w is the
    // parent's first child (a leaf on the level between)
    if (leaf && (b > 1 || (b == 1 && (w & 1u)))) return;
    WideBoxes B;
    for (int k = 0; k < 4; ++k) B.used[k] = false;
    double pad_e = 0.0, pad_d = 0.0;
    uint32_t ref;
    const float lo[3] = {lx, ly, lz};
    if (leaf) {
        const uint32_t first = leaf >> LEAF_SHIFT, c = leaf & LEAF_MASK;
        ref = 0x80000000u | (first << 6) | (c << 2);
        float all_lo[3] = {INFINITY, INFINITY, INFINITY}, all_hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (uint32_t k = 0; k < 4; ++k) {
            for (int a = 0; a < 3; ++a) {
                B.lo[k][a] = INFINITY;
                B.hi[k][a] = -INFINITY;
            }
            for (uint32_t i = first + (c * k >> 2); i < first + (c * (k + 1) >> 2); ++i) {
                for (int q = 0; q < 3; ++q)
                    for (int a = 0; a < 3; ++a) {
                        const float x = shade[i].v[q][a];
                        B.lo[k][a] = fminf(B.lo[k][a], x);  // a NaN is dropped: its triangle is never hit
                        B.hi[k][a] = fmaxf(B.hi[k][a], x);
                    }
                const double ex = tris[i].e2[0], ey = tris[i].e2[1], ez = tris[i].e2[2];
                pad_e = fmax(pad_e, sqrt(ex * ex + ey * ey + ez * ez));
                tris[i].e2[3] = __uint_as_float(u);
            }
            // (a run without triangles keeps its inverted bounds)
            B.used[k] = B.lo[k][0] <= B.hi[k][0] && B.lo[k][1] <= B.hi[k][1] && B.lo[k][2] <= B.hi[k][2];
            if (B.used[k])
                for (int a = 0; a < 3; ++a) {
                    all_lo[a] = fminf(all_lo[a], B.lo[k][a]);
                    all_hi[a] = fmaxf(all_hi[a], B.hi[k][a]);
                }
        }
        if (all_lo[0] <= all_hi[0]) {
            const double dx = (double)all_hi[0] - all_lo[0], dy = (double)all_hi[1] - all_lo[1],
                         dz = (double)all_hi[2] - all_lo[2];
            pad_d = 1.3 * sqrt(dx * dx + dy * dy + dz * dz);  // distance to v0, and the share of |e1| in the a term
        }
    } else {
        const uint32_t cj = step == 1 ? 2u * j : 4u * j;
        ref = child_off + cj;
        const PairNode P = bin[w];
        for (int s = 0; s < 2; ++s) {
            if (step == 1) {
                set_child(B, s, P, s);  // the root over one level
            } else if (P.leaf[s]) {
                set_child(B, 2 * s, P, s);
            } else {
                const PairNode Q = bin[2u * w + s];
                set_child(B, 2 * s, Q, 0);
                set_child(B, 2 * s + 1, Q, 1);
            }
        }
    }
    double org[3];
    for (int a = 0; a < 3; ++a) {
        double m = 65535.0;
        for (int k = 0; k < 4; ++k)
            if (B.used[k]) m = fmin(m, ((double)B.lo[k][a] - lo[a]) * scale);
        org[a] = floor(fmin(fmax(m, 0.0), 32767.0));
    }
    uint32_t pl[3][4];
    for (int a = 0; a < 3; ++a) {
        uint32_t l[4], h[4];
        for (int k = 0; k < 4; ++k) {
            l[k] = B.used[k] ? half_down(((double)B.lo[k][a] - lo[a]) * scale - org[a]) : 0x7c00u;
            h[k] = B.used[k] ? half_up(((double)B.hi[k][a] - lo[a]) * scale - org[a]) : 0u;
        }
        pl[a][0] = l[0] | (l[1] << 16);
        pl[a][1] = l[2] | (l[3] << 16);
        pl[a][2] = h[0] | (h[1] << 16);
        pl[a][3] = h[2] | (h[3] << 16);
    }
    uint4 *o = reinterpret_cast<uint4 *>(out + (off + j));
    o[0] = make_uint4(pl[0][0], pl[0][1], pl[0][2], pl[0][3]);
    o[1] = make_uint4(pl[1][0], pl[1][1], pl[1][2], pl[1][3]);
    o[2] = make_uint4(pl[2][0], pl[2][1], pl[2][2], pl[2][3]);
    o[3] = make_uint4((uint32_t)org[0] | ((uint32_t)org[1] << 16),
                      (uint32_t)org[2] | (half_up(pad_e * scale) << 16), half_up(pad_d * scale), ref);
}

// The walks' range: coordinates that are finite and whose scaling stays in
// the float range.
static bool wide_range(const HostScene &h, float &ext, float &mag) {
    ext = mag = 0.0f;
    for (int a = 0; a < 3; ++a) {
        if (!isfinite(h.root_lo[a]) || !isfinite(h.root_hi[a])) return false;
        ext = std::max(ext, h.root_hi[a] - h.root_lo[a]);
        mag = std::max({mag, fabsf(h.root_lo[a]), fabsf(h.root_hi[a])});
    }
    return ext > 1e-12f && ext < 1e12f && mag <= 1e4f * ext;
}

// A flat scene's records follow its triangles in their buffer: no kernel and
// no allocation for scenes that are made in half a millisecond.
size_t append_flat(HostScene &h) {
    float ext, mag;
    if (h.n > FLAT_MAX || !wide_range(h, ext, mag)) return 0;
    const size_t n = (size_t)h.n, off = (n * sizeof(TriRec) + 63) & ~size_t(63);
    if (!h.root_leaf)  // the leaves' numbers
        for (uint32_t u = 1; u < h.pairs.size(); ++u)
            for (uint32_t k = 0; k < 2; ++k)
                for (uint32_t i = 0; i < (h.pairs[u].leaf[k] & LEAF_MASK); ++i) {
                    const uint32_t c = 2 * u + k;
                    std::memcpy(&h.tris[(h.pairs[u].leaf[k] >> LEAF_SHIFT) + i].e2[3], &c, 4);
                }
    h.tris.resize((off + n * sizeof(FlatTri) + sizeof(TriRec) - 1) / sizeof(TriRec));
    for (size_t i = 0; i < n; ++i) {
        const TriRec T = h.tris[i];
        double v0[3], e1[3], e2[3], l1 = 0.0, l2 = 0.0;
        for (int a = 0; a < 3; ++a) {
            v0[a] = T.p[a], e1[a] = T.e1[a], e2[a] = T.e2[a];
            l1 += e1[a] * e1[a], l2 += e2[a] * e2[a];
        }
        FlatTri F;
        for (int a = 0; a < 3; ++a) {
            const int b = (a + 1) % 3, c = (a + 2) % 3;
            F.e1[a] = T.e1[a], F.e2[a] = T.e2[a];
            F.w1[a] = (float)(v0[b] * e1[c] - e1[b] * v0[c]);
            F.w2[a] = (float)(v0[b] * e2[c] - e2[b] * v0[c]);
            F.n[a] = (float)(e1[b] * e2[c] - e2[b] * e1[c]);
        }
        const double len = sqrt(l1) + sqrt(l2);
        F.k = len > 1e-15 ? (float)(FLAT_ERR * len) : INFINITY;  // shorter, or NaN: never rejected
        std::memcpy(reinterpret_cast<char *>(h.tris.data()) + off + i * sizeof(FlatTri), &F, sizeof(F));
    }
    return off;
}

// Scenes outside the tree's range keep the binary walk: 2^25 triangles or
// more (a run's reference), coordinates outside wide_range.  flat: where
// append_flat put the records, or 0.
int32_t build_wide(rm_scene *s, size_t flat) {
    SceneView &v = s->view;
    v.wide = nullptr;
    v.flat = 0;
    v.flat_tris = nullptr;
    const HostScene &h = s->host;
    float ext, mag;
    if (h.n >= (int64_t(1) << 25) || !wide_range(h, ext, mag)) return RM_OK;
    if (flat) {
        v.flat = (int32_t)h.n;
        v.flat_b = 3.0f * mag;
        v.flat_tris = reinterpret_cast<const FlatTri *>(s->tris.as<char>() + flat);
        return RM_OK;
    }
    const int e = (int)floor(log2(30000.0 / (double)ext));
    const double scale = ldexp(1.0, e);
    for (int a = 0; a < 3; ++a) v.wide_lo[a] = (float)((double)h.root_lo[a] - 1000.0 / scale);
    v.wide_scale = (float)scale;
    v.wide_rscale = (float)(1.0 / scale);
    const int leaf_level = h.depth - 1;  // the deepest leaves' level
    struct Level { int level, step; uint32_t off; };
    std::vector<Level> levels;
    uint32_t total = 0;
    for (int l = 0; l <= leaf_level;) {
        const int step = l == 0 && (leaf_level & 1) ? 1 : 2;
        levels.push_back(Level{l, step, total});
        total += std::max(4u, 1u << l);
        l += step;
    }
    const int32_t rc = s->wide.alloc((size_t)total * sizeof(WideNode));
    if (rc) return rc;
    for (size_t i = 0; i < levels.size(); ++i) {
        const Level &L = levels[i];
        const uint32_t child = i + 1 < levels.size() ? levels[i + 1].off : 0u;
        hipLaunchKernelGGL(k_wide_build, dim3(((1u << L.level) + 255) / 256), dim3(256), 0, nullptr, v.nodes,
                           s->tris.as<TriRec>(), v.shade, s->wide.as<WideNode>(), L.off, L.level, L.step, child,
                           v.wide_lo[0], v.wide_lo[1], v.wide_lo[2], scale);
    }
    RM_HIP(hipGetLastError());
    // the caller may use the scene on any stream next
    RM_HIP(hipStreamSynchronize(nullptr));
    v.wide = s->wide.as<WideNode>();
    return RM_OK;
}

}  // namespace rm
