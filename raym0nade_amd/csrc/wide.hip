// Builds the four-wide tree (wide.h) of an uploaded scene on the GPU, from
// the binary tree and the triangles that rm_scene_create put there.
//
// Levels of the binary heap are taken two at a time, such that the deepest
// leaves' level is one of those kept; an odd rest goes to the root.  Slot
// (level l, position j) of a kept level is the child of one node only, so a
// node's children sit side by side and every slot is filled by one thread
// without looking at any other.  A leaf one level above a kept level takes the
// slot of its first would-be descendant.
#include <algorithm>
#include <cstring>
#include <mutex>

#include "rm_internal.h"
#include "wide.h"

namespace rm {

constexpr uint32_t MAX_BIG = 8;

// fp16 bits of v >= 0 rounded down or up (up: at most 65504, or infinity).
__device__ __forceinline__ uint32_t half_down(double v) {
    if (!(v > 0.0)) return 0u;
    const _Float16 h = (_Float16)v;
    uint32_t b = __builtin_bit_cast(unsigned short, h);
    if (b > 0x7bffu) b = 0x7bffu;
    return (double)__builtin_bit_cast(_Float16, (unsigned short)b) > v ? b - 1u : b;
}
__device__ __forceinline__ uint32_t half_up(double v) {
    if (!(v > 0.0)) return 0u;
    if (v == INFINITY) return 0x7c00u;
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

// A node's E from its children's v: a child whose triangles are much larger
// than its siblings', so that the growth at the scene's size would show beside
// the node's own (`size`), is flagged instead.
__device__ __forceinline__ uint32_t flag_children(const double (&v)[4], const bool (&used)[4], double size, double reach,
                                                  double &e) {
    double least = INFINITY;
    for (int k = 0; k < 4; ++k)
        if (used[k]) least = fmin(least, v[k]);
    uint32_t flags = 0u;
    e = 0.0;
    for (int k = 0; k < 4; ++k) {
        if (!used[k]) continue;
        if (v[k] > 4.0 * least && WIDE_ERR * v[k] * reach > size * 0.0625)
            flags |= 1u << k;
        else
            e = fmax(e, v[k]);
    }
    return flags;
}

// |e2|, infinite where the reference's rejection bounds nothing because the
// square of |e1| leaves the float range, 0 for a triangle that is never hit.
__host__ __device__ inline double growth_edge(const TriRec &T) {
    double l1 = 0.0, l2 = 0.0;
    for (int a = 0; a < 3; ++a) {
        l1 += (double)T.e1[a] * T.e1[a];
        l2 += (double)T.e2[a] * T.e2[a];
    }
    if (!(l1 > 0.0 && l2 >= 0.0)) return 0.0;
    return l1 > 1e-30 ? sqrt(l2) : INFINITY;
}

// What the records of all levels are made from.
struct WideBuild {
    const PairNode *bin;
    TriRec *tris;
    const TriShade *shade;
    WideNode *out;
    float lo[3];
    double scale, reach, big;
    uint32_t *found;    // the large triangles: their number and slots, unless known
    uint32_t *host;     // where the number found goes in the end
};
// A kept level: its nodes are at `off`, the next kept one's at `child`.
struct WideLevel {
    int32_t level, step;
    uint32_t off, child;
};

// The record of node j of a level.
__device__ __forceinline__ void wide_node(const WideBuild &A, const WideLevel &L, uint32_t j) {
    const PairNode *bin = A.bin;
    TriRec *tris = A.tris;
    const TriShade *shade = A.shade;
    WideNode *out = A.out;
    const float lo[3] = {A.lo[0], A.lo[1], A.lo[2]};
    const double scale = A.scale, big = A.big;
    const int level = L.level;
    if (level == 0 && A.host) *A.host = A.found[0];  // the last level
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
    double v[4] = {0.0, 0.0, 0.0, 0.0};  // the largest |e2| below each child, scaled
    uint32_t ref;
    if (leaf) {
        const uint32_t first = leaf >> LEAF_SHIFT, c = leaf & LEAF_MASK;
        ref = 0x80000000u | (first << 6) | (c << 2);
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
                const double l = growth_edge(tris[i]);
                if (l > big) {
                    if (A.found) {  // found[0] of them, the first ones' slots behind
                        const uint32_t q = atomicAdd(A.found, 1u);
                        if (q < MAX_BIG) A.found[1 + q] = i;
                    }
                } else {
                    v[k] = fmax(v[k], l * scale);
                }
                tris[i].e2[3] = __uint_as_float(u);
            }
            // (a run without triangles keeps its inverted bounds)
            B.used[k] = B.lo[k][0] <= B.hi[k][0] && B.lo[k][1] <= B.hi[k][1] && B.lo[k][2] <= B.hi[k][2];
        }
    } else {
        const int step = L.step;
        const uint32_t cj = step == 1 ? 2u * j : 4u * j;
        ref = L.child + cj;
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
        for (int k = 0; k < 4; ++k)  // (the upper bits of an fp16 number)
            if (B.used[k])
                v[k] = (double)__builtin_bit_cast(_Float16, (unsigned short)((out[ref + k].m[2] >> 16 & 0xfffu) << 3));
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
    // how far from the node's origin each child's triangles reach, the large
    // ones before the walk left out: over them, and not over the boxes, which
    // one ground triangle can stretch to the scene's size
    double far[4] = {0.0, 0.0, 0.0, 0.0}, size = 0.0;
    for (int k = 0; k < 4; ++k) {
        if (!B.used[k]) continue;
        double q = 0.0;
        for (int a = 0; a < 3; ++a) {
            const double x = ((double)B.hi[k][a] - lo[a]) * scale - org[a];
            q += x > 0.0 ? x * x : 0.0;
        }
        far[k] = sqrt(q);
        size = fmax(size, far[k]);
        if (!leaf) {
            // (a child's D leaves its own flagged children out, which E here
            // may count: then its box stands)
            const WideNode &C = out[ref + k];
            const double x = (double)(C.m[0] & 0xffffu) - org[0], y = (double)(C.m[0] >> 16) - org[1],
                         z = (double)(C.m[1] & 0xffffu) - org[2];
            const double r = (double)__builtin_bit_cast(_Float16, (unsigned short)(C.m[2] & 0xffffu));
            if (!(C.m[2] >> 28)) far[k] = fmin(far[k], sqrt(x * x + y * y + z * z) + r);
        } else {
            const uint32_t first = leaf >> LEAF_SHIFT, c = leaf & LEAF_MASK;
            double reach = 0.0;
            for (uint32_t i = first + (c * k >> 2); i < first + (c * (k + 1) >> 2); ++i) {
                if (growth_edge(tris[i]) > big) continue;
                for (int p = 0; p < 3; ++p) {
                    q = 0.0;
                    for (int a = 0; a < 3; ++a) {
                        const double x = ((double)shade[i].v[p][a] - lo[a]) * scale - org[a];
                        q += x * x;
                    }
                    reach = fmax(reach, sqrt(q));
                }
            }
            far[k] = fmin(far[k], reach);
        }
    }
    double e;
    const uint32_t flags = flag_children(v, B.used, size, A.reach, e);
    const uint32_t all = (half_up(fmax(fmax(v[0], v[1]), fmax(v[2], v[3]))) + 7u) >> 3;
    // D, and one unit more for the roundings of a walk's distance to the origin
    double d = 0.0;
    for (int k = 0; k < 4; ++k)
        if (B.used[k] && !(flags >> k & 1u)) d = fmax(d, far[k]);
    d += 1.0;
    uint4 *o = reinterpret_cast<uint4 *>(out + (L.off + j));
    o[0] = make_uint4(pl[0][0], pl[0][1], pl[0][2], pl[0][3]);
    o[1] = make_uint4(pl[1][0], pl[1][1], pl[1][2], pl[1][3]);
    o[2] = make_uint4(pl[2][0], pl[2][1], pl[2][2], pl[2][3]);
    o[3] = make_uint4((uint32_t)org[0] | ((uint32_t)org[1] << 16),
                      (uint32_t)org[2] | (half_up(e) << 16), half_up(d) | (all << 16) | (flags << 28), ref);
}

__global__ __launch_bounds__(256) void k_wide_build(WideBuild A, WideLevel L) {
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    if (j < (1u << L.level)) wide_node(A, L, j);
}

// All levels of a small tree in one block, children first.  A scene of
// 1000 triangles is made in 161 us with it, in 214 with a launch a level, and in
// 113 without the tree.
constexpr int SMALL_LEVELS = 6;  // levels of at most 2^10 nodes
struct WideLevels {
    WideLevel l[SMALL_LEVELS];
    int32_t n;
};
__global__ __launch_bounds__(1024) void k_wide_build_small(WideBuild A, WideLevels W) {
    for (int i = W.n - 1; i >= 0; --i) {
        const WideLevel L = W.l[i];
        if (threadIdx.x < (1u << L.level)) wide_node(A, L, threadIdx.x);
        __threadfence_block();
        __syncthreads();
    }
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

// Where most triangles lie, whatever a few far ones (a ground) span: the mean
// of up to 1024 of them and the side of a uniform distribution of their spread.
// big: 16 times their median |e2|.  A scene of so few triangles has its larger
// ones' slots (at most MAX_BIG, else none) in the record of the heap's node 0,
// which no walk reads; k_wide_build finds those of others.
WideCore wide_core(HostScene &h) {
    const int64_t n = std::min<int64_t>(h.n, 1024);
    WideCore c;
    c.reach = 0.0;
    for (int a = 0; a < 3; ++a) {
        double s = 0.0, q = 0.0, m = 0.0;
        const double l = h.root_lo[a];
        for (int64_t i = 0; i < n; ++i) {
            const double x = (double)h.tris[i * h.n / n].p[a] - l;
            if (!(fabs(x) < 1e30)) continue;
            s += x, q += x * x, m += 1.0;
        }
        c.mid[a] = l + (m > 0.0 ? s / m : 0.0);
        if (m > 0.0) c.reach = std::max(c.reach, sqrt(std::max(0.0, 12.0 * (q / m - s / m * (s / m)))));
    }
    std::vector<double> e((size_t)n);
    for (int64_t i = 0; i < n; ++i) e[(size_t)i] = growth_edge(h.tris[i * h.n / n]);
    std::vector<double> o(e);
    std::nth_element(o.begin(), o.begin() + n / 2, o.end());
    c.big = 16.0 * o[(size_t)(n / 2)];
    c.n_big = h.n == n ? 0 : -1;
    if (c.n_big == 0) {
        uint32_t *slots = reinterpret_cast<uint32_t *>(h.pairs.data()) + 1;
        for (int64_t i = 0; i < n && c.n_big >= 0; ++i)
            if (e[(size_t)i] > c.big) {
                if (c.n_big == (int)MAX_BIG)
                    c.n_big = -2;
                else
                    slots[c.n_big++] = (uint32_t)i;
            }
        if (c.n_big < 0) c.n_big = 0, c.big = INFINITY;  // too many: the tree bounds them all
    }
    return c;
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
// more (a run's reference), coordinates outside wide_range, and sizes that
// WIDE_SCENE excludes.  flat: where
// append_flat put the records, or 0.
int32_t build_wide(rm_scene *s, size_t flat, const WideCore &core) {
    SceneView &v = s->view;
    v.wide = nullptr;
    v.flat = 0;
    v.flat_tris = nullptr;
    v.n_big = 0;
    v.big = nullptr;
    const HostScene &h = s->host;
    float ext, mag;
    if (h.n >= (int64_t(1) << 25) || !wide_range(h, ext, mag)) return RM_OK;
    if (flat) {
        v.flat = (int32_t)h.n;
        v.flat_b = 3.0f * mag;
        v.flat_tris = reinterpret_cast<const FlatTri *>(s->tris.as<char>() + flat);
        return RM_OK;
    }
    if (!(WIDE_ERR * core.reach <= WIDE_SCENE)) return RM_OK;
    const int e = (int)floor(log2(30000.0 / (double)ext));
    const double scale = ldexp(1.0, e);
    for (int a = 0; a < 3; ++a) v.wide_lo[a] = (float)((double)h.root_lo[a] - 1000.0 / scale);
    v.wide_scale = (float)scale;
    v.wide_rscale = (float)(1.0 / scale);
    for (int a = 0; a < 3; ++a) v.wide_mid[a] = (float)((core.mid[a] - v.wide_lo[a]) * scale);
    v.wide_reach = (float)(core.reach * scale);
    const int leaf_level = h.depth - 1;  // the deepest leaves' level
    std::vector<WideLevel> levels;
    uint32_t total = 0;
    for (int l = 0; l <= leaf_level;) {
        const int step = l == 0 && (leaf_level & 1) ? 1 : 2;
        levels.push_back(WideLevel{l, step, total, total + std::max(4u, 1u << l)});
        total = levels.back().child;
        l += step;
    }
    // a scene that fits without the tree walks the binary one
    const int32_t rc = s->wide.alloc((size_t)total * sizeof(WideNode));
    if (rc) return rc == RM_ERR_OOM ? RM_OK : rc;
    static_assert((1 + MAX_BIG) * sizeof(uint32_t) <= sizeof(PairNode), "room for the slots in node 0's record");
    uint32_t *found = s->nodes.as<uint32_t>();
    double big = core.big;
    uint32_t got = 0, *pin = nullptr;
    std::unique_lock<std::mutex> lock;
    if (core.n_big < 0) {
        // the number found comes back in pinned memory, kept until the process
        // ends (a copy's wait takes 40 us more); one scene at a time
        static std::mutex mu;
        static uint32_t *kept = nullptr;
        lock = std::unique_lock<std::mutex>(mu);
        if (!kept) RM_HIP(hipHostMalloc((void **)&kept, sizeof(uint32_t), hipHostMallocPortable));
        pin = kept;
    }
    while (true) {
        const WideBuild A{v.nodes, s->tris.as<TriRec>(), v.shade, s->wide.as<WideNode>(),
                          {v.wide_lo[0], v.wide_lo[1], v.wide_lo[2]}, scale, core.reach, big,
                          core.n_big < 0 ? found : nullptr, pin};
        if (leaf_level <= 10) {
            WideLevels W{};
            W.n = (int32_t)levels.size();
            std::copy(levels.begin(), levels.end(), W.l);
            hipLaunchKernelGGL(k_wide_build_small, dim3(1), dim3(1024), 0, nullptr, A, W);
        } else {
            for (size_t i = levels.size(); i-- > 0;)  // children first: their E
                hipLaunchKernelGGL(k_wide_build, dim3(((1u << levels[i].level) + 255) / 256), dim3(256), 0, nullptr, A,
                                   levels[i]);
        }
        RM_HIP(hipGetLastError());
        // the caller may use the scene on any stream next
        RM_HIP(hipStreamSynchronize(nullptr));
        got = core.n_big < 0 ? *pin : (uint32_t)core.n_big;
        if (got <= MAX_BIG) break;
        big = INFINITY;  // as in wide_core
        RM_HIP(hipMemset(found, 0, sizeof(PairNode)));
    }
    v.n_big = (int32_t)got;
    v.big = found + 1;
    v.wide = s->wide.as<WideNode>();
    return RM_OK;
}

}  // namespace rm
