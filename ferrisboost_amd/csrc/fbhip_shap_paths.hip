// fbhip_shap_paths.hip -- TreeSHAP contributions and interactions of trees of
// at most SHAP_PATHS_DEPTH split levels, without divides on the path.
//
// Notation. A path feature i has the zero fraction z_i (the product of its
// branch weights along the path) and the one fraction o_i (1 when the row
// meets every one of its splits). With p_i = o_i / z_i - 1, which is
// a_i = 1/z_i - 1 or -1, a leaf contributes to feature i
//     v * prod(z) * Integral_0^1 p_i * prod_{j != i} (1 + p_j t) dt
// (src/model/explain.rs:141-401 takes the same integral by an 8-point rule).
// The integrand has degree at most 7 for 8 distinct features, so the 4-point
// Gauss-Legendre rule gives it exactly.
//
// For a node with children L and R, let C(t) be the product of the factors
// above it (times the quadrature weight) and Q(t) the sum over the leaves
// below it of v * prod(z) * the product of the factors below it. Then
//     D = p_L Q_L + p_R Q_R,   Q = Q_L + Q_R + t D,
//     phi[feature] += sum_q C_q D_q,   C_L = C + p_L (t C),  C_R = C + p_R (t C):
// 8 multiply-adds a node and quadrature point, no divide and no select but the
// two p. A node whose children are both leaves needs D and phi once, not at
// every point. A feature that comes back on a path divides its older factor out
// (1 / (1 + P t), P the older p): the only reciprocals, on those nodes alone.
//
// Every row visits every node, so a wave of 64 rows walks each tree's split
// nodes in preorder with the node's constants in scalar registers, requested one
// node ahead; the only per-row input is one go-left bit a node, which
// shap_masks_kernel has left as one 64-bit lane mask a (64 rows, node): a scalar
// load that the select reads as it is. A wave's sums live in LDS, one float a
// (feature, row), added with ds_add_f32 (each address has one writer, so the
// order is the program's); trees are split into at most SHAP_PATHS_CHUNKS runs,
// one wave each, whose sums are added in a fixed order, so that a few thousand
// rows fill the device and the values do not depend on the number of rows.
//
// Measured against the host-order kernels (8 points with correctly rounded divides,
// the path in registers or scratch, the row's sums read and written in place for
// every tree): contributions of 100k rows x 200 features, 100 trees of depth 8,
// 61.8 -> 17.4 ms; 20k x 28, 300 trees of depth 6, 39.0 -> 2.7 ms of kernels;
// interactions of 2,000 x 28, 100 trees of depth 6, 48.5 -> 0.5 ms of kernels. Error
// against 64-bit results: 2.0e-7 -> 1.4e-7, 3.3e-7 -> 2.1e-7, 3.9e-7 -> 2.1e-7.
// Bound: the latency of a wave's chain at the waves a CU holds. The sums of 200
// features take 52 KB of LDS a wave, so a CU has three waves; each waits in 53 % of its
// cycles and VALU issue is 18 % of its peak (counters of 55,872 rows). Of 10.9 ms a
// batch the masks take 1.4, scalar work for the most part.

#include "fbhip_internal.h"

#include <algorithm>

namespace fbh {

// v_writelane_b32, which has no builtin here: `old` with `v` in lane `lane`.
extern __device__ uint32_t write_lane(uint32_t v, uint32_t lane,
                                      uint32_t old) __asm("llvm.amdgcn.writelane.i32");

namespace {

constexpr int D_MAX = SHAP_PATHS_DEPTH;
constexpr int Q4 = 4;
// 4-point Gauss-Legendre nodes and weights on [0, 1].
__device__ constexpr float T4[Q4] = {0.0694318442029737f, 0.330009478207572f, 0.669990521792428f,
                                     0.930568155797026f};
__device__ constexpr float W4[Q4] = {0.173927422568727f, 0.326072577431273f, 0.326072577431273f,
                                     0.173927422568727f};
// Floats between two features of a wave's LDS sums: odd, so that the lanes of
// both the additions (consecutive rows) and the write-out (consecutive
// features) fall in distinct banks.
constexpr uint32_t TILE_PITCH = SHAP_PATHS_PITCH;

typedef __attribute__((address_space(4))) const PathTestDev *TestP;
typedef __attribute__((address_space(4))) const uint64_t *MaskP;
typedef __attribute__((address_space(3))) float *LdsP;

// One wave's position in a tree.
template <bool INTER>
struct Walk {
    const unsigned char *nodes;  // the next split node in preorder (the same for
    uint32_t at;                 // every lane, in vector registers), at byte `at`
    PathNodeDev next;
    MaskP masks;                 // and its lane mask
    uint64_t next_mask;
    float p[D_MAX];     // the path's p by depth
    // interactions: p / (1 + p t) of the path, and its features
    float e[INTER ? D_MAX : 1][Q4];
    uint32_t feat[INTER ? D_MAX : 1];
    LdsP tile;          // contributions: the lane's column of the LDS sums
    float *pairs;       // interactions: the lane's column of the pair sums
};

// The node at byte `at` of the tree's nodes. A node's constants are operands of
// selects and multiply-adds that take one scalar register at most, so they are
// loaded as vectors (every lane the same 32 bytes).
__device__ __forceinline__ PathNodeDev load_node(const unsigned char *nodes, uint32_t at) {
    const float4 *p = reinterpret_cast<const float4 *>(nodes + at);
    const float4 x = p[0], y = p[1];
    PathNodeDev n;
    n.meta = __float_as_uint(x.x);
    n.al = x.y;
    n.ar = x.z;
    n.vl = x.w;
    n.vr = y.x;
    n.s0 = y.y;
    return n;
}

// Index of an unordered pair of features in the triangular pair sums.
__device__ __forceinline__ uint32_t pair_of(uint32_t a, uint32_t b) {
    const uint32_t hi = max(a, b), lo = min(a, b);
    return hi * (hi + 1) / 2 + lo;
}

template <int D, bool INTER>
__device__ __forceinline__ void visit(Walk<INTER> &w, const float (&c_in)[Q4], float (&Q)[Q4]) {
    PathNodeDev r = w.next;
    const bool left = __builtin_amdgcn_inverse_ballot_w64(w.next_mask);
    r.meta = __builtin_amdgcn_readfirstlane(r.meta);
    w.at += sizeof(PathNodeDev);
    w.masks++;
    w.next = load_node(w.nodes, w.at);
    w.next_mask = *w.masks;
    float pl = left ? r.al : -1.0f, pr = left ? -1.0f : r.ar;
    float c[Q4], inv[Q4], old;
#pragma unroll
    for (int q = 0; q < Q4; q++) c[q] = c_in[q];
    const bool again = D > 0 && (r.meta & PATH_AGAIN);
    if (again) {
        const uint32_t a = (r.meta >> PATH_OLDER) & 7u;
        old = w.p[0];
#pragma unroll
        for (int k = 1; k < D; k++) {
            const float pk = w.p[k];
            old = a == (uint32_t)k ? pk : old;
        }
        const bool met = old > -1.0f;  // 1/z - 1 where the older splits are met, else -1
        pl = met ? pl : -1.0f;
        pr = met ? pr : -1.0f;
#pragma unroll
        for (int q = 0; q < Q4; q++) {
            inv[q] = __builtin_amdgcn_rcpf(__builtin_fmaf(old, T4[q], 1.0f));
            c[q] *= inv[q];
        }
    }
    // what the leaf children give (vl, vr are 0 for a split child)
    const float d0 = __builtin_fmaf(pl, r.vl, pr * r.vr);
    float d[Q4], phi;
    const bool leaves = (r.meta & (PATH_LEAF_L | PATH_LEAF_R)) == (PATH_LEAF_L | PATH_LEAF_R);
    if (D == D_MAX - 1 || leaves) {
#pragma unroll
        for (int q = 0; q < Q4; q++) {
            Q[q] = __builtin_fmaf(T4[q], d0, r.s0);
            if (INTER) d[q] = d0;
        }
        phi = d0 * ((c[0] + c[1]) + (c[2] + c[3]));
    } else {
        float s[Q4];
#pragma unroll
        for (int q = 0; q < Q4; q++) {
            s[q] = r.s0;
            d[q] = d0;
        }
        if (INTER) w.feat[INTER ? D : 0] = r.meta >> PATH_FEATURE;
#pragma unroll 1
        for (uint32_t side = 0; side < 2; side++) {
            asm volatile("" : "+s"(r.meta));
            if ((r.meta >> side) & 1u) continue;  // a leaf
            const float p = side ? pr : pl;
            w.p[D] = p;
            float cc[Q4], qc[Q4];
#pragma unroll
            for (int q = 0; q < Q4; q++) {
                // t C is taken anew for the second child: held across the
                // first it costs four registers a level
                asm volatile("" : "+v"(c[q]));
                cc[q] = __builtin_fmaf(c[q] * T4[q], p, c[q]);
                if (INTER)
                    w.e[INTER ? D : 0][q] = p * __builtin_amdgcn_rcpf(__builtin_fmaf(p, T4[q], 1.0f));
            }
            if constexpr (D + 1 < D_MAX) visit<D + 1, INTER>(w, cc, qc);
#pragma unroll
            for (int q = 0; q < Q4; q++) {
                s[q] += qc[q];
                d[q] = __builtin_fmaf(p, qc[q], d[q]);
            }
        }
        phi = 0.0f;
#pragma unroll
        for (int q = 0; q < Q4; q++) {
            Q[q] = __builtin_fmaf(T4[q], d[q], s[q]);
            phi = __builtin_fmaf(c[q], d[q], phi);
        }
    }
    // keeps the tests of r.meta below from being taken, and held, before the
    // children
    asm volatile("" : "+s"(r.meta));
    if (D > 0 && (r.meta & PATH_AGAIN)) {
        float sub = 0.0f;
#pragma unroll
        for (int q = 0; q < Q4; q++) {
            Q[q] *= inv[q];
            sub = __builtin_fmaf(c[q], Q[q], sub);
            if (INTER) d[q] = __builtin_fmaf(-old, Q[q], d[q]);
        }
        phi = __builtin_fmaf(-old, sub, phi);
    }
    if (!INTER) {
        __builtin_amdgcn_ds_faddf(w.tile + (r.meta >> PATH_FEATURE) * TILE_PITCH, phi, 0, 0, false);
        return;
    }
    const uint32_t feat = r.meta >> PATH_FEATURE;
    unsafeAtomicAdd(w.pairs + (uint64_t)pair_of(feat, feat) * 64, phi);
#pragma unroll
    for (int k = 0; k < D; k++)
        if ((r.meta >> (PATH_PARTNERS + k)) & 1u) {
            float x = 0.0f;
#pragma unroll
            for (int q = 0; q < Q4; q++) x = __builtin_fmaf(c[q] * d[q], w.e[INTER ? k : 0][q], x);
            unsafeAtomicAdd(w.pairs + (uint64_t)pair_of(feat, w.feat[INTER ? k : 0]) * 64, x);
        }
}

// One wave: 64 rows (blockIdx.x) through one run of trees (blockIdx.y).
// Contributions: part[run][row][nf], row-major. Interactions: the zeroed pair
// sums part[run][tile][pair][64].
template <bool INTER>
__global__ __launch_bounds__(64) void shap_paths_kernel(
    const PathNodeDev *nodes, const uint32_t *__restrict__ first, uint32_t n_trees,
    uint32_t run_trees, const uint64_t *masks, uint32_t stride, uint32_t n_rows, uint32_t nf,
    float *__restrict__ part) {
    extern __shared__ float sums[];
    const uint32_t lane = threadIdx.x, tile = blockIdx.x, run = blockIdx.y;
    Walk<INTER> w;
    w.tile = (LdsP)(sums + lane);
    w.pairs = part + ((uint64_t)run * gridDim.x + tile) * (nf * (nf + 1) / 2) * 64 + lane;
    if (!INTER)
        for (uint32_t f = 0; f < nf; f++) sums[f * TILE_PITCH + lane] = 0.0f;
    const uint32_t t1 = min(n_trees, (run + 1) * run_trees);
    for (uint32_t t = run * run_trees; t < t1; t++) {
        const uint32_t b = first[t];
        if (b == first[t + 1]) continue;  // a single leaf contributes to no feature
        w.nodes = reinterpret_cast<const unsigned char *>(nodes + b);
        w.at = 0;
        asm volatile("" : "+v"(w.at));
        w.masks = (MaskP)(masks + ((uint64_t)tile * n_trees + t) * stride);
        w.next = load_node(w.nodes, w.at);
        w.next_mask = *w.masks;
        float c[Q4], q[Q4];
#pragma unroll
        for (int i = 0; i < Q4; i++) c[i] = W4[i];
        visit<0, INTER>(w, c, q);
    }
    if (INTER) return;
    __syncthreads();  // one wave; orders the additions before the reads
    const uint32_t nr = min(64u, n_rows - tile * 64);
    float *o = part + ((uint64_t)run * n_rows + (uint64_t)tile * 64) * nf;
    for (uint32_t r = 0; r < nr; r++)
        for (uint32_t f = lane; f < nf; f += 64) o[r * nf + f] = sums[f * TILE_PITCH + r];
}

// categorical::goes_left (src/data/categorical.rs:334-370) of a value that is
// not NaN: a listed category goes right.
__device__ __forceinline__ bool cat_left(float v, const uint32_t *words, uint32_t len) {
    if (v < 0.0f || v >= 16777216.0f) return true;
    const uint32_t cat = (uint32_t)v;
    return cat / 32 >= len || !((words[cat / 32] >> (cat % 32)) & 1u);
}

// The go-left lane masks of 64 rows (blockIdx.x) for every split node, in the
// trees' preorder: mask[(tile * n_trees + tree) * stride + node]. The rows are
// staged in LDS with an odd stride (a feature's 64 cells in distinct banks); a
// node's test is one comparison whose 64 results are the mask, and lane i of the
// wave keeps node i's mask, so a wave writes 64 masks at once.
__global__ __launch_bounds__(256) void shap_masks_kernel(
    const PathTestDev *tests, const uint32_t *__restrict__ first, uint32_t n_trees,
    const uint32_t *__restrict__ cats, const float *__restrict__ rows, uint32_t n_rows,
    uint32_t nf, uint32_t stride, uint64_t *__restrict__ masks) {
    extern __shared__ float xs[];
    const uint32_t S = nf | 1u, lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile = blockIdx.x, nr = min(64u, n_rows - tile * 64);
    const float *src = rows + (uint64_t)tile * 64 * nf;
    // Cells tid, tid + 256, ... of the rows' contiguous memory (rows past the last repeat
    // it), eight requested before the first is put down. One at a time they were 160
    // waits in turn for 64 rows of 600 features: one tree's contributions 146 -> 105 us a
    // call, of 64 x 200 read over the link 101 -> 66.
    const uint32_t cells = 64 * nf, dr = 256 / nf, df = 256 - dr * nf;
    uint32_t r = threadIdx.x / nf, f = threadIdx.x - r * nf;
    for (uint32_t i = threadIdx.x; i < cells; i += 8 * 256) {
        float v[8];
        uint32_t at[8];
#pragma unroll
        for (uint32_t k = 0; k < 8; k++) {
            const bool in = i + k * 256 < cells;
            v[k] = src[in ? min(r, nr - 1) * nf + f : 0u];
            at[k] = r * S + f;
            r += dr;
            f += df;
            if (f >= nf) {
                f -= nf;
                r++;
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < 8; k++)
            if (i + k * 256 < cells) xs[at[k]] = v[k];
    }
    __syncthreads();
    const float *x = xs + lane * S;
    for (uint32_t t = blockIdx.y * 4 + wave; t < n_trees; t += 4 * gridDim.y) {
        const uint32_t b = first[t], n = first[t + 1] - b;
        const TestP test = (TestP)(tests + b);
        uint64_t *out = masks + ((uint64_t)tile * n_trees + t) * stride;
        for (uint32_t j0 = 0; j0 < n; j0 += 64) {
            const uint32_t m = min(64u, n - j0);
            uint32_t lo = 0, hi = 0;
            // eight nodes at a time, their cells all requested before the
            // first is compared; tests past the tree's last are not stored
            for (uint32_t j1 = 0; j1 < m; j1 += 8) {
                uint32_t ff[8];
                float cond[8], v[8];
#pragma unroll
                for (uint32_t k = 0; k < 8; k++) {
                    ff[k] = test[j0 + j1 + k].ff;
                    cond[k] = test[j0 + j1 + k].cond;
                }
#pragma unroll
                for (uint32_t k = 0; k < 8; k++) v[k] = x[ff[k] & PATH_FEAT];
#pragma unroll
                for (uint32_t k = 0; k < 8; k++) {
                    uint64_t g;
                    if (ff[k] & PATH_CAT) {
                        const TestP c = test + j0 + j1 + k;
                        g = __ballot(v[k] != v[k] ? (ff[k] & PATH_DEFAULT_LEFT) != 0
                                                  : cat_left(v[k], cats + c->cat_offset, c->cat_len));
                    } else if (ff[k] & PATH_DEFAULT_LEFT) {
                        g = ~__ballot(v[k] >= cond[k]);  // NaN is not >= anything: left
                    } else {
                        g = __ballot(v[k] < cond[k]);
                    }
                    lo = write_lane((uint32_t)g, j1 + k, lo);
                    hi = write_lane((uint32_t)(g >> 32), j1 + k, hi);
                }
            }
            if (lane < m) out[j0 + lane] = (uint64_t)hi << 32 | lo;
        }
    }
}

// The runs' sums in run order, and the bias column.
__global__ __launch_bounds__(256) void shap_paths_sum_kernel(
    const float *__restrict__ part, uint32_t runs, uint32_t n_rows, uint32_t nf,
    const float *__restrict__ margin, float bias, float root_mean, float *__restrict__ out) {
    const uint32_t nc = nf + 1;
    const uint64_t total = (uint64_t)n_rows * nc;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < total;
         i += (uint64_t)gridDim.x * 256) {
        const uint32_t row = (uint32_t)(i / nc), f = (uint32_t)(i - (uint64_t)row * nc);
        float v;
        if (f == nf) {
            v = root_mean + (margin ? margin[row] : bias);
        } else {
            v = 0.0f;
            for (uint32_t k = 0; k < runs; k++)
                v += part[((uint64_t)k * n_rows + row) * nf + f];
        }
        out[i] = v;
    }
}

// One wave: 64 rows (blockIdx.x) of matrix line blockIdx.y, from the runs' pair
// sums in run order. An unordered pair's sum is shared by its two cells
// (interaction_row, src/model/explain.rs:790-810); the diagonal is the feature's
// contribution less its line's interactions.
__global__ __launch_bounds__(64) void shap_pairs_out_kernel(
    const float *__restrict__ part, uint32_t runs, uint32_t n_rows, uint32_t nf,
    const float *__restrict__ margin, float bias, float root_mean, float *__restrict__ out) {
    const uint32_t lane = threadIdx.x, tile = blockIdx.x, r = blockIdx.y, nc = nf + 1;
    const uint32_t row = tile * 64 + lane;
    if (row >= n_rows) return;
    float *o = out + ((uint64_t)row * nc + r) * nc;
    if (r == nf) {
        for (uint32_t c = 0; c < nf; c++) o[c] = 0.0f;
        o[nf] = root_mean + (margin ? margin[row] : bias);
        return;
    }
    const uint32_t pairs = nf * (nf + 1) / 2;
    auto sum = [&](uint32_t pair) {
        float v = 0.0f;
        for (uint32_t k = 0; k < runs; k++)
            v += part[(((uint64_t)k * gridDim.x + tile) * pairs + pair) * 64 + lane];
        return v;
    };
    float diag = sum(pair_of(r, r));
    for (uint32_t c = 0; c < nf; c++) {
        if (c == r) continue;
        const float v = 0.5f * sum(pair_of(r, c));
        o[c] = v;
        diag -= v;
    }
    o[r] = diag;
    o[nf] = 0.0f;
}

hipError_t opt_in_lds(const void *fn) {
    return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
}

}  // namespace

uint64_t shap_paths_tile_bytes(const ShapPaths &m, bool inter) {
    const uint64_t masks = 8ull * m.n_trees * m.stride;
    const uint64_t nf = m.n_features;
    return masks + 256ull * m.runs * (inter ? nf * (nf + 1) / 2 : nf);
}

hipError_t launch_shap_paths(const ShapPaths &m, bool inter, const float *rows, uint64_t n_rows,
                             const float *margin, float *out, void *work, uint64_t work_bytes,
                             hipStream_t s) {
    const uint64_t per_tile = shap_paths_tile_bytes(m, inter);
    const uint64_t cap = std::min<uint64_t>(work_bytes / per_tile, 1u << 16);
    if (cap == 0) return hipErrorInvalidValue;
    const uint32_t nf = m.n_features, nc = nf + 1;
    const size_t xs = (size_t)256 * (nf | 1u);
    const size_t sums = inter ? 0 : (size_t)4 * TILE_PITCH * nf;
    hipError_t e;
    if (xs > 64 * 1024 &&
        (e = opt_in_lds(reinterpret_cast<const void *>(&shap_masks_kernel))) != hipSuccess)
        return e;
    if (sums > 64 * 1024 &&
        (e = opt_in_lds(reinterpret_cast<const void *>(&shap_paths_kernel<false>))) != hipSuccess)
        return e;
    for (uint64_t r0 = 0; r0 < n_rows; r0 += cap * 64) {
        const uint32_t n = (uint32_t)std::min<uint64_t>(cap * 64, n_rows - r0);
        const uint32_t tiles = (n + 63) / 64;
        uint64_t *masks = static_cast<uint64_t *>(work);
        float *part = reinterpret_cast<float *>(masks + (uint64_t)tiles * m.n_trees * m.stride);
        const float *x = rows + r0 * nf, *mg = margin ? margin + r0 : nullptr;
        // 768 workgroups of four waves fill the device; fewer tiles share
        // their trees among several
        const uint32_t split = std::min((m.n_trees + 3) / 4, std::max(1u, 768u / tiles));
        hipLaunchKernelGGL(shap_masks_kernel, dim3(tiles, split), dim3(256), xs, s, m.tests,
                           m.first, m.n_trees, m.cats, x, n, nf, m.stride, masks);
        if (!inter) {
            hipLaunchKernelGGL(shap_paths_kernel<false>, dim3(tiles, m.runs), dim3(64), sums, s,
                               m.nodes, m.first, m.n_trees, m.run_trees, masks, m.stride, n, nf,
                               part);
            const uint64_t blocks = ((uint64_t)n * nc + 255) / 256;
            hipLaunchKernelGGL(shap_paths_sum_kernel, dim3((uint32_t)std::min<uint64_t>(blocks, 1u << 20)),
                               dim3(256), 0, s, part, m.runs, n, nf, mg, m.bias, m.root_mean,
                               out + r0 * nc);
        } else {
            const uint64_t cells = (uint64_t)m.runs * tiles * (nf * (uint64_t)(nf + 1) / 2) * 64;
            if ((e = launch_fill_f32(part, 0.0f, cells, s)) != hipSuccess) return e;
            hipLaunchKernelGGL(shap_paths_kernel<true>, dim3(tiles, m.runs), dim3(64), sums, s,
                               m.nodes, m.first, m.n_trees, m.run_trees, masks, m.stride, n, nf,
                               part);
            hipLaunchKernelGGL(shap_pairs_out_kernel, dim3(tiles, nc), dim3(64), 0, s, part, m.runs,
                               n, nf, mg, m.bias, m.root_mean, out + r0 * (uint64_t)nc * nc);
        }
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace fbh
