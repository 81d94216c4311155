// fbhip_predict.hip -- prediction with a workgroup's rows and a run of whole
// trees in LDS (predict_margin_soa[_cat], src/backend/cuda/histogram.cu:
// 2459-2494, 3600-3642; leaf_row, src/model/explain.rs:689-702).
//
// A walk is a chain of two dependent gathers a node, the node and the row's cell
// of its feature. From global memory and LDS (predict_lds4_kernel) a step took
// about 150 cycles of a CU a wave, most of it the node's way through L1 and L2.
// Here both are LDS reads, and a wave walks ILP trees of a row at once, so
// that one chain's latency covers the others'. Nodes are 8 bytes, a node's
// children side by side; a leaf's child is itself, so that trees of different
// depth walk in step. Cells are staged as order-preserving keys, so that one
// unsigned comparison decides a node, missing values among them: nine vector
// instructions a step. The next run of trees and the next rows are requested into
// registers while the current ones are walked.
//
// One workgroup a CU holds the rows and a run of up to 32 trees: the walks in flight
// are rows times trees, and a CU's LDS split between the two in one piece holds
// twice as many as in two halves. Its 16 waves share one, two or four groups of 64
// rows (as many as fit: each group reads the trees once more) and take a group's
// trees in turn, their leaf values meeting in LDS, where one wave adds a row's
// values in tree order, the host's f32 additions (Model::predict_margin,
// src/model/tree.rs:486-510). Calls of too few rows to fill the device split the
// runs over workgroups, which leave each tree's value in memory for
// predict_sum_kernel.
//
// Measured (margins; predict_lds4_kernel before): 1M x 200, 100 trees of depth 8
// 2.92 -> 1.08 ms; 200k x 50 with 6 categorical features, 300 trees of depth 6
// 0.67 -> 0.56 ms; 64 x 28, 100 trees of depth 6 124 -> 12 us with the sum kernel.
// VALU issue is 38 % of its peak and a wave waits in 56 % of its cycles: what remains
// is the latency of a step's two reads and each run's barriers. Where a run holds few
// trees, most waves have no walk, and predict_tiles_pay leaves the call to
// predict_lds4_kernel or predict_kernel.

#include "fbhip_internal.h"
#include "fb_expf.h"

#include <algorithm>
#include <cmath>

namespace fbh {

namespace {

constexpr int WAVES = 16;
constexpr int TPB = 64 * WAVES;
constexpr int ILP = 2;
constexpr int BATCH = WAVES * ILP;  // (tree, 64 rows) walks in flight
// The next tile's cells and the next run's nodes a thread holds while the
// current ones are walked: 64 rows of 208 features, 128 of 104 and 256 of 52; wider
// rows load the rest between two barriers, and more registers would leave fewer waves.
// 200k rows, one run of 8 trees of 63 nodes: 28 features 36 us (22 MB), 200 61 (160 MB,
// 3.5 TB/s beside the launch), 400 139 (320 MB, 2.6).
constexpr int XPRE = 13;
constexpr int NPRE = 7;
static_assert(NPRE * TPB * 2 >= (int)PRED_RUN_NODES, "a run fits its registers");

typedef __attribute__((address_space(4))) const PredRun *RunP;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// A barrier for LDS alone: __syncthreads would also wait for the global loads
// that are meant to arrive during the next walk.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A value's key: unsigned order is the order of <, the two zeros are one, and NaN
// is KEY_NAN, above every other by more than the 2 a default-left node adds to key
// and threshold, which wraps KEY_NAN alone to below every threshold.
constexpr uint32_t KEY_NAN = PRED_KEY_NAN;
__device__ __forceinline__ uint32_t key_of(float v) {
    const uint32_t u = __float_as_uint(v + 0.0f);
    const uint32_t k = u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
    return v != v ? KEY_NAN : k;
}
__device__ __forceinline__ float key_value(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? k ^ 0x80000000u : ~k);
}

template <int G, bool CATS>
__global__ __launch_bounds__(TPB) void predict_tile_kernel(
    const PredTrees P, const float *__restrict__ rows, uint64_t n_rows,
    const float *__restrict__ init, float base, uint32_t mode, float *__restrict__ vals,
    float *__restrict__ out) {
    constexpr int SHARE = WAVES / G;         // waves that share 64 rows
    constexpr uint32_t TREES = SHARE * ILP;  // trees those walk at once
    extern __shared__ uint4 smem[];
    float *leafv = reinterpret_cast<float *>(smem);  // leaf values of a batch
    uint32_t *xs = reinterpret_cast<uint32_t *>(leafv + BATCH * 64);  // cells' keys
    const uint32_t nf = P.n_features, S = nf | 1u, tid = threadIdx.x;
    u32x4 *nodes4 = reinterpret_cast<u32x4 *>(xs + ((G * 64 * S + 3) & ~3u));
    const uint2 *nodes = reinterpret_cast<const uint2 *>(nodes4);
    // a tree's first node, and the words of the run's category sets
    const uint32_t *first = reinterpret_cast<const uint32_t *>(nodes4);
    const uint32_t lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t group = wave / SHARE, turn = wave % SHARE;
    const uint32_t tiles = (uint32_t)((n_rows + 64 * G - 1) / (64 * G));
    // this workgroup's runs (all of them unless the call splits them)
    const uint32_t per = (P.n_runs + gridDim.y - 1) / gridDim.y;
    const uint32_t c0 = min(P.n_runs, blockIdx.y * per), c1 = min(P.n_runs, c0 + per);
    u32x4 npre[NPRE];
    float xpre[XPRE];
    PredRun next{};
    auto request_nodes = [&](uint32_t c) {
        const RunP r = (RunP)P.runs + c;
        next.tree0 = r->tree0;
        next.n_trees = r->n_trees;
        next.node0 = r->node0;
        next.n_nodes = r->n_nodes;
        const u32x4 *src = reinterpret_cast<const u32x4 *>(P.nodes + next.node0);
        const uint32_t n = (next.n_nodes + 1) / 2;
        // past the end the last entry again: a load under a condition would be
        // waited for where it is issued
#pragma unroll
        for (int k = 0; k < NPRE; k++) npre[k] = src[min(tid + k * TPB, n - 1)];
    };
    auto tile_cells = [&](uint32_t tile) {
        return (uint32_t)min<uint64_t>(64 * G, n_rows - (uint64_t)tile * (64 * G)) * nf;
    };
    auto request_rows = [&](uint32_t tile) {
        const float *src = rows + (uint64_t)tile * (64 * G) * nf;
        const uint32_t cells = tile_cells(tile);
#pragma unroll
        for (int k = 0; k < XPRE; k++) xpre[k] = src[min(tid + k * TPB, cells - 1)];
    };
    if (blockIdx.x < tiles) request_rows(blockIdx.x);
    if (c0 < c1) request_nodes(c0);
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint64_t r0 = (uint64_t)tile * (64 * G);
        const uint64_t row = r0 + group * 64 + lane;
        const bool live = row < n_rows;
        const uint64_t lives = __ballot(live);
        const uint32_t *x = xs + (group * 64 + lane) * S;
        lds_barrier();  // the previous tile's walks are done
        {
            // cells tid, tid + TPB, ... of the rows' contiguous memory, to an odd
            // stride (the 64 lanes' cells of one feature fall in distinct banks)
            const float *src = rows + r0 * nf;
            const uint32_t cells = tile_cells(tile), dr = TPB / nf, df = TPB - dr * nf;
            uint32_t r = tid / nf, f = tid - r * nf;
            auto put = [&](float v) {
                xs[r * S + f] = key_of(v);
                r += dr;
                f += df;
                if (f >= nf) {
                    f -= nf;
                    r++;
                }
            };
#pragma unroll
            for (int k = 0; k < XPRE; k++)
                if (tid + k * TPB < cells) put(xpre[k]);
            for (uint32_t i = tid + XPRE * TPB; i < cells; i += TPB) put(src[i]);
        }
        float m = 0.0f;
        if (turn == 0 && live && mode <= PRED_OUT_SIGMOID) {
            m = base;
            if (init) {
                m = init[row];
                asm volatile("" : "+v"(m));  // waited for here, not in the walk
            }
        }
        for (uint32_t c = c0; c < c1; c++) {
            const PredRun run = next;
            if (c > c0) lds_barrier();  // the previous run's walks are done
            if (c1 - c0 > 1 || tile == blockIdx.x) {
#pragma unroll
                for (int k = 0; k < NPRE; k++)
                    if (tid + k * TPB < (run.n_nodes + 1) / 2) nodes4[tid + k * TPB] = npre[k];
                if (c1 - c0 > 1) request_nodes(c + 1 < c1 ? c + 1 : c0);
            }
            if (c + 1 == c1 && tile + gridDim.x < tiles) request_rows(tile + gridDim.x);
            lds_barrier();
            for (uint32_t b = 0; b < run.n_trees; b += TREES) {
                uint32_t idx[ILP], value[ILP];
#pragma unroll
                for (int j = 0; j < ILP; j++)  // past the run's last tree: the last one again
                    idx[j] = first[min(b + turn + j * SHARE, run.n_trees - 1)];
                if (b + turn < run.n_trees)
                    for (;;) {
                        uint2 n[ILP];
#pragma unroll
                        for (int j = 0; j < ILP; j++) n[j] = nodes[idx[j]];
                        uint32_t v[ILP];
                        uint64_t open = 0;
#pragma unroll
                        for (int j = 0; j < ILP; j++) {
                            v[j] = x[(n[j].y >> PRED_FEAT) & PRED_FEAT_MASK];
                            value[j] = n[j].x;
                            open |= __ballot((int32_t)n[j].y >= 0);
                        }
                        if ((open & lives) == 0) break;
#pragma unroll
                        for (int j = 0; j < ILP; j++) {
                            bool right = v[j] + (n[j].y & PRED_DL_BIT) >= n[j].x;
                            if (CATS && (n[j].y & PRED_CAT_BIT)) {
                                // categorical::goes_left (src/data/categorical.rs:334-370);
                                // a missing value's key is that of a NaN, which is not >= 0
                                const float f = key_value(v[j]);
                                right = v[j] == KEY_NAN && !(n[j].y & PRED_DL_BIT);
                                if (f >= 0.0f && f < 16777216.0f) {
                                    const uint32_t cat = (uint32_t)f;
                                    if (cat / 32 < n[j].x >> 16)
                                        right = (first[(n[j].x & 0xFFFFu) + cat / 32] >> (cat % 32)) & 1u;
                                }
                            }
                            right &= (int32_t)n[j].y >= 0;  // a leaf stays
                            idx[j] = ((n[j].y >> PRED_CHILD) & PRED_CHILD_MASK) + (right ? 1u : 0u);
                        }
                    }
                float *lv = leafv + group * TREES * 64 + lane;
#pragma unroll
                for (int j = 0; j < ILP; j++) {
                    const uint32_t k = b + turn + j * SHARE;
                    if (k >= run.n_trees) break;
                    if (mode == PRED_OUT_LEAF) {
                        if (live)
                            out[row * P.n_trees + run.tree0 + k] =
                                (float)P.ids[run.node0 + idx[j]];
                    } else if (mode == PRED_OUT_VALUES) {
                        if (live)
                            vals[(uint64_t)(run.tree0 + k) * n_rows + row] = __uint_as_float(value[j]);
                    } else {
                        lv[(turn + j * SHARE) * 64] = __uint_as_float(value[j]);
                    }
                }
                if (mode > PRED_OUT_SIGMOID) continue;
                lds_barrier();
                if (turn == 0) {
                    const uint32_t n = min(TREES, run.n_trees - b);
                    for (uint32_t k = 0; k < n; k += 8) {
                        float v[8];
#pragma unroll
                        for (uint32_t i = 0; i < 8; i++) v[i] = lv[min(k + i, n - 1) * 64];
#pragma unroll
                        for (uint32_t i = 0; i < 8; i++)
                            if (k + i < n) m += v[i];
                    }
                }
                // (the next run's barriers do this for a run's last batch)
                if (b + TREES < run.n_trees) lds_barrier();
            }
        }
        if (turn == 0 && live && mode <= PRED_OUT_SIGMOID)
            out[row] = mode == PRED_OUT_SIGMOID ? fb_sigmoid(m) : m;
    }
}

// A row's margin from the values of its trees, in tree order.
__global__ __launch_bounds__(64) void predict_sum_kernel(const float *__restrict__ vals,
                                                         uint32_t n_trees, uint32_t n_rows,
                                                         const float *__restrict__ init, float base,
                                                         uint32_t mode, float *__restrict__ out) {
    const uint32_t row = blockIdx.x * 64 + threadIdx.x;
    if (row >= n_rows) return;
    float m = init ? init[row] : base;
    for (uint32_t t0 = 0; t0 < n_trees; t0 += 16) {
        float v[16];
#pragma unroll
        for (uint32_t k = 0; k < 16; k++)
            v[k] = t0 + k < n_trees ? vals[(uint64_t)(t0 + k) * n_rows + row] : 0.0f;
#pragma unroll
        for (uint32_t k = 0; k < 16; k++)
            if (t0 + k < n_trees) m += v[k];
    }
    out[row] = mode == PRED_OUT_SIGMOID ? fb_sigmoid(m) : m;
}

size_t tile_lds(const PredTrees &P, uint32_t g) {
    const size_t cells = ((size_t)64 * g * (P.n_features | 1u) + 3) & ~(size_t)3;
    return 4 * (BATCH * 64 + cells) + 8 * (size_t)((P.most_nodes + 1) & ~1u);
}

template <int G, bool CATS>
hipError_t launch_tile(const PredTrees &P, uint32_t split, const float *rows, uint64_t n,
                       const float *init, float base, uint32_t mode, float *vals, float *out,
                       hipStream_t s) {
    const size_t lds = tile_lds(P, G);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(
            reinterpret_cast<const void *>(&predict_tile_kernel<G, CATS>),
            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
    }
    // one workgroup a CU (its registers), each taking tile after tile
    const uint64_t tiles = (n + 64 * G - 1) / (64 * G);
    hipLaunchKernelGGL((predict_tile_kernel<G, CATS>),
                       dim3((uint32_t)std::min<uint64_t>(tiles, PRED_CUS), split), dim3(TPB), lds, s, P, rows,
                       n, init, base, mode, vals, out);
    return hipGetLastError();
}

template <bool CATS>
hipError_t launch_groups(uint32_t g, const PredTrees &P, uint32_t split, const float *rows,
                         uint64_t n, const float *init, float base, uint32_t mode, float *vals,
                         float *out, hipStream_t s) {
    if (g == 4) return launch_tile<4, CATS>(P, split, rows, n, init, base, mode, vals, out, s);
    if (g == 2) return launch_tile<2, CATS>(P, split, rows, n, init, base, mode, vals, out, s);
    return launch_tile<1, CATS>(P, split, rows, n, init, base, mode, vals, out, s);
}

// The groups of 64 rows a workgroup takes, and the workgroups that share the runs of
// its rows.
struct TileShape {
    uint32_t groups, split;
};
TileShape tile_shape(const PredTrees &P, uint64_t n_rows, uint32_t mode, bool work) {
    const uint64_t tiles = (n_rows + 63) / 64;
    if (work || (mode == PRED_OUT_LEAF && tiles < PRED_FILL_TILES))
        return {1, (uint32_t)std::min<uint64_t>(P.n_runs, (PRED_FILL_TILES + tiles - 1) / tiles)};
    // More groups of 64 rows a workgroup read the trees fewer times; fewer leave
    // less of the device idle in the last round of tiles. The most groups within
    // a tenth of the least rounds' rows.
    uint32_t g = 1;
    uint64_t least = ~0ull;
    for (uint32_t k = 1; k <= P.groups; k *= 2) {
        const uint64_t t = (tiles + k - 1) / k;
        const uint64_t rounds = (t + PRED_CUS - 1) / PRED_CUS * k;
        if (rounds * 10 <= least * 11 || least == ~0ull) g = k;
        least = std::min(least, rounds);
    }
    return {g, 1};
}

}  // namespace

uint64_t predict_tiles_work(const PredTrees &P, uint64_t n_rows, uint32_t mode) {
    const uint64_t tiles = (n_rows + 63) / 64;
    if (mode > PRED_OUT_SIGMOID || P.n_runs < 2 || tiles >= PRED_FILL_TILES) return 0;
    const uint64_t bytes = 4 * n_rows * P.n_trees;
    return bytes <= PRED_WORK_BYTES ? bytes : 0;
}

// Estimates in microseconds. Here a CU takes 2.6 to 4 for a run of trees, whether 16
// waves share 32 small trees or one walks a tree that fills the run, and no less than
// its rows take to arrive. The walks that read the nodes from memory take a time for
// each (tree, 64 rows), longer for deeper trees and, up to 255 features, for the
// fewer workgroups whose rows fit a CU; few rows wait for one tree after the other.
// Measured (200k rows, here against there): 28 features, 8 runs of 1, 5 and 12 trees
// 229, 239, 247 against 68, 149, 258 us; 200 features 401, 395, 419 against 199, 426,
// 711; 400 features, where the other walk reads rows in place, 8 runs of 1 and 2 trees
// 452, 443 against 352, 616, and one run of 1 and 8 trees of 63 nodes 139 against 32
// and 160. Of 201 such measurements (1k to 200k rows, 63 to 12,783 nodes a tree) the
// rule takes a walk more than 7 % slower than the other in three, 16 % at most.
bool predict_tiles_pay(const PredTrees &P, uint64_t n_rows, uint32_t mode) {
    const bool work = predict_tiles_work(P, n_rows, mode) != 0;
    const TileShape shape = tile_shape(P, n_rows, mode, work);
    const double tiles = (double)((n_rows + 63) / 64), nf = P.n_features, trees = P.n_trees;
    const uint64_t blocks = ((n_rows + 63) / 64 + shape.groups - 1) / shape.groups * shape.split;
    const double rounds = (double)((blocks + PRED_CUS - 1) / PRED_CUS);
    const uint32_t runs = (P.n_runs + shape.split - 1) / shape.split;
    const bool in_lds = P.n_features <= PRED_LDS4_MAX_F;
    if (in_lds && rounds == 1 && runs == 1) return true;
    const double fill = std::min(1.0, (double)P.n_entries / P.n_runs / PRED_RUN_NODES);
    const double rows_us = in_lds ? 0.011 * nf * shape.groups : 0.0235 * nf;
    const double here = rounds * std::max(runs * (2.6 + 1.4 * fill), rows_us + 0.9) + (work ? 2 : 0);
    const double depth = std::log2(P.n_entries / trees + 1);
    double there;
    if (in_lds) {
        const uint32_t held = std::min(8u, PRED_LDS_BYTES / (256 * ((P.n_features | 1u) + 32)));
        const double each = (0.45 + 5.2 / held) * std::pow(depth / 13.6, 1.5);
        there = std::max(tiles * ((0.11 + 0.0005 * nf) * nf + trees * each) * 1e-3,
                         trees * 0.05 * depth);
    } else {
        there = std::max(tiles * trees * std::min(10.5, depth) * 1e-3, trees * 0.25 * depth);
    }
    return here <= 1.05 * there;
}

hipError_t launch_predict_tiles(const PredTrees &P, const float *rows, uint64_t n_rows,
                                const float *init, float base, uint32_t mode, float *out,
                                void *work, hipStream_t s) {
    if (n_rows == 0) return hipSuccess;
    const uint64_t tiles = (n_rows + 63) / 64;
    const TileShape shape = tile_shape(P, n_rows, mode, work != nullptr);
    const uint32_t g = shape.groups, split = shape.split;
    const uint32_t mk = work ? PRED_OUT_VALUES : mode;
    float *vals = static_cast<float *>(work);
    hipError_t e = P.categorical
                       ? launch_groups<true>(g, P, split, rows, n_rows, init, base, mk, vals, out, s)
                       : launch_groups<false>(g, P, split, rows, n_rows, init, base, mk, vals, out, s);
    if (e != hipSuccess || !work) return e;
    hipLaunchKernelGGL(predict_sum_kernel, dim3((uint32_t)tiles), dim3(64), 0, s, vals, P.n_trees,
                       (uint32_t)n_rows, init, base, mode, out);
    return hipGetLastError();
}

}  // namespace fbh
