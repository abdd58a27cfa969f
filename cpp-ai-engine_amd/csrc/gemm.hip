// gemm.hip -- fp32 GEMM on CDNA4 matrix cores: C = op(A) op(B) + beta C,
// batched, with the transposed operand modes the backward pass needs
// (dA = dC B^T, dB = A^T dC) and a deterministic split-K for tall-skinny
// products such as the convolution weight gradients.
//
// Tiling. Products large enough for staged tiles run gemm_kernel (gemm_split.hpp): fp32
// operands split into three bf16 parts while a tile is staged in LDS, six part products on
// v_mfma_f32_16x16x32_bf16, fp32 accumulation. Products with outputs too small to fill the
// chip that way run the fp32 instructions: K-sliced 32 x 32 tiles (gemm_kslice,
// gemm_kernel.hpp), 16 x 16 panels of a long K, and the vector kernels of the smallest.
//
// MFMA register layout of the fp32 tiles (CDNA3/CDNA4 ISA, v_mfma_f32_32x32x2f32):
//   A operand: lane l holds A[i = l % 32][k = l / 32]
//   B operand: lane l holds B[k = l / 32][j = l % 32]
//   D result : lane l, register r holds D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32]
//
// Ordering. Workgroups are numbered so that consecutive tiles land on the
// same XCD (the hardware deals workgroups round-robin over the 8 XCDs, each
// with its own L2), then grouped GROUP_M tile-rows at a time so neighbours
// share A rows and B columns in that L2.
//
// Determinism. The K order inside a tile is fixed, split-K partials are
// summed in split order by a second kernel: the result depends only on the
// shape. It is not bit-equal to the reference's serial i-k-j loop
// (src/tensor_ops.cpp:539-562); the parity tests bound the difference.

#include <algorithm>
#include <atomic>
#include <mutex>
#include <vector>

#include "gemm_split.hpp"

namespace ehip {
namespace gemm_detail {

// C[b] = sum over splits of W[s][b], then the epilogue; with a column sum,
// the n values after each split's C partials are summed the same way into
// colsum. A block is RL split lanes x (256 / RL) outputs: lane l adds splits
// l, l + RL, ... in order, then one thread per output adds the lanes in
// order. RL grows with the number of splits, so a few outputs with many
// splits still spread over the block instead of one long serial chain per
// output; the order depends only on the shape.
__global__ __launch_bounds__(256) void splitk_reduce(const float* __restrict__ w, float* c,
                                                     GemmArgs g, int64_t batch, int splits,
                                                     int rl) {
    const int64_t m = g.m, n = g.n;
    __shared__ float lanes[256];
    const int cw = 256 / rl;
    const int lane = threadIdx.x / cw, cl = threadIdx.x % cw;
    const int64_t mn = m * n;
    const int64_t e = int64_t(blockIdx.x) * cw + cl;
    const int64_t step = g.ws_stride;
    const int64_t outputs = batch * mn + (g.colsum ? n : 0);
    float acc = 0.0f;
    if (e < outputs && lane < splits) {
        const float* p = w + e + int64_t(lane) * step;
        const int64_t stride = int64_t(rl) * step;
        const int count = (splits - lane + rl - 1) / rl;
        acc = p[0];
        int s = 1;
        for (; s + 8 <= count; s += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = p[int64_t(s + u) * stride];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc += v[u];
        }
        for (; s < count; ++s) acc += p[int64_t(s) * stride];
    }
    lanes[threadIdx.x] = acc;
    __syncthreads();
    if (lane == 0 && e < outputs) {
        float sum = lanes[cl];
        for (int l = 1; l < rl && l < splits; ++l) sum += lanes[l * cw + cl];
        if (e >= batch * mn) {
            g.colsum[e - batch * mn] = sum;
            return;
        }
        const int64_t b = e / mn, rc = e % mn;
        const int64_t row = rc / n, col = rc % n;
        float* dst = c + batch_offset(b, g.inner, g.stride_c, g.stride_c2) + row * g.ldc + col;
        *dst = epilogue(g, b, row, col, sum, dst);
    }
}

// splitk_reduce's sums for up to 8 splits (one split lane) and no column sums,
// four outputs of one row per thread: every split's float4 is loaded before
// the first add, then added in split order -- the same sum per output -- and
// the row and column are decomposed once per four outputs instead of once per
// output (its 64-bit divisions dominated the two-split reductions of the
// 1024 x 4096 weight gradients: 18.7 us for 48 MB).
constexpr int kReduce4MaxSplits = 8;

template <bool PLAIN>
__global__ __launch_bounds__(256) void splitk_reduce4(const float* __restrict__ w, float* c,
                                                      GemmArgs g, int64_t batch, int splits) {
    const int64_t mn = g.m * g.n;
    const int64_t e = 4 * (int64_t(blockIdx.x) * 256 + threadIdx.x);
    if (e >= batch * mn) return;
    float4 v[kReduce4MaxSplits];
#pragma unroll
    for (int sp = 0; sp < kReduce4MaxSplits; ++sp)
        if (sp < splits) v[sp] = *reinterpret_cast<const float4*>(w + e + int64_t(sp) * g.ws_stride);
    float4 acc = v[0];
#pragma unroll
    for (int sp = 1; sp < kReduce4MaxSplits; ++sp) {
        if (sp < splits) {
            acc.x += v[sp].x;
            acc.y += v[sp].y;
            acc.z += v[sp].z;
            acc.w += v[sp].w;
        }
    }
    const int64_t b = batch == 1 ? 0 : e / mn, rc = batch == 1 ? e : e % mn;
    const int64_t row = rc / g.n, col = rc % g.n;
    float* dst = c + batch_offset(b, g.inner, g.stride_c, g.stride_c2) + row * g.ldc + col;
    if (PLAIN) {
        *reinterpret_cast<float4*>(dst) = acc;
        return;
    }
    const float r[4] = {acc.x, acc.y, acc.z, acc.w};
    float o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] = epilogue(g, b, row, col + t, r[t], dst + t);
    *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
}

int splitk_finish(const float* ws, float* out, const GemmArgs& gr, int64_t batch, int splits,
                  hipStream_t s) {
    if (splits <= kReduce4MaxSplits && gr.colsum == nullptr && gr.n % 4 == 0 && gr.ldc % 4 == 0 &&
        gr.stride_c % 4 == 0 && gr.stride_c2 % 4 == 0 && aligned16(out) && aligned16(ws) &&
        batch * gr.m * gr.n / 4 < (int64_t(1) << 39)) {
        const unsigned grid = unsigned(ceil_div(batch * gr.m * gr.n / 4, 256));
        if (plain_epilogue(gr))
            EHIP_LAUNCH("gemm_splitk_reduce", splitk_reduce4<true>, dim3(grid), dim3(256), 0, s,
                        ws, out, gr, batch, splits);
        else
            EHIP_LAUNCH("gemm_splitk_reduce", splitk_reduce4<false>, dim3(grid), dim3(256), 0, s,
                        ws, out, gr, batch, splits);
        return EHIP_OK;
    }
    // Split lanes: up to 16, about one per 8 splits, so that no lane chain
    // is longer than ~8 loads deep when the outputs are few.
    int rl = 1;
    while (rl < 16 && rl * 8 < splits) rl *= 2;
    const int64_t total = gr.ws_stride;  // C partials, then the column sums
    const int64_t per_block = 256 / rl;
    EHIP_LAUNCH("gemm_splitk_reduce", splitk_reduce, dim3(unsigned(ceil_div(total, per_block))),
                dim3(256), 0, s, ws, out, gr, batch, splits, rl);
    return EHIP_OK;
}

}  // namespace gemm_detail
}  // namespace ehip

namespace ehip {
namespace {

using namespace gemm_detail;

// Where split-K partials go: the library's grow-only scratch (base == nullptr),
// or a caller-fixed block of cap_bytes that must hold them (the no-allocation
// entry point).
struct Workspace {
    float* base = nullptr;
    size_t cap_bytes = 0;
};

// The grid's z extent: products beyond it run as further launches.
constexpr int64_t kGridZ = 65535;

template <int BM, int BN, int WM, int WN, int STAGES, int MINW, bool TA, bool TB>
int launch_shape(const GemmArgs& g, const dim3& grid, hipStream_t s) {
    constexpr int kThreads = TileThreads<BM, BN, WM, WN>::value;
    if constexpr (!TB) {  // column sums exist only for a K x N B
        if (g.colsum != nullptr) {
            EHIP_LAUNCH("gemm", (gemm_kernel<BM, BN, WM, WN, STAGES, MINW, TA, TB, true>), grid,
                        dim3(kThreads), 0, s, g);
            return EHIP_OK;
        }
    }
    EHIP_LAUNCH("gemm", (gemm_kernel<BM, BN, WM, WN, STAGES, MINW, TA, TB, false>), grid,
                dim3(kThreads), 0, s, g);
    return EHIP_OK;
}

// A product as staged tiles. The most K splits are planned on bm x bn tiles of bk (the
// planner's class): when the tile grid cannot fill the chip ("fill" is 256 workgroups of the
// largest class and two per CU of the smaller ones) and K is long, up to ~512 workgroups, each
// at least 8 K steps long.
int class_splits(int64_t m, int64_t n, int64_t k, int64_t batch, int bm, int bn, int bk) {
    const int64_t tiles = ceil_div(m, bm) * ceil_div(n, bn) * batch;
    const int64_t fill = bm * bn >= 256 * 256 ? 256 : 512;
    if (tiles >= fill || k < 16 * bk) return 1;
    const int64_t want = std::min({ceil_div(512, tiles), k / (8 * bk), int64_t(256)});
    const int64_t chunk = ceil_div(ceil_div(k, want), bk) * bk;
    return int(ceil_div(k, chunk));
}

template <bool TA, bool TB>
int launch_staged(const GemmArgs& g0, int64_t batch, int bm, int bn, int bk, hipStream_t s,
                  const Workspace& wsp, bool unsplit = false) {
    GemmArgs g = g0;
    const int most = unsplit ? 1 : class_splits(g.m, g.n, g.k, batch, bm, bn, bk);
    StagedPlan plan = plan_staged(g.m, g.n, g.k, batch, most);
    // Causal products skip by row bands of the tile, so they take the class's rows; the splits
    // are those of the product without skipping, and so are the bits. The products whose tiles
    // above the diagonal are left out write little but C: 64 columns at a time (256 heads of
    // 512 x 512 x 64: 68 -> 64 us).
    if (g.causal != 0) plan.shape = bm == 64 ? 3 : bn == 64 || g.causal == 1 || g.causal == 4 ? 2 : 1;
    const int shape = plan.shape;
    g.k_chunk = ceil_div(ceil_div(g.k, plan.splits), kSplitBK) * kSplitBK;
    const int splits = int(ceil_div(g.k, g.k_chunk));
    g.splits = splits;
    // Unstored tiles would leave their split-K partials unwritten for the
    // reduction to read: split products store them as mode 1 does.
    if (splits > 1 && g.causal == 4) g.causal = 1;
    float* out = g.c;
    g.ws_stride = batch * g.m * g.n + (g.colsum ? g.n : 0);
    // The no-allocation entry point admits what its array holds of the class's plan.
    const size_t split_bytes = size_t(g.ws_stride) * sizeof(float);
    if (wsp.base != nullptr && most > 1 && most * split_bytes > wsp.cap_bytes)
        return fail(EHIP_EINVAL,
                    "gemm (no allocation): %d K-splits of %lld x %lld need %zu bytes of "
                    "workspace, more than the fixed %zu",
                    most, (long long)g.m, (long long)g.n, most * split_bytes, wsp.cap_bytes);
    if (splits > 1) {
        g.c = wsp.base != nullptr ? wsp.base : static_cast<float*>(scratch(splits * split_bytes));
        if (g.c == nullptr) return EHIP_ENOMEM;
    }
    g.tiles_m = int(ceil_div(g.m, kShapes[shape].bm));
    g.tiles_n = int(ceil_div(g.n, kShapes[shape].bn));
    const int64_t tiles = int64_t(g.tiles_m) * g.tiles_n;
    // Split K only below ~512 workgroups, so a split product is one launch;
    // longer batches run in ranges of the grid's z extent.
    for (int64_t z0 = 0; z0 < batch; z0 += kGridZ) {
        g.batch0 = z0;
        const dim3 grid{unsigned(tiles), unsigned(splits),
                        unsigned(batch - z0 < kGridZ ? batch - z0 : kGridZ)};
        const int rc = shape == 0   ? launch_shape<256, 128, 64, 64, 2, 2, TA, TB>(g, grid, s)
                       : shape == 1 ? launch_shape<128, 128, 64, 32, 1, 4, TA, TB>(g, grid, s)
                       : shape == 2 ? launch_shape<128, 64, 64, 32, 1, 3, TA, TB>(g, grid, s)
                                    : launch_shape<64, 64, 32, 32, 2, 3, TA, TB>(g, grid, s);
        if (rc) return rc;
    }
    if (splits > 1) {
        GemmArgs gr = g0;  // the caller's output and epilogue, the workspace geometry
        gr.ws_stride = g.ws_stride;
        return splitk_finish(g.c, out, gr, batch, splits, s);
    }
    return EHIP_OK;
}

double padding(int64_t m, int64_t n, int bm, int bn) {
    return double(ceil_div(m, bm) * bm) * double(ceil_div(n, bn) * bn) / (double(m) * double(n)) - 1.0;
}

// 32 x 32 tiles with K sliced over the workgroup's waves (gemm_kslice): one
// launch, no workspace. W, the waves per workgroup, doubles while the grid
// stays within 2048 waves (8 per CU) and each wave keeps at least 32 k.
template <int W, bool TA, bool TB>
int launch_kslice_w(GemmArgs g, int64_t batch, bool whole, hipStream_t s) {
    const bool epi = !plain_epilogue(g);
    for (int64_t z0 = 0; z0 < batch; z0 += kGridZ) {
        g.batch0 = z0;
        const dim3 grid{unsigned(int64_t(g.tiles_m) * g.tiles_n), 1u,
                        unsigned(batch - z0 < kGridZ ? batch - z0 : kGridZ)};
        if (whole && !epi)
            EHIP_LAUNCH("gemm", (gemm_kslice<W, TA, TB, false, false>), grid, dim3(64 * W), 0, s,
                        g);
        else if (whole)
            EHIP_LAUNCH("gemm", (gemm_kslice<W, TA, TB, false, true>), grid, dim3(64 * W), 0, s, g);
        else if (!epi)
            EHIP_LAUNCH("gemm", (gemm_kslice<W, TA, TB, true, false>), grid, dim3(64 * W), 0, s, g);
        else
            EHIP_LAUNCH("gemm", (gemm_kslice<W, TA, TB, true, true>), grid, dim3(64 * W), 0, s, g);
    }
    return EHIP_OK;
}

// The waves per workgroup of the K-sliced tiles: W doubles while the grid
// stays within 2048 waves (8 per CU) and each wave keeps at least 64 k. More
// waves also shorten each wave's serial accumulation chain: with at most 4
// per CU (about 5 % faster on 512^3) the char-Transformer's 10-step loss
// trajectory drifts past 1e-5 of the reference's at step 9; with 8 it stays
// within 4e-6.
int kslice_waves(int64_t tiles, int64_t k) {
    int w = 1;
    while (w < 8 && tiles * 2 * w <= 2048 && k >= 64 * w) w *= 2;
    return w;
}

void kslice_geometry(GemmArgs& g, int w) {
    g.tiles_m = int(ceil_div(g.m, 32));
    g.tiles_n = int(ceil_div(g.n, 32));
    g.k_chunk = ceil_div(ceil_div(g.k, w), 32) * 32;
    g.splits = 1;
}

bool kslice_whole(const GemmArgs& g) {
    return g.vec && g.m % 32 == 0 && g.n % 32 == 0 && g.k % 32 == 0;
}

template <bool TA, bool TB>
int launch_kslice(GemmArgs g, int64_t batch, hipStream_t s) {
    const int w = kslice_waves(ceil_div(g.m, 32) * ceil_div(g.n, 32) * batch, g.k);
    kslice_geometry(g, w);
    const bool whole = kslice_whole(g);
    switch (w) {
        case 1: return launch_kslice_w<1, TA, TB>(g, batch, whole, s);
        case 2: return launch_kslice_w<2, TA, TB>(g, batch, whole, s);
        case 4: return launch_kslice_w<4, TA, TB>(g, batch, whole, s);
        default: return launch_kslice_w<8, TA, TB>(g, batch, whole, s);
    }
}

// Tile classes, largest first:
//   L, M, S, T  staged tiles, whose K split is planned on 256 x 256, 128 x 128, 128 x 64 and
//      64 x 64 tiles; launch_staged then picks the shape that runs
//   K  32 x 32 per workgroup, K sliced over its waves: outputs too small for
//      the larger tiles to fill the chip (512^3, the char-Transformer's layers)
//   U  products of K's sizes that staged tiles do faster, K unsplit: like K's they
//      use no workspace, which overlapping calls on several streams would share
//   P  16 x 16 per workgroup of kPanelWaves waves, each a part of K: A^T B products of few
//      tiles over a long K (weight gradients of narrow layers), one load round trip per 128 k
//      of a wave, no workspace
// A tile size is taken when its grid fills the 256 CUs (with split-K where K
// is long) and the padding it adds to the output stays small.
enum class Tile { L, M, S, K, T, U, P };

// ------------------------------------------------------------ panel products
//
// C (m x n, few 16 x 16 tiles) = A^T B over a long K, A stored K x M and B
// K x N (a weight gradient X^T dY). One workgroup of kPanelWaves waves per
// output tile; wave w takes k in [w kw, (w + 1) kw) and issues the loads of
// kPanelSteps MFMA steps (4 k each) at once: lane l reads A(k0 + l / 16,
// m0 + l % 16) and B(k0 + l / 16, n0 + l % 16), sixteen consecutive floats
// of a row per lane group, which are exactly the operands of
// v_mfma_f32_16x16x4f32 (A: i = lane % 16, k = lane / 16; B: j = lane % 16,
// k = lane / 16; D: j = lane % 16, i = 4 (lane / 16) + register). The waves'
// tiles are then added in wave order through LDS, and the epilogue applied.
// With a column sum (the bias gradient), each lane adds its B values in k
// order, and the tile row 0 workgroups add lanes and waves in a fixed order.
// The K-sliced 32 x 32 tiles pull the panels of 32 rows and columns through
// as few CUs; the 16 x 16 tiles spread them over four times as many.
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kPanelWaves = 4;
constexpr int kPanelSteps = 32;

// One output tile of a panel product (the workgroup's whole work).
template <bool CHECK, bool EPI>
__device__ __forceinline__ void panel_tile(const GemmArgs& g, int tile) {
    // The checked form takes half the steps per round trip: its rows are often
    // unaligned (a 121-float row's 64-byte segments straddle cache lines), and
    // more loads in flight then only add line traffic (17.0 against 14.2 us).
    constexpr int kSteps = CHECK ? kPanelSteps / 2 : kPanelSteps;
    __shared__ float red[kPanelWaves][256];
    __shared__ float cred[kPanelWaves][64];
    const int64_t m0 = int64_t(tile / g.tiles_n) * 16, n0 = int64_t(tile % g.tiles_n) * 16;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / 64);
    const int lane = int(threadIdx.x) % 64;
    const int li = lane % 16, lk = lane / 16;
    const int64_t kb = int64_t(wave) * g.k_chunk;
    const int64_t ke = kb + g.k_chunk < g.k ? kb + g.k_chunk : g.k;
    const bool col_sums = g.colsum != nullptr && m0 == 0;
    const bool row_in = !CHECK || m0 + li < g.m, col_in = !CHECK || n0 + li < g.n;
    // Lane offsets within a step's four rows; the rows' bases are uniform.
    const int32_t offa = int32_t(lk * g.lda + m0 + li), offb = int32_t(lk * g.ldb + n0 + li);
    floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    float cs = 0.0f;
    for (int64_t k0 = kb; k0 < ke; k0 += 4 * kSteps) {
        float a[kSteps], b[kSteps];
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            const float* ra = g.a + (k0 + 4 * u) * g.lda;
            const float* rb = g.b + (k0 + 4 * u) * g.ldb;
            if (CHECK) {
                const bool kin = k0 + 4 * u + lk < ke;
                a[u] = kin && row_in ? ra[offa] : 0.0f;
                b[u] = kin && col_in ? rb[offb] : 0.0f;
            } else {
                a[u] = ra[offa];
                b[u] = rb[offb];
            }
        }
        // Every load of the chunk issued before the first wait.
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kSteps; ++u)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b[u], acc, 0, 0, 0);
        if (col_sums) {
#pragma unroll
            for (int u = 0; u < kSteps; ++u) cs = cs + b[u];
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][(4 * lk + r) * 16 + li] = acc[r];
    cred[wave][lane] = cs;
    __syncthreads();
    for (int o = int(threadIdx.x); o < 256; o += 64 * kPanelWaves) {
        const int i = o / 16, j = o % 16;
        float v = red[0][o];
#pragma unroll
        for (int w = 1; w < kPanelWaves; ++w) v = v + red[w][o];
        const int64_t row = m0 + i, col = n0 + j;
        if (!CHECK || (row < g.m && col < g.n)) {
            float* dst = g.c + row * g.ldc + col;
            *dst = EPI ? epilogue(g, 0, row, col, v, dst) : v;
        }
    }
    if (col_sums && threadIdx.x < 16) {
        const int j = int(threadIdx.x);
        float v = 0.0f;
        for (int w = 0; w < kPanelWaves; ++w)
#pragma unroll
            for (int q = 0; q < 4; ++q) v = v + cred[w][16 * q + j];
        if (n0 + j < g.n) g.colsum[n0 + j] = v;
    }
}

template <bool CHECK, bool EPI>
__global__ __launch_bounds__(64 * kPanelWaves) void gemm_tn_panel(GemmArgs g) {
    panel_tile<CHECK, EPI>(g, int(blockIdx.x));
}

// Independent panel products in one launch (ehip_gemm_batch_f32): workgroups
// first[j] .. first[j + 1] - 1 are product j's tiles, each formed exactly as
// its own launch would, in the form (mode[j]: bit 0 checked tiles, bit 1 the
// epilogue) its own launch takes; the branch is uniform per workgroup.
constexpr int kPanelGroupMax = 12;
struct PanelGroup {
    GemmArgs g[kPanelGroupMax];
    int first[kPanelGroupMax + 1];
    int mode[kPanelGroupMax];
    int count;
};
static_assert(sizeof(PanelGroup) <= 4096, "kernel arguments of at most 4 KB");

__global__ __launch_bounds__(64 * kPanelWaves) void gemm_tn_panel_group(PanelGroup p) {
    const int b = int(blockIdx.x);
    int j = 0;
    while (j + 1 < p.count && b >= p.first[j + 1]) ++j;
    j = __builtin_amdgcn_readfirstlane(j);
    const int tile = b - p.first[j];
    switch (__builtin_amdgcn_readfirstlane(p.mode[j])) {
        case 0: panel_tile<false, false>(p.g[j], tile); break;
        case 1: panel_tile<true, false>(p.g[j], tile); break;
        case 2: panel_tile<false, true>(p.g[j], tile); break;
        default: panel_tile<true, true>(p.g[j], tile); break;
    }
}

// Independent K-sliced products A B (neither operand transposed) of one
// kernel form in one launch (ehip_gemm_batch_f32; the projections of one
// input, e.g. attention's query, key and value): workgroups first[j] ..
// first[j + 1] - 1 are product j's tiles, each formed with the K slicing its
// own launch would use.
template <int W, bool CHECK, bool EPI>
__global__ __launch_bounds__(64 * W) void gemm_kslice_group(PanelGroup p) {
    __shared__ __attribute__((aligned(16))) float lds[KsliceLds<W>::kFloats];
    const int b = int(blockIdx.x);
    int j = 0;
    while (j + 1 < p.count && b >= p.first[j + 1]) ++j;
    j = __builtin_amdgcn_readfirstlane(j);
    kslice_tile<W, false, false, CHECK, EPI, 4>(p.g[j], b - p.first[j], 0, lds, W);
}

// The panel product's k per wave: whole chunks of 4 kPanelSteps k (the
// unchecked kernel loads them without guards), else a multiple of 4.
int64_t panel_wave_k(int64_t k, bool whole) {
    const int64_t q = whole ? 4 * kPanelSteps : 4;
    return ceil_div(ceil_div(k, kPanelWaves), q) * q;
}

bool operands_aligned(const GemmArgs& g) {
    return aligned16(g.a) && aligned16(g.b) && g.lda % 4 == 0 && g.ldb % 4 == 0 &&
           g.stride_a % 4 == 0 && g.stride_b % 4 == 0 &&
           (g.inner == 1 || (g.stride_a2 % 4 == 0 && g.stride_b2 % 4 == 0));
}

// Per operand: bit 0 when A's rows are 16-byte aligned, bit 1 for B's.
int operand_alignment(const GemmArgs& g) {
    const bool a = aligned16(g.a) && g.lda % 4 == 0 && g.stride_a % 4 == 0 &&
                   (g.inner == 1 || g.stride_a2 % 4 == 0);
    const bool b = aligned16(g.b) && g.ldb % 4 == 0 && g.stride_b % 4 == 0 &&
                   (g.inner == 1 || g.stride_b2 % 4 == 0);
    return (a ? 1 : 0) | (b ? 2 : 0);
}

// Whether 32 x 32 tiles with K sliced over the waves beat staged tiles of unsplit K on an
// output too small for 512 of the latter (MI355X, us, sliced : staged). In whole tiles of 32, up
// to about 1.2e9 multiply-adds (512^3 5.8 : 10.5, 768^3 17.0 : 17.7, 3392 x 192 x 1984 42.6 :
// 32.4). With edges, by how the sliced tiles fill the chip:
//   - to one per CU they win at every K beyond two staged steps (A B 3337 x 21 x 3303 62 : 73,
//     A^T B 700 x 300 x 801 14 : 22, A^T B^T 8000 x 21 x 530 12 : 18), except A B^T from
//     unaligned rows, whose loads are by element along both k: there only up to 256 k (8000 x 21
//     x 250 9.5 : 10.0, x 801 22.6 : 21.6) and on few tiles (2100 x 21 x 2031 45 : 48);
//   - to 448 tiles, A^T B (rows of both operands contiguous: 11000 x 31 x 1021 25 : 28.5, but x
//     97 8.2 : 7.2) and, of aligned rows, A^T B^T (800 x 516 x 152 8.0 : 8.7) and the others
//     at short K (A B 552 x 472 x 152 7.2 : 8.6, x 1012 25.9 : 26.1);
//   - to 512, two per CU, A^T B of long K (3825 x 104 x 1651 38.3 : 43.5, 668 x 757 x 484 15.3 :
//     16.5; 179 x 2523 x 436 15.4 : 14.8, and beyond 512 a third round, 172 x 2852 x 1090 0.67 of
//     the sliced time);
//   - beyond, none (900 x 700 x 2031: A B 98 : 49, A B^T 142 : 48), but for batches of matrices of
//     up to 32 rows over one staged step: half of every 64 x 64 tile is empty there, or five
//     eighths of columns that end in the first half of a tile, and from 768 tiles (three per CU,
//     one round), or 512, the sliced ones do less (400 x (31 x 72 x 31) 8.2 : 9.8, 390 x
//     (14 x 120 x 14) 7.9 : 9.3, 305 x (19 x 96 x 19) 6.8 : 7.5; 329 x (14 x 127 x 14) 7.8 : 7.1);
//     and for batches of more than 512 results of A B^T of up to 24 x 24 (672 x (14 x 14 x 72)
//     7.8 : 9.2, 611 x (23 x 23 x 88) 8.5 : 9.5; 560 x (26 x 26 x 96) 8.9 : 8.4).
// The two sum in different orders, so the rule goes by the shape alone ("aligned rows": those of
// operands stored without gaps), not by addresses or leading dimensions: a product's bits do not
// depend on where its operands lie. Causal products keep the bits of the full product either way.
// From 2^24 tiles of 64 x 64 (2^30 rows), whose 2^32 threads are more than a launch takes, the
// sliced ones' single wave per tile still fits.
bool kslice_wins(const GemmArgs& g, int64_t batch, bool ta, bool tb) {
    if (ceil_div(g.m, 64) * ceil_div(g.n, 64) >= int64_t(1) << 24) return true;
    const bool rows = (ta ? g.m : g.k) % 4 == 0 && (tb ? g.k : g.n) % 4 == 0;
    if (g.m % 32 == 0 && g.n % 32 == 0 && g.k % 32 == 0)
        return double(g.m) * double(g.n) * double(g.k) * double(batch) < 1.2e9;
    const int64_t tiles = ceil_div(g.m, 32) * ceil_div(g.n, 32) * batch;
    if (tiles > 448) {
        const int64_t staged = ceil_div(g.m, 64) * ceil_div(g.n, 64) * batch;
        if (g.m <= 32 && g.k <= 32) return staged > (8 * tiles <= 12 * staged ? 512 : 768);
        if (!ta && tb && g.m <= 24 && g.n <= 24) return tiles > 512;
        return ta && !tb && batch == 1 && tiles <= 512 && g.k > 480;
    }
    if (!ta && rows) return tiles <= 256 || g.k <= (tb ? 256 : 512);
    if (!ta && tb) return tiles < 100 ? g.k > 64 : tiles <= 256 && g.k > 96 && g.k <= 256;
    if (tiles <= 256 || (ta && tb && rows)) return g.k > 64;
    return ta && !tb && g.k > 160;
}

Tile plan_tile(const GemmArgs& g, int64_t batch, bool ta, bool tb) {
    const int64_t tl = ceil_div(g.m, 256) * ceil_div(g.n, 256) * batch;
    const int64_t tm = ceil_div(g.m, 128) * ceil_div(g.n, 128) * batch;
    const int64_t ts = ceil_div(g.m, 128) * ceil_div(g.n, 64) * batch;
    const bool long_k = g.k >= 2048;
    if (tl >= 256 && padding(g.m, g.n, 256, 256) < 0.15 && g.k >= 256) return Tile::L;
    if ((tm >= 128 || (tm >= 32 && long_k)) && padding(g.m, g.n, 128, 128) < 0.25) return Tile::M;
    // Causal skipping from below (mode 3, the attention backward's dV = W^T dO
    // and dK = dS^T Q) skips more in 64-row bands: the 64 x 64 tile there
    // (measured on MI355X in cfg5's step, 256 heads of 512 x 64 x 512: 60.5 ->
    // 51.3 us; for mode 2 it measured slower in the step, 58.4 -> 61.0 us, and
    // without skipping the 128 x 64 tile is 3 % ahead). Only where neither tile
    // splits K (at least 512 of the 128 x 64 tiles), so that the skipping
    // product keeps the bits of the same product without it.
    if ((ts >= 128 || (ts >= 32 && long_k)) && padding(g.m, g.n, 128, 64) < 0.25)
        return g.causal == 3 && ts >= 512 ? Tile::T : Tile::S;
    // Weight gradients of narrow layers: few output tiles, long K.
    if (ta && !tb && batch == 1 && g.causal == 0 && g.k >= 1024 &&
        ceil_div(g.m, 16) * ceil_div(g.n, 16) <= 1024)
        return Tile::P;
    // A B column sum is computed only by the staged tiles: with one, K's sizes are T's, and U's,
    // whose unsplit tiles form it as well, stay U's.
    if (ceil_div(g.m, 32) * ceil_div(g.n, 32) * batch >= 64) {
        if (!kslice_wins(g, batch, ta, tb)) return Tile::U;
        if (g.colsum == nullptr) return Tile::K;
    }
    return Tile::T;
}

// A panel product's tile grid and k per wave; returns true for the unchecked
// (whole) form.
bool panel_geometry(GemmArgs& g) {
    g.tiles_m = int(ceil_div(g.m, 16));
    g.tiles_n = int(ceil_div(g.n, 16));
    const bool whole = g.m % 16 == 0 && g.n % 16 == 0 && g.k % (4 * kPanelSteps) == 0 &&
                       g.lda * g.k < (int64_t(1) << 31) && g.ldb * g.k < (int64_t(1) << 31);
    g.k_chunk = panel_wave_k(g.k, whole);
    g.splits = 1;
    return whole;
}

int launch_panel(GemmArgs g, hipStream_t s) {
    const bool whole = panel_geometry(g);
    const unsigned tiles = unsigned(int64_t(g.tiles_m) * g.tiles_n);
    const bool epi = !plain_epilogue(g);
    const dim3 block(64 * kPanelWaves);
    if (whole && !epi)
        EHIP_LAUNCH("gemm", (gemm_tn_panel<false, false>), dim3(tiles), block, 0, s, g);
    else if (whole)
        EHIP_LAUNCH("gemm", (gemm_tn_panel<false, true>), dim3(tiles), block, 0, s, g);
    else if (!epi)
        EHIP_LAUNCH("gemm", (gemm_tn_panel<true, false>), dim3(tiles), block, 0, s, g);
    else
        EHIP_LAUNCH("gemm", (gemm_tn_panel<true, true>), dim3(tiles), block, 0, s, g);
    return EHIP_OK;
}

template <bool TA, bool TB>
int gemm_modes(GemmArgs g, int64_t batch, hipStream_t s, const Workspace& wsp) {
    // The unchecked kernels need whole tiles and 16-byte aligned float4 rows;
    // the checked ones still load whole float4s away from the edges when the
    // rows are aligned.
    g.vec = operands_aligned(g) ? 1 : 0;
    g.vec_ab = operand_alignment(g);
    switch (plan_tile(g, batch, TA, TB)) {
        case Tile::L: return launch_staged<TA, TB>(g, batch, 256, 256, 16, s, wsp);
        case Tile::M: return launch_staged<TA, TB>(g, batch, 128, 128, 32, s, wsp);
        case Tile::S: return launch_staged<TA, TB>(g, batch, 128, 64, 32, s, wsp);
        case Tile::K: return launch_kslice<TA, TB>(g, batch, s);
        case Tile::P: return launch_panel(g, s);
        case Tile::U: return launch_staged<TA, TB>(g, batch, 64, 64, 16, s, wsp, true);
        default: return launch_staged<TA, TB>(g, batch, 64, 64, 16, s, wsp);
    }
}

// The backward's two products in one launch when both take the K-sliced tiles
// (g0: dA = dC B^T, g1: dB = A^T dC; plain batch-1 products); returns false
// when they do not, and the caller runs them one by one.
bool try_kslice_pair(GemmArgs g0, GemmArgs g1, hipStream_t s, int* rc) {
    g0.vec = operands_aligned(g0) ? 1 : 0;
    g1.vec = operands_aligned(g1) ? 1 : 0;
    g0.vec_ab = operand_alignment(g0);
    g1.vec_ab = operand_alignment(g1);
    if (plan_tile(g0, 1, false, true) != Tile::K || plan_tile(g1, 1, true, false) != Tile::K)
        return false;
    // Each product is sliced as its own launch would slice it (same bits).
    const int64_t t0 = ceil_div(g0.m, 32) * ceil_div(g0.n, 32);
    const int64_t t1 = ceil_div(g1.m, 32) * ceil_div(g1.n, 32);
    const int w0 = kslice_waves(t0, g0.k), w1 = kslice_waves(t1, g1.k);
    const int w = w0 > w1 ? w0 : w1;
    kslice_geometry(g0, w0);
    kslice_geometry(g1, w1);
    const int64_t tiles = t0 + t1;
    const bool check = !kslice_whole(g0) || !kslice_whole(g1);
    const bool epi = !plain_epilogue(g0) || !plain_epilogue(g1);
    const dim3 grid{unsigned(tiles)};
#define EHIP_PAIR(W)                                                                               \
    do {                                                                                           \
        if (check && epi)                                                                          \
            EHIP_LAUNCH("gemm_pair", (gemm_kslice_pair<W, true, true>), grid, dim3(64 * W), 0, s,   \
                        g0, g1, w0, w1);                                                           \
        else if (check)                                                                            \
            EHIP_LAUNCH("gemm_pair", (gemm_kslice_pair<W, true, false>), grid, dim3(64 * W), 0, s,  \
                        g0, g1, w0, w1);                                                           \
        else if (epi)                                                                              \
            EHIP_LAUNCH("gemm_pair", (gemm_kslice_pair<W, false, true>), grid, dim3(64 * W), 0, s,  \
                        g0, g1, w0, w1);                                                           \
        else                                                                                       \
            EHIP_LAUNCH("gemm_pair", (gemm_kslice_pair<W, false, false>), grid, dim3(64 * W), 0,    \
                        s, g0, g1, w0, w1);                                                        \
        return EHIP_OK;                                                                            \
    } while (0)
    const auto launch = [&]() -> int {
        switch (w) {
            case 1: EHIP_PAIR(1);
            case 2: EHIP_PAIR(2);
            case 4: EHIP_PAIR(4);
            default: EHIP_PAIR(8);
        }
    };
#undef EHIP_PAIR
    *rc = launch();
    return true;
}

// ------------------------------------------------------------ small products
//
// Products too small to fill the chip with MFMA tiles are latency-bound: a
// 64 x 784 x 10 layer is one 64 x 64 tile, split six ways along K, and spends
// its time in load round trips rather than matrix math. Two vector kernels
// take them instead:
//   thread per output (K <= 128): the K products summed in k order from zero,
//     zero A elements skipped -- the reference's i-k-j loop
//     (src/tensor_ops.cpp:553-560) term for term, so the result is
//     bit-identical to the CPU's;
//   wave per output (few outputs, long K): lane l sums k = l, l + 64, ... and
//     the lanes are combined by a fixed butterfly: deterministic, within the
//     K-term tolerance.
// Both finish with the MFMA kernel's epilogue (alpha, addend, beta).

// Measured on MI355X: the vector kernels win while the whole product is about
// a million multiply-adds or less (cfg2's 64 x 784 x 10 layer: 4 + 6 + 4 us
// against 16 + 11 + 5 for the MFMA tiles); larger ones go to MFMA, and K
// beyond 2048 to split-K MFMA, which spreads one output over many CUs.
constexpr int64_t kSmallThreadK = 128;
constexpr int64_t kSmallThreadWork = int64_t(1) << 21;  // outputs * K
constexpr int64_t kSmallWaveOutputs = 16384;
constexpr int64_t kSmallWaveMaxK = 2048;
constexpr int64_t kSmallWaveWork = int64_t(1) << 21;

// Outputs first, first + step, ... of a thread-per-output product.
template <bool TA, bool TB>
__device__ __forceinline__ void small_thread_outputs(const GemmArgs& g, unsigned total,
                                                     unsigned first, unsigned step) {
    const unsigned n = unsigned(g.n), m = unsigned(g.m);
    for (unsigned o = first; o < total; o += step) {
        const unsigned t = o / n, j = o - t * n;
        const unsigned bi = t / m, i = t - bi * m;
        const float* a = g.a + batch_offset(bi, g.inner, g.stride_a, g.stride_a2) +
                         (TA ? int64_t(i) : int64_t(i) * g.lda);
        const float* b = g.b + batch_offset(bi, g.inner, g.stride_b, g.stride_b2) +
                         (TB ? int64_t(j) * g.ldb : int64_t(j));
        const int64_t ak = TA ? g.lda : 1, bk = TB ? 1 : g.ldb;
        float acc = 0.0f;
        int64_t k = 0;
        // Sixteen terms' loads in flight at a time (the sums stay in k order):
        // a thread's chain of dependent load round trips is K / 16 long.
        for (; k + 16 <= g.k; k += 16) {
            float av[16], bv[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                av[u] = a[(k + u) * ak];
                bv[u] = b[(k + u) * bk];
            }
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const float s = acc + av[u] * bv[u];
                acc = av[u] != 0.0f ? s : acc;
            }
        }
        for (; k + 4 <= g.k; k += 4) {
            float av[4], bv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                av[u] = a[(k + u) * ak];
                bv[u] = b[(k + u) * bk];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float s = acc + av[u] * bv[u];
                acc = av[u] != 0.0f ? s : acc;
            }
        }
        for (; k < g.k; ++k) {
            const float av = a[k * ak];
            const float s = acc + av * b[k * bk];
            acc = av != 0.0f ? s : acc;
        }
        float* dst = g.c + batch_offset(bi, g.inner, g.stride_c, g.stride_c2) + int64_t(i) * g.ldc + j;
        *dst = epilogue(g, bi, i, j, acc, dst);
    }
}

template <bool TA, bool TB>
__global__ __launch_bounds__(256) void gemm_small_thread(GemmArgs g, unsigned total) {
    small_thread_outputs<TA, TB>(g, total, blockIdx.x * 256u + threadIdx.x, gridDim.x * 256u);
}

// The three gradients of a small Linear layer in one launch: blocks
// [0, bdx) compute dx = dy w^T and [bdx, bdx + bdw) dw = x^T dy as
// gemm_small_thread does, the rest db[c] = sum over rows of dy[r][c] in row
// order from zero as sum_axis_serial does -- the separate launches' results
// bit for bit, in about the time of the longest.
__global__ __launch_bounds__(256) void linear_backward_small(GemmArgs gdx, unsigned ndx,
                                                             unsigned bdx, GemmArgs gdw,
                                                             unsigned ndw, unsigned bdw,
                                                             const float* __restrict__ dy,
                                                             float* __restrict__ db, int rows,
                                                             int cols) {
    const unsigned b = blockIdx.x;
    if (b < bdx) {
        small_thread_outputs<false, true>(gdx, ndx, b * 256u + threadIdx.x, bdx * 256u);
    } else if (b < bdx + bdw) {
        small_thread_outputs<true, false>(gdw, ndw, (b - bdx) * 256u + threadIdx.x, bdw * 256u);
    } else {
        const int c = int(b - bdx - bdw) * 256 + int(threadIdx.x);
        if (c >= cols) return;
        float acc = 0.0f;
        int r = 0;
        for (; r + 8 <= rows; r += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = dy[int64_t(r + u) * cols + c];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc += v[u];
        }
        for (; r < rows; ++r) acc += dy[int64_t(r) * cols + c];
        db[c] = acc;
    }
}

template <bool TA, bool TB>
__global__ __launch_bounds__(256) void gemm_small_wave(GemmArgs g, unsigned total) {
    const unsigned lane = threadIdx.x % 64u;
    const unsigned o = blockIdx.x * 4u + threadIdx.x / 64u;
    if (o >= total) return;  // whole waves leave together
    const unsigned n = unsigned(g.n), m = unsigned(g.m);
    const unsigned t = o / n, j = o - t * n;
    const unsigned bi = t / m, i = t - bi * m;
    const float* a = g.a + batch_offset(bi, g.inner, g.stride_a, g.stride_a2) +
                     (TA ? int64_t(i) : int64_t(i) * g.lda);
    const float* b = g.b + batch_offset(bi, g.inner, g.stride_b, g.stride_b2) +
                     (TB ? int64_t(j) * g.ldb : int64_t(j));
    const int64_t ak = TA ? g.lda : 1, bk = TB ? 1 : g.ldb;
    float acc = 0.0f;
    int64_t k = lane;
    for (; k + 192 < g.k; k += 256) {
        float av[4], bv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            av[u] = a[(k + 64 * u) * ak];
            bv[u] = b[(k + 64 * u) * bk];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) acc += av[u] * bv[u];
    }
    for (; k < g.k; k += 64) acc += a[k * ak] * b[k * bk];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) {
        float* dst = g.c + batch_offset(bi, g.inner, g.stride_c, g.stride_c2) + int64_t(i) * g.ldc + j;
        *dst = epilogue(g, bi, i, j, acc, dst);
    }
}

template <bool TA, bool TB>
int gemm_small(const GemmArgs& g, int64_t batch, bool wave, hipStream_t s) {
    const int64_t total = batch * g.m * g.n;
    if (wave) {
        EHIP_LAUNCH("gemm_small", (gemm_small_wave<TA, TB>), dim3(unsigned(ceil_div(total, 4))),
                    dim3(256), 0, s, g, unsigned(total));
    } else {
        int64_t grid = ceil_div(total, 256);
        if (grid > 65536) grid = 65536;
        EHIP_LAUNCH("gemm_small", (gemm_small_thread<TA, TB>), dim3(unsigned(grid)), dim3(256), 0,
                    s, g, unsigned(total));
    }
    return EHIP_OK;
}

// Which small kernel, if any: 0 none, 1 thread per output, 2 wave per output.
int small_kind(int64_t batch, int64_t m, int64_t n, int64_t k) {
    const int64_t outputs = batch * m * n;
    if (outputs > 0xffffffffLL / 2) return 0;
    if (k <= kSmallThreadK && outputs * k <= kSmallThreadWork) return 1;
    if (outputs >= 64 && outputs <= kSmallWaveOutputs && k >= 256 && k <= kSmallWaveMaxK &&
        outputs * k <= kSmallWaveWork)
        return 2;
    return 0;
}

// Bias gradients of mid-sized Linear layers from the dW product's column sums
// (ehip_linear_backward_f32): where dy is at most 2^21 elements, the separate
// two-pass column sum is two launch-bound launches (the char-Transformer step:
// 1,597 -> 1,846 steps/s with them folded into the products), while for larger
// dy the staged column sums cost the product more than the separate pass
// (cfg5: 73.9 -> 74.5 ms per step). Up to 64 rows (or 16384+ columns) the
// serial sum of the small-layer launch keeps the reference's order. Only
// products of a class that is the same with and without the column sum
// qualify, so dw keeps the bits of the plain product: not K, which with one
// would be T.
std::atomic<bool> g_bias_from_dw{true};

bool bias_from_dw(int64_t rows, int64_t in, int64_t out) {
    if (!g_bias_from_dw.load() || rows <= 64 || out >= 16384 || rows * out > (int64_t(1) << 21))
        return false;
    if (small_kind(1, in, out, rows) != 0) return false;
    GemmArgs g{};
    g.m = in;
    g.n = out;
    g.k = rows;
    return plan_tile(g, 1, true, false) != Tile::K;
}

// ------------------------------------------------------------ timing probe
//
// ehip_gemm_probe_arm / _read: an event pair on the product's stream around
// every launch of an armed product shape (the tile kernel and its split-K
// reduction), for measuring chosen products inside a real workload.
struct GemmProbe {
    std::mutex mu;
    std::atomic<bool> armed{false};
    int trans_a = 0, trans_b = 0;
    std::vector<int64_t> shapes;  // m, n, k triples
    std::vector<hipEvent_t> events;  // start, end pairs
    size_t used = 0;
    double flop = 0.0;
};
GemmProbe g_probe;

int gemm_dispatch(const ehip_gemm_ex_t& d, hipStream_t s, const Workspace& wsp);

// Validation shared by both entry points, then the kernel choice (bracketed
// by the probe's events when the product is one it is armed for).
int gemm_run(const ehip_gemm_ex_t& d, hipStream_t s, const Workspace& wsp = Workspace{}) {
    if (!g_probe.armed.load(std::memory_order_relaxed)) return gemm_dispatch(d, s, wsp);
    hipEvent_t start = nullptr, end = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_probe.mu);
        bool match = d.batch == 1 && d.trans_a == g_probe.trans_a && d.trans_b == g_probe.trans_b &&
                     g_probe.used + 2 <= g_probe.events.size();
        bool shape = false;
        for (size_t i = 0; match && !shape && i + 3 <= g_probe.shapes.size(); i += 3)
            shape = g_probe.shapes[i] == d.m && g_probe.shapes[i + 1] == d.n &&
                    g_probe.shapes[i + 2] == d.k;
        if (match && shape) {
            start = g_probe.events[g_probe.used];
            end = g_probe.events[g_probe.used + 1];
            g_probe.used += 2;
            g_probe.flop += 2.0 * double(d.m) * double(d.n) * double(d.k);
        }
    }
    if (start == nullptr) return gemm_dispatch(d, s, wsp);
    if (hipEventRecord(start, s) != hipSuccess) return fail(EHIP_ELAUNCH, "gemm probe: event record");
    const int rc = gemm_dispatch(d, s, wsp);
    if (hipEventRecord(end, s) != hipSuccess) return fail(EHIP_ELAUNCH, "gemm probe: event record");
    return rc;
}

GemmArgs args_of(const ehip_gemm_ex_t& d) {
    GemmArgs g{};
    g.a = d.a;
    g.b = d.b;
    g.c = d.c;
    g.m = d.m;
    g.n = d.n;
    g.k = d.k;
    g.lda = d.lda;
    g.ldb = d.ldb;
    g.ldc = d.ldc;
    g.causal = d.causal;
    g.stride_a = d.stride_a;
    g.stride_b = d.stride_b;
    g.stride_c = d.stride_c;
    g.inner = d.inner;
    g.stride_a2 = d.stride_a_inner;
    g.stride_b2 = d.stride_b_inner;
    g.stride_c2 = d.stride_c_inner;
    g.alpha = d.alpha;
    g.add = d.addend;
    g.ld_add = d.ld_addend;
    g.stride_add = d.stride_addend;
    g.add_period = d.addend ? d.addend_period : 1;
    g.beta = d.beta;
    g.relu = d.relu;
    g.res = d.residual;
    g.ld_res = d.ld_residual;
    g.colsum = d.colsum_b;
    return g;
}

// True when gemm_dispatch would run the descriptor (already checked) as a
// panel product.
bool takes_panel(const ehip_gemm_ex_t& d) {
    if (d.batch != 1 || d.k == 0 || !d.trans_a || d.trans_b || d.m == 0 || d.n == 0 ||
        small_kind(1, d.m, d.n, d.k) != 0)
        return false;
    return plan_tile(args_of(d), 1, true, false) == Tile::P;
}

// True when gemm_dispatch would run the descriptor (already checked) as an
// unsplit K-sliced A B product that ehip_gemm_batch_f32 can group; g is then
// its launch arguments (geometry set) and form its kernel: waves index
// (0..3 for 1..8 waves) * 4 + checked tiles + 2 * epilogue.
bool takes_kslice_nn(const ehip_gemm_ex_t& d, GemmArgs& g, int& form) {
    if (d.batch != 1 || d.k == 0 || d.trans_a || d.trans_b || d.causal || d.colsum_b ||
        small_kind(1, d.m, d.n, d.k) != 0)
        return false;
    g = args_of(d);
    g.vec = operands_aligned(g) ? 1 : 0;
    g.vec_ab = operand_alignment(g);
    if (plan_tile(g, 1, false, false) != Tile::K) return false;
    const int w = kslice_waves(ceil_div(g.m, 32) * ceil_div(g.n, 32), g.k);
    kslice_geometry(g, w);
    form = (w == 1 ? 0 : w == 2 ? 1 : w == 4 ? 2 : 3) * 4 + (kslice_whole(g) ? 0 : 1) +
           (plain_epilogue(g) ? 0 : 2);
    return true;
}

template <int W>
int launch_kslice_group(const PanelGroup& p, int form, hipStream_t s) {
    const dim3 grid(unsigned(p.first[p.count])), block(64 * W);
    switch (form % 4) {
        case 0: EHIP_LAUNCH("gemm_batch", (gemm_kslice_group<W, false, false>), grid, block, 0, s, p); break;
        case 1: EHIP_LAUNCH("gemm_batch", (gemm_kslice_group<W, true, false>), grid, block, 0, s, p); break;
        case 2: EHIP_LAUNCH("gemm_batch", (gemm_kslice_group<W, false, true>), grid, block, 0, s, p); break;
        default: EHIP_LAUNCH("gemm_batch", (gemm_kslice_group<W, true, true>), grid, block, 0, s, p); break;
    }
    return EHIP_OK;
}

int gemm_dispatch(const ehip_gemm_ex_t& d, hipStream_t s, const Workspace& wsp) {
    GemmArgs g{};
    g.a = d.a;
    g.b = d.b;
    g.c = d.c;
    g.m = d.m;
    g.n = d.n;
    g.k = d.k;
    g.lda = d.lda;
    g.ldb = d.ldb;
    g.ldc = d.ldc;
    g.causal = d.causal;
    g.stride_a = d.stride_a;
    g.stride_b = d.stride_b;
    g.stride_c = d.stride_c;
    g.inner = d.inner;
    g.stride_a2 = d.stride_a_inner;
    g.stride_b2 = d.stride_b_inner;
    g.stride_c2 = d.stride_c_inner;
    g.alpha = d.alpha;
    g.add = d.addend;
    g.ld_add = d.ld_addend;
    g.stride_add = d.stride_addend;
    g.add_period = d.addend ? d.addend_period : 1;
    g.beta = d.beta;
    g.relu = d.relu;
    g.res = d.residual;
    g.ld_res = d.ld_residual;
    const int64_t batch = d.batch;
    const bool ta = d.trans_a != 0, tb = d.trans_b != 0;
    // K = 0 (only reached from the extended entry point): acc = 0, then the
    // epilogue, through the thread-per-output kernel.
    const int kind = d.k == 0 ? 1 : small_kind(batch, d.m, d.n, d.k);
    if (kind != 0 && d.colsum_b != nullptr) {
        // The vector kernels do not stage B: its column sums are a reduction
        // of their own (zero for K = 0).
        if (d.k == 0) {
            if (int rc = ehip_fill_f32(d.colsum_b, d.n, 0.0f, s)) return rc;
        } else if (int rc = column_sums(d.b, 1, d.k, d.n, d.ldb, 0, d.colsum_b, s)) {
            return rc;
        }
    } else {
        g.colsum = d.colsum_b;
    }
    if (kind != 0) {
        const bool wave = kind == 2;
        if (!ta && !tb) return gemm_small<false, false>(g, batch, wave, s);
        if (!ta && tb) return gemm_small<false, true>(g, batch, wave, s);
        if (ta && !tb) return gemm_small<true, false>(g, batch, wave, s);
        return gemm_small<true, true>(g, batch, wave, s);
    }
    if (!ta && !tb) return gemm_modes<false, false>(g, batch, s, wsp);
    if (!ta && tb) return gemm_modes<false, true>(g, batch, s, wsp);
    if (ta && !tb) return gemm_modes<true, false>(g, batch, s, wsp);
    return gemm_modes<true, true>(g, batch, s, wsp);
}

int check_desc(const ehip_gemm_ex_t& d) {
    if (d.batch < 0 || d.m < 0 || d.n < 0 || d.k < 0) return fail(EHIP_EINVAL, "gemm: negative extent");
    if (d.batch == 0 || d.m == 0 || d.n == 0) return EHIP_OK;
    if (!d.c) return fail(EHIP_EINVAL, "gemm: null C");
    if (d.k > 0 && (!d.a || !d.b)) return fail(EHIP_EINVAL, "gemm: null operand");
    if (d.lda < (d.trans_a ? d.m : d.k) || d.ldb < (d.trans_b ? d.k : d.n) || d.ldc < d.n)
        return fail(EHIP_EINVAL, "gemm: leading dimension too small");
    if (d.stride_a < 0 || d.stride_b < 0 || d.stride_c < 0 || d.stride_a_inner < 0 ||
        d.stride_b_inner < 0 || d.stride_c_inner < 0)
        return fail(EHIP_EINVAL, "gemm: negative batch stride");
    if (d.inner < 1) return fail(EHIP_EINVAL, "gemm: inner batch count %lld < 1", (long long)d.inner);
    if (d.addend && (d.ld_addend < 0 || d.stride_addend < 0 || d.addend_period < 1))
        return fail(EHIP_EINVAL, "gemm: bad addend geometry");
    if (d.colsum_b && (d.batch != 1 || d.trans_b))
        return fail(EHIP_EINVAL, "gemm: column sums need batch 1 and a K x N B");
    if (d.causal < 0 || d.causal > 4) return fail(EHIP_EINVAL, "gemm: causal mode %d", d.causal);
    if (d.residual && (d.batch != 1 || d.ld_residual < d.n))
        return fail(EHIP_EINVAL, "gemm: a residual needs batch 1 and ld_residual >= n");
    if (d.m > (int64_t(1) << 31) || d.n > (int64_t(1) << 31))
        return fail(EHIP_EINVAL, "gemm: extent beyond 2^31");
    return EHIP_OK;
}

const OccupancyKernel kGemmKernels[] = {
    {"gemm_kernel 256x128x32, 8 waves of 64x64 (NN)",
     reinterpret_cast<const void*>(&gemm_kernel<256, 128, 64, 64, 2, 2, false, false, false>), 512},
    {"gemm_kernel 256x128x32, 8 waves of 64x64 (TN: dW)",
     reinterpret_cast<const void*>(&gemm_kernel<256, 128, 64, 64, 2, 2, true, false, false>), 512},
    {"gemm_kernel 128x128x32, 8 waves of 64x32 (NT)",
     reinterpret_cast<const void*>(&gemm_kernel<128, 128, 64, 32, 1, 4, false, true, false>), 512},
    {"gemm_kernel 128x64x32, 4 waves of 64x32 (NN)",
     reinterpret_cast<const void*>(&gemm_kernel<128, 64, 64, 32, 1, 3, false, false, false>), 256},
    {"gemm_kernel 64x64x32, 4 waves of 32x32 (TN)",
     reinterpret_cast<const void*>(&gemm_kernel<64, 64, 32, 32, 2, 3, true, false, false>), 256},
    {"gemm_kslice 32x32, 8 waves (NN)",
     reinterpret_cast<const void*>(&gemm_kslice<8, false, false, false, false>), 512},
    {"gemm_tn_panel 16x16 (TN: narrow dW)",
     reinterpret_cast<const void*>(&gemm_tn_panel<false, false>), 64 * kPanelWaves},
    {"gemm_small_thread (NN)", reinterpret_cast<const void*>(&gemm_small_thread<false, false>), 256},
    {"gemm_splitk_reduce", reinterpret_cast<const void*>(&splitk_reduce), 256},
};
const OccupancyEntries kGemmKernelsReg(kGemmKernels);

}  // namespace
}  // namespace ehip

using namespace ehip;

namespace ehip_noalloc {

// The split-K workspace of ehip_gemm_f32_noalloc: a file-scope device array,
// so the entry point never allocates. Each GPU the library runs on holds its
// own copy until the process ends; its address on a device comes from
// hipGetSymbolAddress (the array's name in host code is only a stand-in).
constexpr size_t kScratchBytes = size_t(32) << 20;
static __device__ __align__(256) float scratch[kScratchBytes / sizeof(float)];

constexpr int kMaxDevices = 64;
std::mutex g_mu;
void* g_ptr[kMaxDevices] = {};  // the array's device address, per device

// The current device's copy of `scratch`, looked up once per device with that
// device current.
int workspace(ehip::Workspace* out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return ehip::fail(EHIP_ENODEV, "gemm (no allocation): hipGetDevice: %s",
                          hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices)
        return ehip::fail(EHIP_ENODEV, "gemm (no allocation): device %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_ptr[dev] == nullptr) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr)
            return ehip::fail(EHIP_ENODEV, "gemm (no allocation): hipGetSymbolAddress: %s",
                              hipGetErrorString(e));
        g_ptr[dev] = p;
    }
    out->base = static_cast<float*>(g_ptr[dev]);
    out->cap_bytes = kScratchBytes;
    return EHIP_OK;
}

}  // namespace ehip_noalloc

namespace ehip {
namespace {

int gemm_plain(int trans_a, int trans_b, int64_t batch, int64_t m, int64_t n, int64_t k,
               const float* a, int64_t lda, int64_t stride_a, const float* b, int64_t ldb,
               int64_t stride_b, float beta, float* c, int64_t ldc, int64_t stride_c,
               void* stream, const Workspace& wsp) {
    ehip_gemm_ex_t d{};
    d.trans_a = trans_a;
    d.trans_b = trans_b;
    d.batch = batch;
    d.inner = 1;
    d.m = m;
    d.n = n;
    d.k = k;
    d.a = a;
    d.lda = lda;
    d.stride_a = stride_a;
    d.b = b;
    d.ldb = ldb;
    d.stride_b = stride_b;
    d.c = c;
    d.ldc = ldc;
    d.stride_c = stride_c;
    d.alpha = 1.0f;
    d.beta = beta;
    if (int rc = check_desc(d)) return rc;
    if (batch == 0 || m == 0 || n == 0) return EHIP_OK;
    if (k == 0) {  // C = beta C
        if (beta == 0.0f) {
            for (int64_t bi = 0; bi < batch; ++bi)
                for (int64_t r = 0; r < m; ++r)
                    if (int rc = ehip_fill_f32(c + bi * stride_c + r * ldc, n, 0.0f, stream))
                        return rc;
        } else if (beta != 1.0f) {
            for (int64_t bi = 0; bi < batch; ++bi)
                for (int64_t r = 0; r < m; ++r)
                    if (int rc = ehip_scale_f32(c + bi * stride_c + r * ldc, n, beta, stream))
                        return rc;
        }
        return EHIP_OK;
    }
    return gemm_run(d, as_stream(stream), wsp);
}

}  // namespace
}  // namespace ehip

extern "C" {

int ehip_gemm_f32(int trans_a, int trans_b, int64_t batch, int64_t m, int64_t n, int64_t k,
                  const float* a, int64_t lda, int64_t stride_a, const float* b, int64_t ldb,
                  int64_t stride_b, float beta, float* c, int64_t ldc, int64_t stride_c,
                  void* stream) {
    EHIP_READY();
    return gemm_plain(trans_a, trans_b, batch, m, n, k, a, lda, stride_a, b, ldb, stride_b, beta,
                      c, ldc, stride_c, stream, Workspace{});
}

int ehip_gemm_f32_noalloc(int trans_a, int trans_b, int64_t batch, int64_t m, int64_t n,
                          int64_t k, const float* a, int64_t lda, int64_t stride_a,
                          const float* b, int64_t ldb, int64_t stride_b, float beta, float* c,
                          int64_t ldc, int64_t stride_c, void* stream) {
    EHIP_READY();
    Workspace wsp;
    if (int rc = ehip_noalloc::workspace(&wsp)) return rc;
    return gemm_plain(trans_a, trans_b, batch, m, n, k, a, lda, stride_a, b, ldb, stride_b, beta,
                      c, ldc, stride_c, stream, wsp);
}

int ehip_matmul_backward_f32(int64_t m, int64_t k, int64_t n, const float* a, int64_t lda,
                             const float* b, int64_t ldb, const float* dc, int64_t lddc, float* da,
                             int64_t ldda, float beta_a, float* db, int64_t lddb, float beta_b,
                             void* stream) {
    EHIP_READY();
    if (m < 0 || k < 0 || n < 0) return fail(EHIP_EINVAL, "matmul_backward: negative extent");
    if ((da && (!dc || !b)) || (db && (!dc || !a)))
        return fail(EHIP_EINVAL, "matmul_backward: null operand");
    if (da && db && m > 0 && k > 0 && n > 0 && lddc >= n && ldb >= n && lda >= k && ldda >= k &&
        lddb >= n) {
        // dA = dC B^T (m x k, K = n) and dB = A^T dC (k x n, K = m).
        const auto args = [](const float* x, int64_t ldx, const float* y, int64_t ldy, float* out,
                             int64_t ldo, int64_t rows, int64_t cols, int64_t kk, float beta) {
            GemmArgs g{};
            g.a = x;
            g.b = y;
            g.c = out;
            g.m = rows;
            g.n = cols;
            g.k = kk;
            g.lda = ldx;
            g.ldb = ldy;
            g.ldc = ldo;
            g.inner = 1;
            g.alpha = 1.0f;
            g.add_period = 1;
            g.beta = beta;
            return g;
        };
        int rc = EHIP_OK;
        if (small_kind(1, m, k, n) == 0 && small_kind(1, k, n, m) == 0 &&
            m <= 0x7fffffff && k <= 0x7fffffff && n <= 0x7fffffff &&
            try_kslice_pair(args(dc, lddc, b, ldb, da, ldda, m, k, n, beta_a),
                            args(a, lda, dc, lddc, db, lddb, k, n, m, beta_b), as_stream(stream),
                            &rc))
            return rc;
    }
    if (da)
        if (int rc = ehip_gemm_f32(0, 1, 1, m, k, n, dc, lddc, 0, b, ldb, 0, beta_a, da, ldda, 0,
                                   stream))
            return rc;
    if (db)
        if (int rc = ehip_gemm_f32(1, 0, 1, k, n, m, a, lda, 0, dc, lddc, 0, beta_b, db, lddb, 0,
                                   stream))
            return rc;
    return EHIP_OK;
}

int ehip_linear_backward_f32(const float* x, const float* w, const float* dy, float* dx,
                             float* dw, float* db, int64_t rows, int64_t in, int64_t out,
                             void* stream) {
    EHIP_READY();
    if (rows < 0 || in < 0 || out < 0) return fail(EHIP_EINVAL, "linear_backward: negative extent");
    if (!dy || (dx && !w) || (dw && !x)) return fail(EHIP_EINVAL, "linear_backward: null operand");
    // One launch when every requested part is a thread-per-output product or
    // a serial column sum (what the separate calls below would pick).
    const bool small = rows > 0 && in > 0 && out > 0 && rows <= 0x7fffffff &&
                       (!dx || small_kind(1, rows, in, out) == 1) &&
                       (!dw || small_kind(1, in, out, rows) == 1) &&
                       (!db || ((rows <= 64 || out >= 16384) && out <= 0x7fffffff));
    if (small) {
        const auto args = [](const float* a, int64_t lda, const float* b, int64_t ldb, float* c,
                             int64_t m, int64_t n, int64_t k) {
            GemmArgs g{};
            g.a = a;
            g.b = b;
            g.c = c;
            g.m = m;
            g.n = n;
            g.k = k;
            g.lda = lda;
            g.ldb = ldb;
            g.ldc = n;
            g.inner = 1;
            g.alpha = 1.0f;
            g.add_period = 1;
            return g;
        };
        const unsigned ndx = dx ? unsigned(rows * in) : 0u, ndw = dw ? unsigned(in * out) : 0u;
        const unsigned bdx = unsigned(ceil_div(ndx, 256)), bdw = unsigned(ceil_div(ndw, 256));
        const unsigned bdb = db ? unsigned(ceil_div(out, 256)) : 0u;
        EHIP_LAUNCH("linear_backward", linear_backward_small, dim3(bdx + bdw + bdb), dim3(256), 0,
                    as_stream(stream), args(dy, out, w, out, dx, rows, in, out), ndx, bdx,
                    args(x, in, dy, out, dw, in, out, rows), ndw, bdw, dy, db, int(rows),
                    int(out));
        return EHIP_OK;
    }
    if (db && dw && bias_from_dw(rows, in, out)) {
        // db from the column sums of dy that the dw product forms from the
        // tiles it stages (the two launches of the separate sum saved).
        if (dx) {
            if (int rc = ehip_gemm_f32(0, 1, 1, rows, in, out, dy, out, 0, w, out, 0, 0.0f, dx, in,
                                       0, stream))
                return rc;
        }
        ehip_gemm_ex_t d{};
        d.trans_a = 1;
        d.batch = 1;
        d.inner = 1;
        d.m = in;
        d.n = out;
        d.k = rows;
        d.a = x;
        d.lda = in;
        d.b = dy;
        d.ldb = out;
        d.c = dw;
        d.ldc = out;
        d.alpha = 1.0f;
        d.addend_period = 1;
        d.colsum_b = db;
        return ehip_gemm_ex_f32(&d, stream);
    }
    // dx = dy w^T and dw = x^T dy: the backward of x w, as one entry point (one
    // launch when both take the K-sliced tiles).
    if (int rc = ehip_matmul_backward_f32(rows, in, out, x, in, w, out, dy, out, dx, in, 0.0f, dw,
                                          out, 0.0f, stream))
        return rc;
    if (db) return ehip_sum_axis_f32(dy, db, 1, rows, out, stream);
    return EHIP_OK;
}

int ehip_linear_bias_from_dw(int on) {
    if (on < 0) return g_bias_from_dw.load() ? 1 : 0;
    return g_bias_from_dw.exchange(on != 0) ? 1 : 0;
}

int ehip_gemm_probe_arm(int trans_a, int trans_b, const int64_t* shapes, int count,
                        int max_products) {
    EHIP_READY();
    if (count < 1 || !shapes || max_products < 1 || max_products > 65536)
        return fail(EHIP_EINVAL, "gemm_probe_arm: %d shapes, %d products", count, max_products);
    std::lock_guard<std::mutex> lock(g_probe.mu);
    if (g_probe.armed.load()) return fail(EHIP_EINVAL, "gemm_probe_arm: already armed");
    g_probe.trans_a = trans_a ? 1 : 0;
    g_probe.trans_b = trans_b ? 1 : 0;
    g_probe.shapes.assign(shapes, shapes + 3 * size_t(count));
    g_probe.events.assign(2 * size_t(max_products), nullptr);
    for (hipEvent_t& e : g_probe.events)
        if (hipEventCreate(&e) != hipSuccess) {
            for (hipEvent_t& f : g_probe.events)
                if (f) (void)hipEventDestroy(f);
            g_probe.events.clear();
            return fail(EHIP_ELAUNCH, "gemm_probe_arm: event creation");
        }
    g_probe.used = 0;
    g_probe.flop = 0.0;
    g_probe.armed.store(true);
    return EHIP_OK;
}

int ehip_gemm_probe_read(double* ms, int64_t* products, double* flop) {
    EHIP_READY();
    std::lock_guard<std::mutex> lock(g_probe.mu);
    if (!g_probe.armed.load()) return fail(EHIP_EINVAL, "gemm_probe_read: not armed");
    g_probe.armed.store(false);
    double total = 0.0;
    int rc = EHIP_OK;
    for (size_t i = 0; i + 1 < g_probe.used; i += 2) {
        float t = 0.0f;
        if (hipEventSynchronize(g_probe.events[i + 1]) != hipSuccess ||
            hipEventElapsedTime(&t, g_probe.events[i], g_probe.events[i + 1]) != hipSuccess) {
            rc = fail(EHIP_ELAUNCH, "gemm_probe_read: event timing");
            break;
        }
        total += double(t);
    }
    for (hipEvent_t& e : g_probe.events) (void)hipEventDestroy(e);
    g_probe.events.clear();
    if (ms) *ms = total;
    if (products) *products = int64_t(g_probe.used / 2);
    if (flop) *flop = g_probe.flop;
    return rc;
}

int ehip_gemm_groupable(const ehip_gemm_ex_t* desc) {
    if (!desc || check_desc(*desc) != EHIP_OK) return 0;
    return takes_panel(*desc) ? 1 : 0;
}

int ehip_gemm_batch_f32(const ehip_gemm_ex_t* descs, int count, void* stream) {
    EHIP_READY();
    if (count < 0 || (count > 0 && !descs)) return fail(EHIP_EINVAL, "gemm_batch: bad list");
    for (int i = 0; i < count; ++i)
        if (int rc = check_desc(descs[i])) return rc;
    hipStream_t s = as_stream(stream);
    // The panel products in launches of up to kPanelGroupMax, the checked ones
    // first (their tiles take the longest: started first, they end with the
    // rest instead of after it); everything else one by one.
    std::vector<GemmArgs> list;
    std::vector<int> modes;
    std::vector<GemmArgs> ks[16];  // K-sliced A B products by kernel form
    for (int i = 0; i < count; ++i) {
        const ehip_gemm_ex_t& d = descs[i];
        if (d.batch == 0 || d.m == 0 || d.n == 0) continue;
        GemmArgs kg;
        int form = 0;
        if (!g_probe.armed.load() && takes_kslice_nn(d, kg, form)) {
            ks[form].push_back(kg);
            continue;
        }
        if (!takes_panel(d) || g_probe.armed.load()) {
            if (int rc = gemm_run(d, s)) return rc;
            continue;
        }
        GemmArgs g = args_of(d);
        g.vec = operands_aligned(g) ? 1 : 0;
        const bool whole = panel_geometry(g);
        list.push_back(g);
        modes.push_back((whole ? 0 : 1) | (plain_epilogue(g) ? 0 : 2));
    }
    std::vector<size_t> order(list.size());
    for (size_t i = 0; i < order.size(); ++i) order[i] = i;
    std::stable_partition(order.begin(), order.end(), [&](size_t i) { return modes[i] & 1; });
    for (size_t base = 0; base < list.size(); base += kPanelGroupMax) {
        PanelGroup p{};
        p.count = int(std::min<size_t>(kPanelGroupMax, list.size() - base));
        p.first[0] = 0;
        for (int j = 0; j < p.count; ++j) {
            p.g[j] = list[order[base + j]];
            p.mode[j] = modes[order[base + j]];
            p.first[j + 1] = p.first[j] + p.g[j].tiles_m * p.g[j].tiles_n;
        }
        EHIP_LAUNCH("gemm_batch", gemm_tn_panel_group, dim3(unsigned(p.first[p.count])),
                    dim3(64 * kPanelWaves), 0, s, p);
    }
    for (int form = 0; form < 16; ++form) {
        const std::vector<GemmArgs>& kl = ks[form];
        for (size_t base = 0; base < kl.size(); base += kPanelGroupMax) {
            PanelGroup p{};
            p.count = int(std::min<size_t>(kPanelGroupMax, kl.size() - base));
            for (int j = 0; j < p.count; ++j) {
                p.g[j] = kl[base + j];
                p.first[j + 1] = p.first[j] + p.g[j].tiles_m * p.g[j].tiles_n;
            }
            const int w = form / 4;
            const int rc = w == 0   ? launch_kslice_group<1>(p, form, s)
                           : w == 1 ? launch_kslice_group<2>(p, form, s)
                           : w == 2 ? launch_kslice_group<4>(p, form, s)
                                    : launch_kslice_group<8>(p, form, s);
            if (rc) return rc;
        }
    }
    return EHIP_OK;
}

int ehip_linear_backward_plan(int64_t rows, int64_t in, int64_t out) {
    if (rows <= 0 || in <= 0 || out <= 0) return 0;
    return bias_from_dw(rows, in, out) ? 1 : 0;
}

int ehip_gemm_ex_f32(const ehip_gemm_ex_t* desc, void* stream) {
    EHIP_READY();
    if (!desc) return fail(EHIP_EINVAL, "gemm_ex: null descriptor");
    const ehip_gemm_ex_t& d = *desc;
    if (int rc = check_desc(d)) return rc;
    if (d.batch == 0 || d.m == 0 || d.n == 0) return EHIP_OK;
    if (d.k == 0 && d.batch * d.m * d.n > 0x7fffffffLL)
        return fail(EHIP_EINVAL, "gemm_ex: K = 0 with more than 2^31 outputs");
    return gemm_run(d, as_stream(stream));
}

}  // extern "C"
