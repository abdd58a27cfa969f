// gemm_split.hpp -- the staged-tile GEMM: fp32 products on the bf16 matrix instructions. Each
// fp32 operand is the exact sum of three bf16 values, and the product is formed from six of the
// nine products of the parts, accumulated in fp32: the three-way split of Henry, Tang and Heinecke
// ("Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations",
// ARITH 2019).
//
// 2^24 x = h + m + l, each the round-to-nearest bf16 of what is left: 24 significand bits in
// 3 x 8. The last bit of an fp32 value is 2^-149 or more, so every part that is not zero is at
// least 2^-125, a normal bf16, and the split is exact for every |x| < 2^104. Of a b's nine part
// products the three smallest (m l, l m, l l: at most 2^-25 of |a b| together) are dropped; the
// six others are formed exactly by the matrix instruction and summed in fp32, 2^48 times their
// value. A part product below the fp32 range at that scale is below 2^-197 of the result's.
// v_mfma_f32_16x16x32_bf16 does 16 times the multiply-adds per cycle of the fp32 instructions,
// so six of them cost 3/8 of the fp32 product's matrix time.
//
// Error, against 64-bit products (2-norms; normal operands): K = 64 4.6e-8, K = 1024 1.13e-7,
// K = 4096 2.1e-7, where the chain of v_mfma_f32_32x32x2f32 that it replaces has 1.4e-7, 5.7e-7
// and 1.15e-6 (half-normal operands, half of them zero: 4.4e-8, 1.12e-7, 2.1e-7 against 1.0e-7,
// 4.0e-7 and 8.1e-7); the mean over a column of 2048 is off by 1.8e-9 of the results' rms at K = 64
// and 2.4e-9 at K = 1024, against 3.3e-9 and 9.2e-9. A step's 32 k are summed apart from the
// accumulator (split_products) and their losses made to cancel (split_flip); all nine part products
// would give the same figures.
//
// What bounds it: the matrix pipe at the clock the chip sustains. The bare instruction reaches
// 1,950 TFLOP/s of its 2,500, i.e. 325 fp32 TFLOP/s with six products; 8192 x 1024 x 4096 runs
// 192-219 by box (fp32 instructions: 127-131), the conversion and the sums taking about half of the
// issue slots beside it. Measured and left out: the 32 x 32 x 16 instruction (212-227 where this
// one, without the sums apart, has 222-236), the conversion before or after the products by
// halves of the waves (200-207), raised priority around the products (216-232), loads two steps
// ahead in a second register set (spills with the sums apart: 203-215).
#ifndef EHIP_GEMM_SPLIT_HPP
#define EHIP_GEMM_SPLIT_HPP

#include "gemm_kernel.hpp"

namespace ehip {
namespace gemm_detail {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
// Four floats at any float's address (global memory takes 16-byte accesses at 4-byte
// alignment on gfx950).
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
// A byte address in global memory, said so: loads through an address whose origin the compiler
// cannot see would otherwise be flat ones, which also occupy the LDS counter.
typedef const __attribute__((address_space(1))) char* global_bytes;

template <class T>
__device__ __forceinline__ T global_load(global_bytes p) {
    return *reinterpret_cast<const __attribute__((address_space(1))) T*>(p);
}

__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){a, b}, bf16x2));
}

// The three parts of a and b (scaled), two bf16 to a word. An operand that is inf or NaN (or
// scales or rounds to inf) leaves NaN in its last part, and so in every result it takes part in.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& h, uint32_t& m,
                                           uint32_t& l) {
    h = bf16_pair(a, b);
    float ra = a - __builtin_bit_cast(float, h << 16);
    float rb = b - __builtin_bit_cast(float, h & 0xffff0000u);
    m = bf16_pair(ra, rb);
    ra = ra - __builtin_bit_cast(float, m << 16);
    rb = rb - __builtin_bit_cast(float, m & 0xffff0000u);
    l = bf16_pair(ra, rb);
}

constexpr int kSplitBK = 32;
// Products of fewer k are formed by the fp32 instructions: one or two roundings there, where the
// dropped parts and the sums' truncation cost more (error against 64 bits at K = 1 2.5e-8 :
// 3.4e-8, K = 2 3.1e-8 : 3.4e-8, K = 3 of half-normal operands 3.0e-8 : 3.2e-8, from K = 4 on
// smaller in parts, 4.0e-8 : 3.2e-8).
constexpr int kSplitMinK = 4;

// The sign bit for odd n. The matrix instruction drops the low bits of its sums towards minus
// infinity, which leaves every result the same fraction of an ulp low: in odd K steps B is staged
// negated and the sum subtracted, and the losses of a pair of steps cancel. In the steps that are
// left of a chunk of K after its whole pairs (from split_pairs on), odd rows of A and odd columns of B
// are negated too and the sums added with the product of the three signs, so that their losses
// cancel over neighbouring rows and columns (mean of 2048 x 2048 results' errors over the results'
// rms, at K = 32, with the steps' signs alone -6.1e-9, so less than its own spread, 2e-11; of
// operands of one sign -2.3e-9, so -1.2e-10).
__device__ __forceinline__ uint32_t split_flip(int n) { return uint32_t(n) << 31; }
__device__ __forceinline__ int split_pairs(int64_t chunk) { return int(chunk / kSplitBK) & ~1; }

// What an operand is multiplied by as it is split: 2^24, which keeps the parts of the smallest
// values inside bf16's range (without it a part is lost from |x| < 2^-110 on: a row of 2^-122
// among rows of 1 kept 13 bits) for about 1 % of the time (8192 x 1024 x 4096 with both its
// backward products 1039 -> 1050 us). With the sign of n: of A's row, or of the step and B's column.
__device__ __forceinline__ float split_scale(int n) {
    return __builtin_bit_cast(float, 0x4b800000u ^ split_flip(n));
}

// One operand's tile of ROWS rows (of op(A), or columns of op(B)) by 32 k. KC: element (r, k)
// is at p[r * ld + k], else at p[k * ld + r]. A thread stages kUnits units of one row by 8
// consecutive k: loaded as two 16-byte loads (KC; four lanes read a row's 128 bytes) or as
// eight 4-byte loads (a wave reads 256 consecutive bytes), either way ending in the eight
// registers that pack into one 16-byte LDS write per part, with no transposition.
//
// LDS: three planes (h, m, l), each 16-row blocks of 1 KiB holding [k / 8][row % 16] 16-byte
// groups, which is the matrix instruction's operand order: one conflict-free ds_read_b128 per
// 16 x 32 block. The row's place is permuted within its group of 16 so that the writes of
// eight lanes also fall on different banks, whether they hold two rows by four k groups (KC)
// or eight rows.
template <int ROWS, bool KC, int THREADS>
struct SplitTile {
    static constexpr int kUnits = ROWS * (kSplitBK / 8) / THREADS;
    static constexpr int kPlane = ROWS * kSplitBK * 2;  // bytes
    static_assert(kUnits >= 1 && kUnits * THREADS == ROWS * (kSplitBK / 8), "tile shape");

    float v[kUnits][8];

    __device__ __forceinline__ static int row(int u) {
        const int q = int(threadIdx.x) + u * THREADS;
        return KC ? q / 4 : q % ROWS;
    }
    __device__ __forceinline__ static int group(int u) {
        const int q = int(threadIdx.x) + u * THREADS;
        return KC ? q % 4 : q / ROWS;
    }
    __device__ __forceinline__ static int slot(int r, int kc) {
        return (r / 16) * 1024 + kc * 256 + (((r & 15) ^ ((r >> 3) & 1) ^ (2 * kc)) << 4);
    }
    // Byte offsets of the thread's units from the tile's first element; rows past the last
    // one repeat it (their results are not stored).
    __device__ __forceinline__ static void offsets(uint32_t (&o)[kUnits], int64_t ld,
                                                   int64_t rows_left) {
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            const int64_t r = row(u) < rows_left ? row(u) : rows_left - 1;
            o[u] = uint32_t(4 * (KC ? r * ld + 8 * group(u) : 8 * group(u) * ld + r));
        }
    }
    __device__ __forceinline__ void load(global_bytes base, const uint32_t (&o)[kUnits],
                                         int64_t ld) {
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            if constexpr (KC) {
                const floatx4u x = global_load<floatx4u>(base + o[u]);
                const floatx4u y = global_load<floatx4u>(base + o[u] + 16);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[u][j] = x[j];
                    v[u][4 + j] = y[j];
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    v[u][j] = global_load<float>(base + 4 * j * ld + o[u]);
            }
        }
    }
    // The same for a tile of which only the first `left` k are in the matrix (zeros after
    // them), with 64-bit offsets: the last step of a K that is no multiple of 32, and every
    // step where a leading dimension is too large for offsets(). KC: units wholly inside load as
    // above (a K of 16 or 24 is one such step: 18 x 242 x 242 x 16, A B^T, 9.0 -> 6.9 us), those
    // wholly outside not at all. Otherwise k past the last read the first again, for mask_tail to
    // zero once the loads have been waited for.
    __device__ __forceinline__ void load_tail(global_bytes base, int64_t ld, int64_t rows_left,
                                              int left) {
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            const int64_t r = row(u) < rows_left ? row(u) : rows_left - 1;
            if constexpr (KC) {
                const int in = left - 8 * group(u);
                const global_bytes p = base + 4 * (r * ld + 8 * group(u));
#pragma unroll
                for (int j = 0; j < 8; ++j) v[u][j] = 0.0f;
                if (in >= 8) {
                    const floatx4u x = global_load<floatx4u>(p);
                    const floatx4u y = global_load<floatx4u>(p + 16);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        v[u][j] = x[j];
                        v[u][4 + j] = y[j];
                    }
                } else if (in > 0) {
#pragma unroll
                    for (int j = 0; j < 7; ++j) {
                        const float x = global_load<float>(p + 4 * (j < in ? j : 0));
                        v[u][j] = j < in ? x : 0.0f;
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int k = 8 * group(u) + j;
                    v[u][j] = global_load<float>(base + 4 * ((k < left ? k : 0) * ld + r));
                }
            }
        }
    }
    __device__ __forceinline__ void mask_tail(int left) {
        if constexpr (!KC) {
#pragma unroll
            for (int u = 0; u < kUnits; ++u)
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    v[u][j] = 8 * group(u) + j < left ? v[u][j] : 0.0f;
        }
    }
    // Splits the registers, times `scale` (split_scale), into the three planes. A thread's units
    // are rows of one parity, that of row(0).
    __device__ __forceinline__ void store(char* lds, float scale) const {
        static_assert(THREADS % 8 == 0 && ROWS % 2 == 0, "rows of one parity");
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            uintx4 h, m, l;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t hj, mj, lj;
                split_pair(v[u][2 * j] * scale, v[u][2 * j + 1] * scale, hj, mj, lj);
                h[j] = hj;
                m[j] = mj;
                l[j] = lj;
            }
            char* d = lds + slot(row(u), group(u));
            *reinterpret_cast<uintx4*>(d) = h;
            *reinterpret_cast<uintx4*>(d + kPlane) = m;
            *reinterpret_cast<uintx4*>(d + 2 * kPlane) = l;
        }
    }
};

// One staged K step (s) of a wave: acc += its 16 FM x 16 FN tile over 32 k; sa and sb are the
// lane's place in the first block of the operands' h planes. One block row of A at a time (all
// of them at once spill in the shapes that run three and four waves per SIMD). Smallest part
// products first; the operands swapped, so that a lane's four results are four consecutive
// columns of a row. The step's sum is formed apart and added to the accumulator once, which
// rounds the accumulator once per 32 k instead of once per 8 k of each part product (K = 1024:
// error 4.85e-7 -> 1.18e-7, for 3 to 6 % of the time).
template <int FM, int FN, int PLANE_A, int PLANE_B>
__device__ __forceinline__ void split_products(floatx4 (&acc)[FM][FN], const char* sa,
                                               const char* sb, int s, int unpaired) {
    // 2^-48, with the sign of the step, of the lane's row of A and of its even or odd columns of B.
    const float even = __builtin_bit_cast(
        float, 0x27800000u ^ split_flip(s ^ (int(threadIdx.x) & unpaired)));
    const float odd =
        __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, even) ^ split_flip(unpaired));
    constexpr int kPart[6][2] = {{1, 1}, {2, 0}, {0, 2}, {0, 1}, {1, 0}, {0, 0}};
    constexpr int SUMS = 2;
    bf16x8 fb[3][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        bf16x8 fa[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            fa[2 - q] = *reinterpret_cast<const bf16x8*>(sa + (2 - q) * PLANE_A + 1024 * i);
            if (i == 0) {
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    fb[q][j] = *reinterpret_cast<const bf16x8*>(sb + q * PLANE_B + 1024 * j);
            }
        }
#pragma unroll
        for (int j0 = 0; j0 < FN; j0 += SUMS) {
            floatx4 t[SUMS];
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int j = 0; j < SUMS; ++j)
                    t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        fb[kPart[q][1]][j0 + j], fa[kPart[q][0]],
                        q == 0 ? (floatx4){0.0f, 0.0f, 0.0f, 0.0f} : t[j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < SUMS; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[i][j0 + j][r] =
                        __builtin_fmaf(t[j][r], r % 2 ? odd : even, acc[i][j0 + j][r]);
        }
    }
}

// Whether the workgroup's tile holds what the split cannot carry: a result that is not finite.
// An inf or NaN among the operands, or a value of 2^104 or more, makes NaN of every result it
// takes part in; 32 k whose products sum to 2^80 or more leave the fp32 range at the sums' scale.
// The whole tile is then formed again by the fp32 instructions. Every wave must have finished
// reading the staged tiles (`lds`).
template <int WAVES, int FM, int FN>
__device__ __forceinline__ bool split_failed(const floatx4 (&acc)[FM][FN], char* lds) {
    bool finite = true;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                finite = finite && fabsf(acc[i][j][r]) < __builtin_inff();
    int* vote = reinterpret_cast<int*>(lds);
    const int failed = __any(!finite) ? 1 : 0;
    if (threadIdx.x % 64 == 0) vote[threadIdx.x / 64] = failed;
    __syncthreads();
    int any = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) any |= vote[w];
    return __builtin_amdgcn_readfirstlane(any) != 0;
}

// Stores the wave's accumulators through the epilogue. Block (i, j), lane l, register r is
// element (16 i + l % 16, 16 j + 4 (l / 16) + r) of the wave's tile: four consecutive columns
// of a row per lane, one 16-byte access each for the output, the addend, the old output and
// the residual. The loads of a block row come before its stores (the compiler cannot move a
// load above an earlier store to C, which may alias it).
template <int FM, int FN, bool CHECK, bool EPI>
__device__ __forceinline__ void split_store(const GemmArgs& g, const floatx4 (&acc)[FM][FN],
                                            float* Cp, int64_t ldc, const float* addp,
                                            int64_t row0, int64_t col0) {
    const auto get = [&](const float* p, int64_t col) {
        if (!CHECK || col + 4 <= g.n) return floatx4(*reinterpret_cast<const floatx4u*>(p));
        floatx4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (col + r < g.n) v[r] = p[r];
        return v;
    };
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int64_t row = row0 + 16 * i;
        if (CHECK && row >= g.m) continue;
        floatx4 add[FN], old[FN], res[FN];
        if constexpr (EPI) {
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int64_t col = col0 + 16 * j;
                const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
                add[j] = old[j] = res[j] = zero;
                if (CHECK && col >= g.n) continue;
                if (addp != nullptr) {
                    if (g.add_row) {
                        const float a = addp[row];
                        add[j] = (floatx4){a, a, a, a};
                    } else {
                        add[j] = get(addp + row * g.ld_add + col, col);
                    }
                }
                if (g.beta != 0.0f) old[j] = get(Cp + row * ldc + col, col);
                if (g.res != nullptr) res[j] = get(g.res + row * g.ld_res + col, col);
            }
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int64_t col = col0 + 16 * j;
            if (CHECK && col >= g.n) continue;
            floatx4 v = acc[i][j];
            if constexpr (EPI) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    v[r] = finish(g, v[r], add[j][r], old[j][r], res[j][r]);
            }
            float* dst = Cp + row * ldc + col;
            if (!CHECK || col + 4 <= g.n) {
                *reinterpret_cast<floatx4u*>(dst) = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (col + r < g.n) dst[r] = v[r];
            }
        }
    }
}

__device__ __forceinline__ int64_t uniform64(int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane(int(uint32_t(v)));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(int(uint32_t(uint64_t(v) >> 32)));
    return int64_t(uint64_t(hi) << 32 | lo);
}

// Whether the byte offsets of SplitTile::offsets fit 32 bits (at most 256 rows of ld floats).
__device__ __forceinline__ bool split_offsets_fit(const GemmArgs& g) {
    return g.lda < (int64_t(1) << 21) && g.ldb < (int64_t(1) << 21);
}

template <int BM, int BN, int WM, int WN>
struct TileThreads {
    static constexpr int value = (BM / WM) * (BN / WN) * 64;
};

template <int BM, int BN, int WM, int WN, int STAGES, int MINW, bool TA, bool TB, bool COLSUM>
__global__ __launch_bounds__((TileThreads<BM, BN, WM, WN>::value), MINW) void gemm_kernel(
    GemmArgs g) {
    constexpr int kThreads = TileThreads<BM, BN, WM, WN>::value, kWaves = kThreads / 64;
    using A = SplitTile<BM, !TA, kThreads>;
    using B = SplitTile<BN, TB, kThreads>;
    constexpr int kStage = 3 * (A::kPlane + B::kPlane);
    constexpr int FM = WM / 16, FN = WN / 16;
    __shared__ __attribute__((aligned(16))) char lds[STAGES * kStage];

    const int tiles = g.tiles_m * g.tiles_n;
    int tm, tn;
    int64_t batch = g.batch0 + blockIdx.z;
    if (g.causal != 0 && gridDim.y == 1) {
        const int64_t lin = int64_t(blockIdx.z) * gridDim.x + blockIdx.x;
        batch = g.batch0 + lin % gridDim.z;
        const int t = int(lin / gridDim.z);
        tm = t / g.tiles_n;
        tn = t % g.tiles_n;
    } else {
        int bid = blockIdx.x;
        if (tiles % 8 == 0) bid = (bid % 8) * (tiles / 8) + bid / 8;
        constexpr int kGroupM = 8;
        const int group = bid / (kGroupM * g.tiles_n);
        const int first_m = group * kGroupM;
        const int gsz = min(g.tiles_m - first_m, kGroupM);
        const int in_group = bid % (kGroupM * g.tiles_n);
        tm = first_m + in_group % gsz;
        tn = in_group / gsz;
    }
    // Uniform by construction; said so, for the scalar addresses below (the divisions above
    // run in vector registers).
    tm = __builtin_amdgcn_readfirstlane(tm);
    tn = __builtin_amdgcn_readfirstlane(tn);
    batch = uniform64(batch);
    const int split = blockIdx.y;
    const float* Ap = g.a + uniform64(batch_offset(batch, g.inner, g.stride_a, g.stride_a2));
    const float* Bp = g.b + uniform64(batch_offset(batch, g.inner, g.stride_b, g.stride_b2));
    const int64_t m0 = int64_t(tm) * BM, n0 = int64_t(tn) * BN;
    int64_t k_begin = int64_t(split) * g.k_chunk;
    int64_t k_end = k_begin + g.k_chunk;
    if (k_end > g.k) k_end = g.k;
    if (g.causal == 4 && n0 >= m0 + BM) return;
    if (g.causal == 1 && n0 >= m0 + BM) {
        k_end = k_begin;
    } else if (g.causal == 2) {
        if (k_end > m0 + BM) k_end = k_begin > m0 + BM ? k_begin : m0 + BM;
    } else if (g.causal == 3) {
        if (k_begin < m0) k_begin = k_end < m0 ? k_end : m0;
    }

    // The signs go by the chunk and count its steps from its first k, so that a product that
    // skips k keeps those of the product that does not (BM and the chunks are multiples of a
    // step). The chunk's pairs are even in number of steps, so this, the first step after them
    // counted from k_begin, is odd where k_begin lies an odd number of steps into the chunk.
    const int64_t chunk0 = int64_t(split) * g.k_chunk;
    const int pairs = __builtin_amdgcn_readfirstlane(
        split_pairs(min(g.k - chunk0, g.k_chunk)) - int((k_begin - chunk0) / kSplitBK));

    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int wm0 = (wave / (BN / WN)) * WM, wn0 = (wave % (BN / WN)) * WN;

    floatx4 acc[FM][FN];
    const auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = (floatx4){0.0f, 0.0f, 0.0f, 0.0f};
    };
    clear();
    const int steps =
        __builtin_amdgcn_readfirstlane(int((k_end - k_begin + kSplitBK - 1) / kSplitBK));
    // Whole steps, loaded without guards.
    const int full = split_offsets_fit(g) ? int((k_end - k_begin) / kSplitBK) : 0;
    const auto pa = (global_bytes)(TA ? Ap + k_begin * g.lda + m0 : Ap + m0 * g.lda + k_begin);
    const auto pb = (global_bytes)(TB ? Bp + n0 * g.ldb + k_begin : Bp + k_begin * g.ldb + n0);
    const int64_t da = 4 * kSplitBK * (TA ? g.lda : 1), db = 4 * kSplitBK * (TB ? 1 : g.ldb);
    uint32_t oa[A::kUnits], ob[B::kUnits];
    A::offsets(oa, g.lda, g.m - m0);
    B::offsets(ob, g.ldb, g.n - n0);
    A ta;
    B tb;
    float csum[COLSUM ? B::kUnits : 1] = {};
    const int fbase = A::slot(lane % 16, lane / 16);

    // The step's base addresses, opaque to the optimiser: it would otherwise carry every
    // load's address through the loop as a 64-bit register pair of its own (91 spilled
    // registers in the A^T B form) instead of a scalar base and a 32-bit offset.
    const auto scalar = [](global_bytes p) {
        asm volatile("" : "+s"(p));
        return p;
    };
    const auto load = [&](int s) {
        ta.load(TA ? scalar(pa + s * da) : pa + s * da, oa, g.lda);
        tb.load(TB ? pb + s * db : scalar(pb + s * db), ob, g.ldb);
    };
    const auto left = [&](int s) {
        return int(min(k_end - k_begin - int64_t(s) * kSplitBK, int64_t(kSplitBK)));
    };
    const auto load_any = [&](int s) {
        if (s < full) {
            load(s);
        } else {
            ta.load_tail(pa + s * da, g.lda, g.m - m0, left(s));
            tb.load_tail(pb + s * db, g.ldb, g.n - n0, left(s));
        }
    };
    const auto mask = [&](int s) {
        if (s >= full) {
            ta.mask_tail(left(s));
            tb.mask_tail(left(s));
        }
    };
    // `unpaired` masks the rows' and columns' signs: none in the steps that the unguarded loops
    // below run, which leave the last two whole steps (a single stage: one) to those after them.
    const auto convert = [&](int s, int unpaired) {
        char* st = lds + (STAGES == 2 ? (s & 1) * kStage : 0);
        ta.store(st, split_scale(A::row(0) & unpaired));
        tb.store(st + 3 * A::kPlane, split_scale((s + pairs) ^ (B::row(0) & unpaired)));
        if constexpr (COLSUM) {
#pragma unroll
            for (int u = 0; u < B::kUnits; ++u) {
                const float* v = tb.v[u];
                csum[u] += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
            }
        }
    };
    const auto multiply = [&](int s, int unpaired) {
        const char* st = lds + (STAGES == 2 ? (s & 1) * kStage : 0);
        split_products<FM, FN, A::kPlane, B::kPlane>(
            acc, st + (wm0 / 16) * 1024 + fbase,
            st + 3 * A::kPlane + (wn0 / 16) * 1024 + fbase, s + pairs, unpaired);
    };

    const auto unpaired = [&](int s) { return s >= pairs ? -1 : 0; };

    // Two stages: while a step's products run, the next step is converted into the other stage
    // and the one after it loaded. One stage: the waves of the CU's other workgroups fill the
    // conversion phase.
    if constexpr (STAGES == 2) {
        if (steps > 0) {
            load_any(0);
            mask(0);
            convert(0, unpaired(0));
            if (steps > 1) load_any(1);
            __syncthreads();
        }
        int s = 0;
        for (; s + 2 < full; ++s) {
            multiply(s, 0);
            convert(s + 1, 0);
            load(s + 2);
            __syncthreads();
        }
        for (; s < steps; ++s) {
            multiply(s, unpaired(s));
            if (s + 1 < steps) {
                mask(s + 1);
                convert(s + 1, unpaired(s + 1));
            }
            if (s + 2 < steps) load_any(s + 2);
            __syncthreads();
        }
    } else {
        if (steps > 0) load_any(0);
        int s = 0;
        for (; s + 1 < full; ++s) {
            convert(s, 0);
            load(s + 1);
            __syncthreads();
            multiply(s, 0);
            __syncthreads();
        }
        for (; s < steps; ++s) {
            mask(s);
            convert(s, unpaired(s));
            if (s + 1 < steps) load_any(s + 1);
            __syncthreads();
            multiply(s, unpaired(s));
            __syncthreads();
        }
    }

    if (g.k < kSplitMinK || split_failed<kWaves>(acc, lds)) {
        clear();
#pragma unroll 1
        for (int64_t k = k_begin; k < k_end; k += 4) {
            const int64_t kk = k + lane / 16;
            const bool in = kk < k_end;
            float fa[FM], fb[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                const int64_t r = m0 + wm0 + 16 * i + lane % 16;
                fa[i] = in && r < g.m ? (TA ? Ap[kk * g.lda + r] : Ap[r * g.lda + kk]) : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int64_t c = n0 + wn0 + 16 * j + lane % 16;
                fb[j] = in && c < g.n ? (TB ? Bp[c * g.ldb + kk] : Bp[kk * g.ldb + c]) : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j], fa[i], acc[i][j], 0, 0, 0);
        }
    }

    if constexpr (COLSUM) {
        // Column sums of B: a thread holds the sums over its k group of every step; the four
        // groups of a column are added in order.
        if (tm == 0) {
            float* part = reinterpret_cast<float*>(lds) + 64;
#pragma unroll
            for (int u = 0; u < B::kUnits; ++u) part[B::group(u) * BN + B::row(u)] = csum[u];
            __syncthreads();
            const int c = threadIdx.x;
            if (c < BN && n0 + c < g.n) {
                const float v = ((part[c] + part[BN + c]) + part[2 * BN + c]) + part[3 * BN + c];
                if (g.splits > 1)
                    g.c[int64_t(split) * g.ws_stride + g.m * g.n + n0 + c] = v;
                else
                    g.colsum[n0 + c] = v;
            }
        }
    }

    float* Cp;
    int64_t ldc;
    if (g.splits > 1) {
        Cp = g.c + int64_t(split) * g.ws_stride + batch * g.m * g.n;
        ldc = g.n;
    } else {
        Cp = g.c + batch_offset(batch, g.inner, g.stride_c, g.stride_c2);
        ldc = g.ldc;
    }
    const float* addp = g.add ? g.add + (int64_t(batch) % g.add_period) * g.stride_add : nullptr;
    const bool inside = m0 + BM <= g.m && n0 + BN <= g.n;
    const bool epi = g.splits == 1 && !plain_epilogue(g);
    const int64_t row0 = m0 + wm0 + lane % 16, col0 = n0 + wn0 + 4 * (lane / 16);
    if (inside && !epi)
        split_store<FM, FN, false, false>(g, acc, Cp, ldc, addp, row0, col0);
    else if (inside)
        split_store<FM, FN, false, true>(g, acc, Cp, ldc, addp, row0, col0);
    else if (!epi)
        split_store<FM, FN, true, false>(g, acc, Cp, ldc, addp, row0, col0);
    else
        split_store<FM, FN, true, true>(g, acc, Cp, ldc, addp, row0, col0);
}

// The staged tiles' shapes (gemm_kernel). per_cu: how many of a shape's workgroups a CU holds
// (LDS and registers); rate: the throughput of a full CU relative to the first shape's,
// measured on MI355X at 8192 x 1024 x 4096 (217-221, 197, 171 and 152 TFLOP/s on one box, before
// the operands were scaled).
struct TileShape {
    int bm, bn, per_cu;
    double rate;
};
inline constexpr TileShape kShapes[] = {{256, 128, 1, 1.0}, {128, 128, 2, 0.9}, {128, 64, 3, 0.78},
                                        {64, 64, 3, 0.67}};
constexpr double kCuFlopPerUs = 0.85e6;  // the first shape's, 218 TFLOP/s on 256 CUs
// What is left of a CU's rate when it holds c of a shape's per_cu workgroups: alone, a
// workgroup has nothing to run in its load and conversion phases (1999 x 1531 x 777 in 192
// workgroups of 128 x 128: 56 us, in 576 of a third of K each: 46 us).
inline double share(int c, int per_cu) {
    if (c >= per_cu) return 1.0;
    return c == 1 ? (per_cu == 2 ? 0.65 : 0.5) : 0.8;
}

struct StagedPlan {
    int shape, splits;
};

// The shape and K split of least estimated time for `batch` products m x n x k, among the shapes
// from `first` on and at most max_splits splits: whole rounds of the chip's 256 CUs, then the
// last one's workgroups spread over them, 3 us of prologue and epilogue per round; a split adds
// its workspace traffic and the reduction (1999 x 1531 in 3 splits: 13 us, which one round of
// 64 x 64 tiles over the whole K saves). No fewer than an eighth of max_splits: the chains of a
// sum grow with fewer splits, and so does its error, with their length's square root -- these
// tiles' is below a quarter of the error of the fp32 chains that max_splits was planned for.
// The largest tile runs one workgroup per CU, so nothing covers its first loads and its stores:
// not below 128 k (A B^T 8192 x 2048 x 16: 27 us, in 128 x 128 tiles 21; x 64 27 : 25; x 128
// 36 : 34, 6564 x 1024 x 128 19 : 19).
// Every shape forms an element by the same chain of instructions; the splits fix its bits.
inline StagedPlan plan_staged(int64_t m, int64_t n, int64_t k, int64_t batch, int max_splits,
                              int first = 0) {
    constexpr int kCount = int(sizeof(kShapes) / sizeof(kShapes[0]));
    StagedPlan best{first, max_splits};
    double best_t = 0.0;
    for (int s = (max_splits + 7) / 8; s <= max_splits; ++s) {
        const int64_t chunk = ceil_div(ceil_div(k, s), kSplitBK) * kSplitBK;
        if (s > 1 && ceil_div(k, chunk) != s) continue;
        const double out = 4.0 * double(m) * double(n) * double(batch);
        const double reduce = s > 1 ? 4.0 + out * (s + 1) / 4e6 + out * (s - 1) / 5e6 : 0.0;
        for (int i = chunk < 128 && first == 0 ? 1 : first; i < kCount; ++i) {
            const TileShape& t = kShapes[i];
            const int64_t work = ceil_div(m, t.bm) * ceil_div(n, t.bn) * batch * s;
            const int64_t slots = int64_t(256) * t.per_cu;
            const double unit = 2.0 * t.bm * t.bn * double(chunk) / (t.rate * kCuFlopPerUs);
            const int last = int(ceil_div(work % slots, 256));
            double time = reduce + double(work / slots) * (t.per_cu * unit + 3.0);
            if (last > 0) time += last * unit / share(last, t.per_cu) + 3.0;
            if (best_t == 0.0 || time < best_t) {
                best = {i, s};
                best_t = time;
            }
        }
    }
    return best;
}

}  // namespace gemm_detail
}  // namespace ehip

#endif  // EHIP_GEMM_SPLIT_HPP
