// hive_fnn.hip -- the FNN leaf evaluation of the self-play search, fused.
//
// The reference evaluates a batch of leaves with a chain of torch ops
// (fnn_mcts_orchestrator.py:243-316 over fnn_network.py:175-220): legal-slot
// masks, row lists, successor features, concatenation, fc1, sigmoid,
// LayerNorm, fc2, value head, action tower over [root | successor]
// embeddings, scatter into [T, 256] logits, softmax, child-Q scatter.  Here
// the whole network runs in one kernel per row kind, with the weights held in
// LDS and the three layer products on matrix cores:
//
//   k_leaf_mlp<root>   per leaf row: embedding e = fc2(LN(sigmoid(fc1 x))),
//                      value tanh(value_fc e), and the root half of the
//                      action tower's first layer r = Wr e + b (Wr =
//                      action_fc1.weight[:, :64]), kept as [T][64];
//   k_leaf_mlp<succ>   per successor row: e as above, child value
//                      tanh(value_fc e), and the action logit
//                      action_fc2(sigmoid(Ws e + r[leaf])) (Ws =
//                      action_fc1.weight[:, 64:]), so [root | successor] is
//                      never materialised;
//   k_leaf_softmax     per leaf: softmax of its logits over its legal slots,
//                      priors / child Q (= -child value) as [T][256] rows,
//                      zero beyond the legal count.
//
// The products run on the bf16 matrix cores at float32's accuracy: a float
// is the exact sum of three bf16 parts (8 significant bits each: the second is
// at most 2^-9 of the first, the third 2^-18), and of the nine products of two
// such sums the six down to 2^-18 of the whole are taken,
// v_mfma_f32_16x16x32_bf16 each, accumulated in float32.  That is six times the
// multiplications at sixteen times the rate of the fp32 matrix instruction;
// what is left out is at most 2^-26, a quarter of a float32 rounding.  The
// weights are split once per evaluation, the activations as they come.
// Measured against the fp32 instruction (427 K successor rows): 143 -> 91 us,
// 78 us with the units' records for features, the sums started from the biases
// and fused multiply-adds around the products; the outputs' distance from
// float64 is the same (1.4e-7 / 1.4e-7 to 8.5e-7 / 7.7e-7 relative over the seeds
// tried).  Bound now by VALU issue (805 a tile besides the products, a third of
// it the splits) and the matrix pipe (168 instructions a tile, 16 cycles each):
// 84 K and 70 K of a SIMD's 171 K cycles, which add up; not by the 96 KB of LDS
// reads a tile: two tiles per read took as long (85.7 us against 85.9 before
// the multiply-adds).
//
// Matrix-core layout (16x16x32, D = A.B + C, A 16x32, B 32x16): lane l holds
// A[l%16][8 (l/16) + j], B[8 (l/16) + j][l%16] (j < 8) and D[4(l/16)+i][l%16]
// in its four accumulator registers i.  A wave evaluates 16 rows at a time
// and computes every layer transposed, out^T = W . in^T: A = 16 output units
// of W, B = the inputs of the 16 rows, so after a layer lane l holds, for row
// l%16, the 16 units {16t + 4(l/16) + i : t, i < 4} of its output.  Those are
// exactly the B operands the next layer needs when the input of step s at
// lane group g = l/16, element j is unit 16 (2s + j/4) + 4g + j%4: no
// transposes, no LDS traffic between layers.  The weights are stored in LDS
// pre-permuted to that order ([step][tile][part][lane], conflict-free 16-byte
// reads).  The first layer's input of step s, lane group g, element j follows
// the features' six sections of 16 classes: a quarter of each section per lane
// group (feature_of), so that a lane can build its 32 inputs from a successor's
// packed record (unit_slice) with the same code in every lane; the counts among
// them (steps 0 and 2) are one bf16 part exactly.
//
// LayerNorm, value and logit reductions over the 64 units of a row are a
// sum over the lane's 16 units plus two cross-lane steps (lanes l, l^16,
// l^32, l^48 share a row).
//
// Rows that come out NaN are worked out again without the split
// (leaf_plain_row): infinite operands have none.
//
// Floating point: everything between the products in fp32 with the reference's
// operations (eps 1e-5, biased variance; sigmoid from the hardware exp2 /
// reciprocal); summation orders differ from torch's GEMMs, so results agree
// with the torch composition to ~1e-6 relative, not bit for bit.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/hive_gpu.h"
#include "hive_leaf.hpp"

namespace {

constexpr int kE = 64;       // hidden / embedding / action-tower width served here
constexpr int kFMax = 128;   // feature rows up to 128 wide (Hive FNN: 122)
constexpr int kSlots = 256;  // legal-slot rows of priors / child Q
// 16 waves share one LDS copy of the split weights (98 KB): one resident block
// per CU, 4 waves per SIMD to overlap the element-wise work and loads with
// the matrix cores
constexpr int kBlockWaves = 16;
constexpr int kMaxBlocks = 256;  // one resident block on each of 256 CUs

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

// The network in the order the MLP kernels keep it in LDS, split into bf16
// parts once per evaluation (pack_net_at, in the evaluation's first launch),
// so that each of their blocks fills LDS with straight 16-byte copies.
// Element [step][tile][part][lane] holds the lane's eight weights.
struct PackedNet {
    b8 w1[4][4][3][64];     // fc1, input feature_of(s, g, j)
    b8 w2[2][4][3][64];     // fc2, input 16 (2s + j/4) + 4g + j%4
    b8 w3[2][2][4][3][64];  // action_fc1: root half, successor half, as fc2
    float vec[7][kE];
};
struct MlpLds {
    b8 w1[4][4][3][64];
    b8 w2[2][4][3][64];
    b8 w3[2][4][3][64];  // action_fc1 root half (root rows) or successor half (successor rows)
    float vec[7][kE];
};
enum { kB1, kLnW, kLnB, kB2, kWv, kWa2, kBa1 };

// x as three bf16 parts, x = p0 + p1 + p2 exactly (each remainder is exact in
// float32 and has eight bits fewer; parts below bf16's range are dropped)
__device__ __forceinline__ void split3(f2 x, b2& p0, b2& p1, b2& p2) {
    p0 = __builtin_convertvector(x, b2);
    const f2 r = x - __builtin_convertvector(p0, f2);
    p1 = __builtin_convertvector(r, b2);
    p2 = __builtin_convertvector(r - __builtin_convertvector(p1, f2), b2);
}

// The feature that fc1's step s takes at lane group g, element j: sections 0
// and 2, 1 and 3, 4 and 5 (top pieces, next to the queen; hands, distances;
// can move, pinned), four classes of each, then eight of the last 32.
__host__ __device__ constexpr int feature_section(int s, int j) { return s == 2 ? 4 + (j >> 2) : s + 2 * (j >> 2); }
__host__ __device__ constexpr int feature_of(int s, int g, int j) {
    return s < 3 ? 16 * feature_section(s, j) + 4 * g + (j & 3) : 96 + 8 * g + j;
}

// Weight i of a [step][tile][lane][j] array: unit m = 16 tile + lane % 16 and
// its input k; at: the element's place in the split array, parts 64 * 8 apart.
__device__ __forceinline__ void perm_index(int i, bool first, int& m, int& k, int& at) {
    const int j = i & 7, l = (i >> 3) & 63, t = (i >> 9) & 3, s = i >> 11, g = l >> 4;
    m = 16 * t + (l & 15);
    k = first ? feature_of(s, g, j) : 16 * (2 * s + (j >> 2)) + 4 * g + (j & 3);
    at = ((s * 4 + t) * 3 * 64 + l) * 8 + j;
}
__device__ __forceinline__ void put_split(__bf16* dst, int at, float w) {
    b2 p0, p1, p2;
    split3(f2{w, 0.0f}, p0, p1, p2);
    dst[at] = p0[0];
    dst[at + 512] = p1[0];
    dst[at + 1024] = p2[0];
}

// thread i of the packing splits weight i of the packed layout (k_leaf_prep's
// packing blocks)
constexpr int kPack1 = 4 * 4 * 64 * 8, kPack2 = 2 * 4 * 64 * 8;
__device__ __forceinline__ void pack_net_at(int i, const float* __restrict__ w1, int F, const float* __restrict__ b1,
                                            const float* __restrict__ lnw, const float* __restrict__ lnb,
                                            const float* __restrict__ w2, const float* __restrict__ b2_,
                                            const float* __restrict__ wv, const float* __restrict__ a1w,
                                            const float* __restrict__ a1b, const float* __restrict__ a2w,
                                            PackedNet* __restrict__ out) {
    int m, k, at;
    if (i < kPack1) {
        perm_index(i, true, m, k, at);
        put_split(reinterpret_cast<__bf16*>(&out->w1), at, k < F ? w1[m * F + k] : 0.0f);
    } else if (i < kPack1 + kPack2) {
        perm_index(i - kPack1, false, m, k, at);
        put_split(reinterpret_cast<__bf16*>(&out->w2), at, w2[m * kE + k]);
    } else if (i < kPack1 + 3 * kPack2) {
        const int j = i - kPack1 - kPack2, half = j / kPack2;
        perm_index(j - half * kPack2, false, m, k, at);
        put_split(reinterpret_cast<__bf16*>(&out->w3[half]), at, a1w[m * 2 * kE + half * kE + k]);
    } else if (i < kPack1 + 3 * kPack2 + kE) {
        const int u = i - kPack1 - 3 * kPack2;
        out->vec[kB1][u] = b1[u];
        out->vec[kLnW][u] = lnw[u];
        out->vec[kLnB][u] = lnb[u];
        out->vec[kB2][u] = b2_[u];
        out->vec[kWv][u] = wv[u];
        out->vec[kWa2][u] = a2w[u];
        out->vec[kBa1][u] = a1b[u];
    }
}
constexpr int kPackThreads = kPack1 + 3 * kPack2 + kE;
constexpr int kPackBlocks = (kPackThreads + 255) / 256;

// The first launch of a fused leaf evaluation, three kinds of 256-thread
// blocks side by side (none waits for another): the successor-row plan of
// up to kPlanLeaves leaves (plan_blocks blocks, hw::rows_plan_block), the
// network in the MLP kernels' layout (kPackBlocks blocks, pack_net_at)
// and, with `stats`, the simulation wave's search counters (one block per
// 1,024 simulations: leaves reached, their legal counts, their virtual-loss
// lengths, rows; integer sums added with device atomics).
__device__ __forceinline__ void leaf_prep(int b, const int32_t* __restrict__ nlegal, int64_t T, int plan_blocks,
    hw::RowsPlan plan, const float* __restrict__ w1, int F,
    const float* __restrict__ b1, const float* __restrict__ lnw,
    const float* __restrict__ lnb, const float* __restrict__ w2,
    const float* __restrict__ b2, const float* __restrict__ wv,
    const float* __restrict__ a1w, const float* __restrict__ a1b,
    const float* __restrict__ a2w, PackedNet* __restrict__ pk,
    const int32_t* __restrict__ leaf_idx,
    const int32_t* __restrict__ vl_lens,
    unsigned long long* __restrict__ stats) {
    if (b < plan_blocks) {
        hw::rows_plan_block(nlegal, T, plan.offsets, plan.total, plan.a2r, plan.mi, b);
        return;
    }
    b -= plan_blocks;
    if (b < kPackBlocks) {
        pack_net_at(b * 256 + (int)threadIdx.x, w1, F, b1, lnw, lnb, w2, b2, wv, a1w, a1b, a2w, pk);
        return;
    }
    b -= kPackBlocks;
    __shared__ unsigned long long part[3][4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    unsigned long long a = 0, n = 0, d = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int64_t i = (int64_t)b * 1024 + k * 256 + tid;
        if (i < T && leaf_idx[i] >= 0) {
            a += 1;
            n += (unsigned long long)(long long)nlegal[i];
            d += (unsigned long long)(long long)vl_lens[i];
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off);
        n += __shfl_xor(n, off);
        d += __shfl_xor(d, off);
    }
    if (lane == 0) {
        part[0][w] = a;
        part[1][w] = n;
        part[2][w] = d;
    }
    __syncthreads();
    if (tid < 3) {
        atomicAdd(&stats[tid], part[tid][0] + part[tid][1] + part[tid][2] + part[tid][3]);
    } else if (tid == 3 && b == 0) {
        atomicAdd(&stats[3], (unsigned long long)T);
    }
}

__global__ __launch_bounds__(256) void k_leaf_prep(const int32_t* __restrict__ nlegal, int64_t T, int plan_blocks,
    hw::RowsPlan plan, const float* __restrict__ w1, int F,
    const float* __restrict__ b1, const float* __restrict__ lnw,
    const float* __restrict__ lnb, const float* __restrict__ w2,
    const float* __restrict__ b2, const float* __restrict__ wv,
    const float* __restrict__ a1w, const float* __restrict__ a1b,
    const float* __restrict__ a2w, PackedNet* __restrict__ pk,
    const int32_t* __restrict__ leaf_idx,
    const int32_t* __restrict__ vl_lens,
    unsigned long long* __restrict__ stats) {
    leaf_prep((int)blockIdx.x, nlegal, T, plan_blocks, plan, w1, F, b1, lnw, lnb, w2, b2, wv, a1w, a1b, a2w, pk, leaf_idx, vl_lens, stats);
}

// sigmoid from the hardware exp2 and reciprocal (v_exp_f32, v_rcp_f32):
// ~1e-6 relative against the correctly rounded form, inside the 1e-5
// tolerance the network's outputs are held to, at a fraction of expf's and
// the IEEE division's instructions (128 sigmoids per successor row)
__device__ __forceinline__ float sigmoidf_(float x) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.44269504088896341f));
}

// sum over the four lanes l, l^16, l^32, l^48 (one row)
__device__ __forceinline__ float row_sum(float v) {
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    return v;
}

// c + a . b over 32 inputs of float32 operands in three parts (see above);
// the smallest products first
__device__ __forceinline__ f4 mfma3(const b8 (&a)[3][64], int lane, const b8 (&b)[3], f4 c) {
    const b8 a0 = a[0][lane], a1 = a[1][lane], a2 = a[2][lane];
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, b[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b[1], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b[0], c, 0, 0, 0);
}
// the same for inputs that are one bf16 part exactly
__device__ __forceinline__ f4 mfma3_whole(const b8 (&a)[3][64], int lane, const b8& b, f4 c) {
    const b8 a0 = a[0][lane], a1 = a[1][lane], a2 = a[2][lane];
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, b, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b, c, 0, 0, 0);
}
// eight inputs x(0) .. x(7) as the three parts of a B operand
template <typename Fn>
__device__ __forceinline__ void split8(Fn x, b8 (&b)[3]) {
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
        b2 p0, p1, p2;
        split3(f2{x(j), x(j + 1)}, p0, p1, p2);
        b[0][j] = p0[0], b[0][j + 1] = p0[1];
        b[1][j] = p1[0], b[1][j + 1] = p1[1];
        b[2][j] = p2[0], b[2][j + 1] = p2[1];
    }
}

__device__ __forceinline__ f4 vec4(const MlpLds& L, int which, int t, int g) {
    return *reinterpret_cast<const f4*>(&L.vec[which][16 * t + 4 * g]);
}

__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Feature f of a record's row (class k), another for each lane; not inlined: the
// MLP kernel, which calls it once in a blue moon, spilled 32 registers
__device__ __attribute__((noinline)) float leaf_record_feature(const hw::UnitRecord* __restrict__ rec, uint32_t k, int f) {
    const int g = f < 96 ? (f >> 2) & 3 : ((f - 96) >> 3) & 3, at = f < 96 ? 4 * (f >> 4) + (f & 3) : 24 + (f & 7);
    float y[32], x = 0.0f;
    hw::unit_slice(rec->u, g, rec->u.dsum[g], k, y);
#pragma unroll
    for (int p = 0; p < 32; p++) x = p == at ? y[p] : x;
    return x;
}

// One row of the network without the split, a wave to it, a unit to each lane
// u, whose inputs are the features x0 = x[u], x1 = x[64 + u].  An infinite
// operand, or one that rounds to a bf16 infinity (past 3.39e38), has no split
// -- its parts are NaN, and so are the row's outputs -- but may have finite
// outputs.
template <bool kRoot>
__device__ __forceinline__ void leaf_plain_row(float x0, float x1, int F, int u, const float* __restrict__ w1,
                                               const float* __restrict__ b1, const float* __restrict__ lnw,
                                               const float* __restrict__ lnb, const float* __restrict__ w2,
                                               const float* __restrict__ b2, const float* __restrict__ wv, float bv,
                                               const float* __restrict__ a1w, const float* __restrict__ a1b,
                                               const float* __restrict__ a2w, float ba2, float* half, float& value,
                                               float& logit) {
    auto product = [&](const float* w, float x, int n, float s) {  // s + w[0] x of lane 0 + ..
#pragma unroll 1
        for (int k = 0; k < n; k++)
            s = __builtin_fmaf(w[k], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), k)), s);
        return s;
    };
    float h = product(w1 + u * F, x0, F < 64 ? F : 64, 0.0f);
    if (F > 64) h = product(w1 + u * F + 64, x1, F - 64, h);
    h = sigmoidf_(h + b1[u]);
    const float d = h - wave_sum_f(h) / (float)kE;
    const float rstd = 1.0f / sqrtf(wave_sum_f(d * d) / (float)kE + 1e-5f);
    const float e = product(w2 + u * kE, d * rstd * lnw[u] + lnb[u], kE, 0.0f) + b2[u];
    value = tanhf(wave_sum_f(e * wv[u]) + bv);
    const float r = product(a1w + u * 2 * kE + (kRoot ? 0 : kE), e, kE, 0.0f);
    if constexpr (kRoot) half[u] = r + a1b[u];
    else logit = wave_sum_f(sigmoidf_(r + half[u]) * a2w[u]) + ba2;
}

// X: [rows][F] features (F even, <= 128, 8-byte aligned rows).
// kRoot: R[rows][64] <- Wr e + b_a1, value[rows] <- tanh(wv . e + bv).
// !kRoot: row -> leaf = succ_leaf[row]; value[rows] <- tanh(wv . e + bv),
//         logit[rows] <- wa2 . sigmoid(Ws e + R[leaf]) + ba2; with `units`
//         and rows enough (leaf_units) the features come from the rows' unit
//         records (X holds the rows marked kRowGeneral only).
template <bool kRoot>
__device__ __forceinline__ void leaf_mlp(MlpLds& L, int64_t block, int64_t blocks, const float* __restrict__ X, int64_t rows, int F,
                                         const int64_t* __restrict__ succ_leaf, int64_t T,
                                         const float* __restrict__ w1, const float* __restrict__ b1,
                                         const float* __restrict__ lnw, const float* __restrict__ lnb,
                                         const float* __restrict__ w2, const float* __restrict__ b2,
                                         const float* __restrict__ wv, float bv, const float* __restrict__ a1w,
                                         const float* __restrict__ a1b, const float* __restrict__ a2w, float ba2,
                                         float* __restrict__ R, float* __restrict__ value,
                                         float* __restrict__ logit, const int64_t* __restrict__ rows_dev,
                                         const PackedNet* __restrict__ pk,
                                         const hw::UnitRecord* __restrict__ units,
                                         const uint32_t* __restrict__ info) {
    if (rows_dev) rows = *rows_dev;  // row count held on the device
    const int64_t ntiles = (rows + 15) >> 4;
    // 16-row tiles dealt over the blocks first (tile = block + grid * (wave +
    // kBlockWaves * round)): a short batch spreads over all CUs, and a block
    // with no tile leaves before filling LDS
    if (block >= ntiles) return;
    if (pk) {  // the packed layout: straight 16-byte copies, every load issued before the first store
        constexpr int kT = 64 * kBlockWaves, k12 = (sizeof(L.w1) + sizeof(L.w2)) / 16, k3 = sizeof(L.w3) / 16;
        constexpr int n12 = (k12 + kT - 1) / kT, n3 = (k3 + kT - 1) / kT;
        static_assert(7 * kE / 4 <= kT && sizeof(L.w1) % 16 == 0, "16-byte copies");
        const int tid = threadIdx.x;
        const f4* src = reinterpret_cast<const f4*>(&pk->w1);
        const f4* s3 = reinterpret_cast<const f4*>(&pk->w3[kRoot ? 0 : 1]);
        f4 c12[n12], c3[n3], cv = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < n12; k++)
            if (tid + k * kT < k12) c12[k] = src[tid + k * kT];  // w1, w2
#pragma unroll
        for (int k = 0; k < n3; k++)
            if (tid + k * kT < k3) c3[k] = s3[tid + k * kT];
        if (tid < 7 * kE / 4) cv = reinterpret_cast<const f4*>(&pk->vec[0][0])[tid];
        f4* dst = reinterpret_cast<f4*>(&L.w1);
        f4* d3 = reinterpret_cast<f4*>(&L.w3);
#pragma unroll
        for (int k = 0; k < n12; k++)
            if (tid + k * kT < k12) dst[tid + k * kT] = c12[k];
#pragma unroll
        for (int k = 0; k < n3; k++)
            if (tid + k * kT < k3) d3[tid + k * kT] = c3[k];
        if (tid < 7 * kE / 4) reinterpret_cast<f4*>(&L.vec[0][0])[tid] = cv;
    } else {  // weights gathered, permuted and split into LDS (perm_index), every load issued before the first split
        constexpr int kT = 64 * kBlockWaves, n1 = kPack1 / kT, n2 = kPack2 / kT;
        static_assert(kPack1 % kT == 0 && kPack2 % kT == 0, "whole rounds");
        float c1[n1], c2[n2], c3[n2];
        int m, k, at;
#pragma unroll
        for (int q = 0; q < n1; q++) {
            perm_index(threadIdx.x + q * kT, true, m, k, at);
            c1[q] = k < F ? w1[m * F + k] : 0.0f;
        }
#pragma unroll
        for (int q = 0; q < n2; q++) {
            perm_index(threadIdx.x + q * kT, false, m, k, at);
            c2[q] = w2[m * kE + k];
            c3[q] = a1w[m * 2 * kE + (kRoot ? 0 : kE) + k];
        }
#pragma unroll
        for (int q = 0; q < n1; q++) {
            perm_index(threadIdx.x + q * kT, true, m, k, at);
            put_split(reinterpret_cast<__bf16*>(&L.w1), at, c1[q]);
        }
#pragma unroll
        for (int q = 0; q < n2; q++) {
            perm_index(threadIdx.x + q * kT, false, m, k, at);
            put_split(reinterpret_cast<__bf16*>(&L.w2), at, c2[q]);
            put_split(reinterpret_cast<__bf16*>(&L.w3), at, c3[q]);
        }
        if (threadIdx.x < kE) {
            const int u = threadIdx.x;
            L.vec[kB1][u] = b1[u];
            L.vec[kLnW][u] = lnw[u];
            L.vec[kLnB][u] = lnb[u];
            L.vec[kB2][u] = b2[u];
            L.vec[kWv][u] = wv[u];
            L.vec[kWa2][u] = a2w[u];
            L.vec[kBa1][u] = a1b[u];
        }
    }
    __syncthreads();

    const int lane = threadIdx.x & 63, g = lane >> 4;
    bool odd = false;  // a row of the wave came out NaN
    for (int64_t tile = block + blocks * (threadIdx.x >> 6); tile < ntiles; tile += blocks * kBlockWaves) {
        // the weights are re-read from LDS in every tile: hoisted out of the
        // loop they would take hundreds of registers and leave one wave per SIMD
        __asm__ volatile("" ::: "memory");
        const int64_t row = tile * 16 + (lane & 15);
        const bool ok = row < rows;
        // successor rows: the leaf's root half of the action tower, fetched once the
        // features' registers are free (before them 14 registers spill)
        f4 rh[4];
        const float* half = nullptr;
        if constexpr (!kRoot) {
            int64_t leaf = ok ? succ_leaf[row] : 0;
            leaf = leaf < 0 ? 0 : (leaf >= T ? T - 1 : leaf);
            half = R + leaf * kE + 4 * g;
        }
        // the lane's 32 features, x[8 s + j] = feature_of(s, g, j)
        float x[32];
        const float* xr = X + (ok ? row : 0) * F;
        auto load_row = [&]() {
#pragma unroll
            for (int p = 0; p < 16; p++) {
                const int s = p >> 2, j = 2 * (p & 3);
                const int at = s < 3 ? 16 * feature_section(s, j) + (j & 3) + 4 * g : 96 + j + 8 * g;
                float2 v = make_float2(0.0f, 0.0f);
                if (ok && at < F) v = *reinterpret_cast<const float2*>(xr + at);
                x[2 * p] = v.x;
                x[2 * p + 1] = v.y;
            }
        };
        f4 acc[4];  // every layer's sums start from its bias
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t] = vec4(L, kB1, t, g);
        const bool packed = !kRoot && units && hw::leaf_units(rows, T);
        if (packed) {
            const uint32_t w = ok ? info[row] : 0u;
            if (w & hw::kRowGeneral) {
                load_row();
            } else {
                const hw::Unit& U = units[(ok ? row : 0) - (int64_t)(w & 255u)].u;
                hw::Unit V;  // the fields a slice reads
                V.cnt = U.cnt, V.hand = U.hand, V.near = U.near, V.pin = U.pin, V.dn = U.dn, V.bn = U.bn;
                V.m = U.m, V.lift = U.lift, V.t = U.t;
                float y[32];
                hw::unit_slice(V, g, U.dsum[g], (w >> 8) & 15u, y);
#pragma unroll
                for (int p = 0; p < 32; p++)
                    x[p] = p < 24 ? y[4 * feature_section(p >> 3, p & 7) + (p & 3)] : y[p];
            }
#pragma unroll
            for (int s = 0; s < 4; s++) {
                b8 b[3];
                split8([&](int j) { return x[8 * s + j]; }, b);
#pragma unroll
                for (int t = 0; t < 4; t++)
                    acc[t] = s & 1 ? mfma3(L.w1[s][t], lane, b, acc[t]) : mfma3_whole(L.w1[s][t], lane, b[0], acc[t]);
            }
        } else {
            load_row();
#pragma unroll
            for (int s = 0; s < 4; s++) {
                b8 b[3];
                split8([&](int j) { return x[8 * s + j]; }, b);
#pragma unroll
                for (int t = 0; t < 4; t++) acc[t] = mfma3(L.w1[s][t], lane, b, acc[t]);
            }
        }
        if constexpr (!kRoot) {
#pragma unroll
            for (int t = 0; t < 4; t++) rh[t] = *reinterpret_cast<const f4*>(half + 16 * t);
        }
        // sigmoid + LayerNorm over the row's 64 units
        float sum = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                acc[t][i] = sigmoidf_(acc[t][i]);
                sum += acc[t][i];
            }
        const float mean = row_sum(sum) / (float)kE;
        float sq = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                acc[t][i] -= mean;
                sq = __builtin_fmaf(acc[t][i], acc[t][i], sq);
            }
        const float rstd = __builtin_amdgcn_rsqf(row_sum(sq) / (float)kE + 1e-5f);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const f4 w = vec4(L, kLnW, t, g), b = vec4(L, kLnB, t, g);
#pragma unroll
            for (int i = 0; i < 4; i++) acc[t][i] = __builtin_fmaf(acc[t][i] * rstd, w[i], b[i]);
        }
        // fc2 -> embedding
        f4 e[4];
#pragma unroll
        for (int t = 0; t < 4; t++) e[t] = vec4(L, kB2, t, g);
#pragma unroll
        for (int s = 0; s < 2; s++) {
            b8 b[3];
            split8([&](int j) { return acc[2 * s + (j >> 2)][j & 3]; }, b);
#pragma unroll
            for (int t = 0; t < 4; t++) e[t] = mfma3(L.w2[s][t], lane, b, e[t]);
        }
        float v = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const f4 w = vec4(L, kWv, t, g);
#pragma unroll
            for (int i = 0; i < 4; i++) v = __builtin_fmaf(e[t][i], w[i], v);
        }
        v = tanhf(row_sum(v) + bv);
        // action tower, first layer (root or successor half)
        f4 h[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if constexpr (kRoot) h[t] = vec4(L, kBa1, t, g);
            else h[t] = rh[t];
        }
#pragma unroll
        for (int s = 0; s < 2; s++) {
            b8 b[3];
            split8([&](int j) { return e[2 * s + (j >> 2)][j & 3]; }, b);
#pragma unroll
            for (int t = 0; t < 4; t++) h[t] = mfma3(L.w3[s][t], lane, b, h[t]);
        }
        if constexpr (kRoot) {
            if (ok) {
#pragma unroll
                for (int t = 0; t < 4; t++)
                    *reinterpret_cast<f4*>(R + row * kE + 16 * t + 4 * g) = h[t];
                if (g == 0) value[row] = v;
            }
            float all = v;
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) all += h[t][i];
            odd |= __ballot(ok && all != all) != 0;
        } else {
            float a = 0.0f;
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const f4 w = vec4(L, kWa2, t, g);
#pragma unroll
                for (int i = 0; i < 4; i++) a = __builtin_fmaf(sigmoidf_(h[t][i]), w[i], a);
            }
            a = row_sum(a) + ba2;
            if (ok && g == 0) {
                value[row] = v;
                logit[row] = a;
            }
            odd |= __ballot(ok && (v != v || a != a)) != 0;
        }
    }
    if (!odd) return;
    __threadfence_block();  // the outputs, read by other lanes
    const int u = hw_opaque(lane);
    // a NaN in the encoder itself is in every output of every row
    bool lost = b1[u] != b1[u] || lnw[u] != lnw[u] || lnb[u] != lnb[u] || b2[u] != b2[u];
#pragma unroll 1
    for (int k = 0; k < F; k++) lost |= w1[u * F + k] != w1[u * F + k];
#pragma unroll 1
    for (int k = 0; k < kE; k++) lost |= w2[u * kE + k] != w2[u * kE + k];
    if (__ballot(lost)) return;
    for (int64_t tile = block + blocks * (threadIdx.x >> 6); tile < ntiles; tile += blocks * kBlockWaves) {
        for (int64_t row = tile * 16; row < rows && row < tile * 16 + 16; row++) {
            float v = value[row], a = kRoot ? R[row * kE + u] : logit[row];
            if (!__ballot(v != v || a != a)) continue;
            const hw::UnitRecord* rec = nullptr;
            uint32_t k = 0;
            if constexpr (!kRoot) {
                if (units && hw::leaf_units(rows, T) && !(info[row] & hw::kRowGeneral)) {
                    rec = units + (row - (int64_t)(info[row] & 255u));
                    k = (info[row] >> 8) & 15u;
                }
            }
            const float x0 = rec ? leaf_record_feature(rec, k, u) : u < F ? X[row * F + u] : 0.0f;
            const float x1 = rec ? leaf_record_feature(rec, k, 64 + u) : 64 + u < F ? X[row * F + 64 + u] : 0.0f;
            if constexpr (kRoot) {
                leaf_plain_row<true>(x0, x1, F, u, w1, b1, lnw, lnb, w2, b2, wv, bv, a1w, a1b, a2w, ba2, R + row * kE, v, a);
            } else {
                int64_t leaf = succ_leaf[row];
                leaf = leaf < 0 ? 0 : (leaf >= T ? T - 1 : leaf);
                leaf_plain_row<false>(x0, x1, F, u, w1, b1, lnw, lnb, w2, b2, wv, bv, a1w, a1b, a2w, ba2, R + leaf * kE, v, a);
                if (u == 0) logit[row] = a;
            }
            if (u == 0) value[row] = v;
        }
    }
}

template <bool kRoot>
__global__ __launch_bounds__(64 * kBlockWaves) void k_leaf_mlp(const float* __restrict__ X, int64_t rows, int F,
                                                  const int64_t* __restrict__ succ_leaf, int64_t T,
                                                  const float* __restrict__ w1, const float* __restrict__ b1,
                                                  const float* __restrict__ lnw, const float* __restrict__ lnb,
                                                  const float* __restrict__ w2, const float* __restrict__ b2,
                                                  const float* __restrict__ wv, float bv, const float* __restrict__ a1w,
                                                  const float* __restrict__ a1b, const float* __restrict__ a2w, float ba2,
                                                  float* __restrict__ R, float* __restrict__ value,
                                                  float* __restrict__ logit, const int64_t* __restrict__ rows_dev,
                                                  const PackedNet* __restrict__ pk,
                                                  const hw::UnitRecord* __restrict__ units = nullptr,
                                                  const uint32_t* __restrict__ info = nullptr) {
    __shared__ MlpLds L;
    leaf_mlp<kRoot>(L, blockIdx.x, gridDim.x, X, rows, F, succ_leaf, T, w1, b1, lnw, lnb, w2, b2, wv, bv, a1w, a1b, a2w, ba2, R, value, logit, rows_dev, pk, units, info);
}

// The first launch of a short evaluation: k_leaf_prep's blocks (their first 256
// threads) beside the root rows' tiles, whose blocks take the weights from the
// network itself instead of waiting for the packed ones.  At kFirstLeaves leaves
// every block has a CU of its own: 128 tile blocks, 81 of packing, the plan's and
// the counters' (219 of 256; sizes between this one and where they no longer do,
// about 2,580 leaves, were not tried).  Base-game leaf evaluation: 2,048 leaves 83
// us, 2,100 (the leaf rows' network in a launch of its own) 100 us.
constexpr int64_t kFirstLeaves = 2048;
__global__ __launch_bounds__(64 * kBlockWaves) void k_leaf_first(
    int root_blocks, const float* __restrict__ X, int64_t T, int F, hw::RowsPlan plan, int plan_blocks,
    const int32_t* __restrict__ nlegal, const float* __restrict__ w1, const float* __restrict__ b1,
    const float* __restrict__ lnw, const float* __restrict__ lnb, const float* __restrict__ w2,
    const float* __restrict__ b2, const float* __restrict__ wv, float bv, const float* __restrict__ a1w,
    const float* __restrict__ a1b, const float* __restrict__ a2w, float ba2, PackedNet* __restrict__ pk,
    float* __restrict__ R, float* __restrict__ value, const int32_t* __restrict__ leaf_idx,
    const int32_t* __restrict__ vl_lens, unsigned long long* __restrict__ stats) {
    __shared__ MlpLds L;
    if ((int)blockIdx.x < root_blocks) {
        leaf_mlp<true>(L, blockIdx.x, root_blocks, X, T, F, nullptr, T, w1, b1, lnw, lnb, w2, b2, wv, bv, a1w, a1b, a2w,
                       ba2, R, value, nullptr, nullptr, nullptr, nullptr, nullptr);
        return;
    }
    if (threadIdx.x >= 256) return;  // whole waves: the barriers below count the others
    leaf_prep((int)blockIdx.x - root_blocks, nlegal, T, plan_blocks, plan, w1, F, b1, lnw, lnb, w2, b2, wv, a1w, a1b,
              a2w, pk, leaf_idx, vl_lens, stats);
}

__device__ __forceinline__ float wave_max_f(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// One wave per leaf t: softmax of logit[offsets[t] .. + n) into priors[t],
// child_q[t][i] = -child value; zero beyond n.
__global__ __launch_bounds__(256) void k_leaf_softmax(const float* __restrict__ logit, const float* __restrict__ cval,
                                                      const int64_t* __restrict__ offsets,
                                                      const int32_t* __restrict__ nlegal, int64_t T,
                                                      float* __restrict__ priors, float* __restrict__ child_q,
                                                      int dense) {
    const int lane = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= T) return;
    int n = nlegal[t];
    n = n < 0 ? 0 : (n > kSlots ? kSlots : n);
    const int64_t base = offsets[t];
    float lg[4], cv[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = lane + 64 * k;
        lg[k] = i < n ? logit[base + i] : -INFINITY;
        cv[k] = i < n ? cval[base + i] : 0.0f;
    }
    const float m = wave_max_f(fmaxf(fmaxf(lg[0], lg[1]), fmaxf(lg[2], lg[3])));
    float ex[4], s = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        ex[k] = lane + 64 * k < n ? expf(lg[k] - m) : 0.0f;
        s += ex[k];
    }
    s = wave_sum_f(s);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = lane + 64 * k;
        if (i < n || dense) {  // `dense`: the rows' tails zeroed, else left as they are
            priors[t * kSlots + i] = i < n ? ex[k] / s : 0.0f;
            child_q[t * kSlots + i] = i < n ? -cv[k] : 0.0f;
        }
    }
}

inline int grid_for(int64_t n, int per) { return (int)((n + per - 1) / per); }
// one block per 16-row tile up to kMaxBlocks (the kernels deal tiles over the
// blocks first, so a short batch runs one tile per CU)
inline int mlp_blocks(int64_t rows) {
    const int64_t b = (rows + 15) / 16;
    return (int)(b < kMaxBlocks ? b : kMaxBlocks);
}

}  // namespace

extern "C" {

int hg_fnn_leaf_eval(const float* features, int64_t T, int64_t N, int F, const int64_t* offsets,
                     const int32_t* num_legal, const int64_t* succ_leaf, const float* fc1_w, const float* fc1_b,
                     const float* ln_w, const float* ln_b, const float* fc2_w, const float* fc2_b,
                     const float* value_w, float value_b, const float* action1_w, const float* action1_b,
                     const float* action2_w, float action2_b, float* workspace, float* priors, float* root_values,
                     float* child_q, void* stream) {
    if (T < 0 || N < 0 || F <= 0 || F > kFMax || (F & 1)) return (int)hipErrorInvalidValue;
    if (((uintptr_t)features & 7) || ((uintptr_t)workspace & 15)) return (int)hipErrorInvalidValue;
    if (T == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    float* R = workspace;           // [T][64]
    float* logit = R + T * kE;      // [N]
    float* cval = logit + N;        // [N]
    hipLaunchKernelGGL(k_leaf_mlp<true>, dim3(mlp_blocks(T)), dim3(64 * kBlockWaves), 0, st, features, T, F,
                       nullptr, T, fc1_w, fc1_b, ln_w, ln_b, fc2_w, fc2_b, value_w, value_b, action1_w, action1_b,
                       action2_w, action2_b, R, root_values, nullptr, nullptr, nullptr);
    if (N > 0)
        hipLaunchKernelGGL(k_leaf_mlp<false>, dim3(mlp_blocks(N)), dim3(64 * kBlockWaves), 0, st, features + T * F,
                           N, F, succ_leaf, T, fc1_w, fc1_b, ln_w, ln_b, fc2_w, fc2_b, value_w, value_b, action1_w,
                           action1_b, action2_w, action2_b, R, cval, logit, nullptr, nullptr);
    hipLaunchKernelGGL(k_leaf_softmax, dim3(grid_for(T, 4)), dim3(256), 0, st, logit, cval, offsets, num_legal, T,
                       priors, child_q, 1);
    return (int)hipGetLastError();
}

int64_t hg_fnn_leaf_eval_lists_workspace(int64_t T, int F) {
    if (T <= 0) return 0;
    const int64_t cap = T * kSlots;
    int64_t b = hg_successor_rows_workspace(T);           // offsets, total, row map
    b = (b + 255) & ~(int64_t)255;
    b += cap * F * (int64_t)sizeof(float);                // successor features
    b = (b + 255) & ~(int64_t)255;
    b += (T * kE + 2 * cap) * (int64_t)sizeof(float);     // root half of the action tower, logits, child values
    b = (b + 255) & ~(int64_t)255;
    b += (int64_t)sizeof(PackedNet);                      // the network in the kernels' LDS order
    b = (b + 255) & ~(int64_t)255;
    b += cap * (int64_t)(sizeof(hw::UnitRecord) + sizeof(uint32_t));  // unit records, a word per row
    return b;
}

int hg_fnn_leaf_eval_lists(const uint8_t* leaf_states, const uint8_t* legal_moves, const int32_t* num_legal,
                           const float* root_features, int64_t T, int F, const float* fc1_w, const float* fc1_b,
                           const float* ln_w, const float* ln_b, const float* fc2_w, const float* fc2_b,
                           const float* value_w, float value_b, const float* action1_w, const float* action1_b,
                           const float* action2_w, float action2_b, void* workspace, float* priors,
                           float* root_values, float* child_q, void* stream) {
    return hw::leaf_eval_lists(leaf_states, legal_moves, num_legal, root_features, T, F, fc1_w, fc1_b, ln_w, ln_b,
                               fc2_w, fc2_b, value_w, value_b, action1_w, action1_b, action2_w, action2_b, workspace,
                               priors, root_values, child_q, nullptr, nullptr, nullptr, (hipStream_t)stream);
}

}  // extern "C"

namespace hw {

int leaf_eval_lists(const uint8_t* leaf_states, const uint8_t* legal_moves, const int32_t* num_legal,
                    const float* root_features, int64_t T, int F, const float* fc1_w, const float* fc1_b,
                    const float* ln_w, const float* ln_b, const float* fc2_w, const float* fc2_b,
                    const float* value_w, float value_b, const float* action1_w, const float* action1_b,
                    const float* action2_w, float action2_b, void* workspace, float* priors, float* root_values,
                    float* child_q, const int32_t* leaf_idx, const int32_t* vl_lens, int64_t* stats,
                    hipStream_t st, bool dense) {
    if (T < 0 || F <= 0 || F > kFMax || (F & 1)) return (int)hipErrorInvalidValue;
    if (((uintptr_t)root_features & 7) || ((uintptr_t)workspace & 255)) return (int)hipErrorInvalidValue;
    if (F != 122) return (int)hipErrorInvalidValue;  // the successor rows are the engine's 122 features
    if (stats && (!leaf_idx || !vl_lens)) return (int)hipErrorInvalidValue;
    if (T == 0) return 0;
    const int64_t cap = T * kSlots;
    uint8_t* base = reinterpret_cast<uint8_t*>(workspace);
    int64_t off = hg_successor_rows_workspace(T);
    const RowsPlan plan = rows_plan_of(workspace, T);
    off = (off + 255) & ~(int64_t)255;
    float* X = reinterpret_cast<float*>(base + off);
    off += cap * F * (int64_t)sizeof(float);
    off = (off + 255) & ~(int64_t)255;
    float* R = reinterpret_cast<float*>(base + off);
    float* logit = R + T * kE;
    float* cval = logit + cap;
    off += (T * kE + 2 * cap) * (int64_t)sizeof(float);
    off = (off + 255) & ~(int64_t)255;
    PackedNet* pk = reinterpret_cast<PackedNet*>(base + off);
    off = (off + (int64_t)sizeof(PackedNet) + 255) & ~(int64_t)255;
    UnitRecord* units = reinterpret_cast<UnitRecord*>(base + off);
    uint32_t* info = reinterpret_cast<uint32_t*>(units + cap);
    // plan, network layout and counters in one launch (the plan of a batch
    // over kPlanLeaves leaves takes its own two launches first)
    int plan_blocks = 0;
    if (T <= kPlanLeaves) {
        plan_blocks = (int)((T + 255) / 256);
    } else {
        int e = successor_rows_plan_large(num_legal, T, workspace, st);
        if (e) return e;
    }
    const int stat_blocks = stats ? (int)((T + 1023) / 1024) : 0;
    const int prep_blocks = plan_blocks + kPackBlocks + stat_blocks;
    unsigned long long* counters = reinterpret_cast<unsigned long long*>(stats);
    const bool first = T <= kFirstLeaves;
    if (first) {
        const int root_blocks = mlp_blocks(T);
        hipLaunchKernelGGL(k_leaf_first, dim3((unsigned)(root_blocks + prep_blocks)), dim3(64 * kBlockWaves), 0, st,
                           root_blocks, root_features, T, F, plan, plan_blocks, num_legal, fc1_w, fc1_b, ln_w, ln_b,
                           fc2_w, fc2_b, value_w, value_b, action1_w, action1_b, action2_w, action2_b, pk, R,
                           root_values, leaf_idx, vl_lens, counters);
    } else {
        hipLaunchKernelGGL(k_leaf_prep, dim3((unsigned)prep_blocks), dim3(256), 0, st, num_legal, T, plan_blocks, plan,
                           fc1_w, F, fc1_b, ln_w, ln_b, fc2_w, fc2_b, value_w, action1_w, action1_b, action2_w, pk,
                           leaf_idx, vl_lens, counters);
    }
    int e = successor_rows_after_plan(leaf_states, legal_moves, T, workspace, X, st, units, info);
    if (e) return e;
    if (!first)
        hipLaunchKernelGGL(k_leaf_mlp<true>, dim3(mlp_blocks(T)), dim3(64 * kBlockWaves), 0, st, root_features, T, F,
                           nullptr, T, fc1_w, fc1_b, ln_w, ln_b, fc2_w, fc2_b, value_w, value_b, action1_w, action1_b,
                           action2_w, action2_b, R, root_values, nullptr, nullptr, pk);
    hipLaunchKernelGGL(k_leaf_mlp<false>, dim3(mlp_blocks(cap)), dim3(64 * kBlockWaves), 0, st, X, cap, F,
                       plan.a2r, T, fc1_w, fc1_b, ln_w, ln_b, fc2_w, fc2_b, value_w, value_b, action1_w, action1_b,
                       action2_w, action2_b, R, cval, logit, plan.total, pk, units, info);
    hipLaunchKernelGGL(k_leaf_softmax, dim3(grid_for(T, 4)), dim3(256), 0, st, logit, cval, plan.offsets,
                       num_legal, T, priors, child_q, dense ? 1 : 0);
    return (int)hipGetLastError();
}

}  // namespace hw
