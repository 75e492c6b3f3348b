// The reference renderer's Aggregator (epcq/epcq.py:406-507) for inference on
// gfx950: the point MLP over every (sample, neighbour) pair, the inverse-
// distance aggregation of its alpha and features per sample, and the colour
// MLP, on the bf16 matrix cores with fp32 accumulation.
//
// Per pair (m, k) with a valid neighbour (the reference's, per chunk of rows):
//   x1 = [f, PE(f, 3), PE([p - s, p*p - s*s], 5)]             284 = 7F + 60, F = 32
//   h2 = lrelu(W2 lrelu(W1 x1 + b1) + b2)                     block1
//   x3 = [h2, rgb, dir - d, dir . d]                          263
//   h4 = lrelu(W4 lrelu(W3 x3 + b3) + b4)                     block3
//   a  = softplus(wa . h4 + ba - 1)                           alpha_branch, alpha_act(alphas - 1)
// with f the point's feature, p its position, s the sample, d the ray
// direction, PE(x, n) = [sin(x_i 2^j), cos(x_i 2^j)] in (i, j) order
// (positional_encoding, epcq.py:389-404), lrelu slope 0.01, softplus with
// threshold 20.  Per sample m, with w_k = (1/(|p_k - s| + 1e-6)) v_k /
// (sum_k (1/(|p_k - s| + 1e-6)) v_k + 1e-6) (calculate_weight, :434-437):
//   alpha = sum_k w_k a_k                                     [M]
//   xc    = [sum_k w_k h4_k, PE(d, 4)]                        280
//   rgb   = sigmoid(C4 lrelu(C3 lrelu(C2 lrelu(C1 xc + c1) + c2) + c3) + c4) * 1.002 - 0.001
//
// Layout.  Each layer is computed transposed, Y^T = W X^T, with the weights as
// the left operand of v_mfma_f32_32x32x16_bf16: a lane then owns one row of the
// batch in every layer (its column of the result), and the accumulators of one
// layer become the right operands of the next by a conversion to bf16 and a
// swap of lane halves (v_permlane32_swap), so activations never leave the
// registers.  A block is four waves of 32 rows; the weights stream from L2
// through LDS in pieces of 64 outputs, copied by the load unit itself
// (global_load_lds) into one buffer while the waves multiply from the other,
// with one barrier per piece.  Two blocks fit on a CU and drift apart, so one's
// encodings, epilogues and reductions run under the other's matrix products.
//
// Pairs are rows: a block takes 128 / K whole samples, rows in order, whichever
// wave they fall to (K = 5 fills 125 of 128 rows).  At the end the rows' last
// activations go to LDS and each half of a wave reduces one sample after
// another into the workspace (bf16, 256 wide); a second kernel runs the colour
// MLP, a row per sample.  Nothing is accumulated across waves, so results do
// not depend on scheduling.
//
// What bounds it: the matrix cores, at the clock that they leave (about 1.7 of
// 2.4 GHz), for two thirds of a block's time, then the encodings and
// reductions.  Measured, both kernels, against weight chunks of 16 inputs that
// passed through registers, activations in LDS and rows padded to a power of
// two: 1.28M samples of 8 neighbours 7.9 -> 5.9 ms, 100k of 9 1.19 -> 0.58,
// 100k of 5 0.68 -> 0.37, 20k of 8 0.20 -> 0.14.
#include <math.h>

#include <type_traits>

#include "epcq_common.h"

namespace epcq {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWave = 64;
constexpr int kWaves = 4;
constexpr int kBlock = kWave * kWaves;
constexpr int kWaveRows = 32;
constexpr int kRows = kWaves * kWaveRows;  // rows of a block
constexpr int kFeat = 32;               // F: block1 takes 7F + 60 = 284 inputs
constexpr int kX1 = 288, kH = 256, kX3 = 272, kXc = 288, kC = 128;
constexpr int kPieceTiles = 2;          // tiles of 32 outputs in a weight piece
constexpr int kPiece = 32 * kPieceTiles;
constexpr int kPieceBytes = kPiece * kX1 * 2;  // the longest rows
constexpr int kLdsStride = kH + 8;      // bf16 per row of last activations (8: rows start on different banks)
static_assert(2 * kWaveRows * kLdsStride * 2 <= kPieceBytes, "a buffer holds two waves' rows");

// Round to nearest even (the hardware conversion, v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint16_t to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// Two floats rounded to bf16 by one packed conversion, lo in the low half.
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// sin and cos of x for the positional encodings, whose results are rounded
// to bf16: one range reduction to [-1/2, 1/2] revolution and the hardware
// sine and cosine.  The rounding of x / 2 pi bounds the phase error by
// |x| 2^-24 (6e-5 rad at |x| = 1024), far below the bf16 step of 2^-8 near
// 1; the library's sincosf beyond.
// CHECKED false: the caller has established |x| < 1024 (no branch here).
template <bool CHECKED = true>
__device__ __forceinline__ void pe_sincos(float x, float& s, float& c) {
    if (!CHECKED || fabsf(x) < 1024.0f) {
        float r = x * 0.15915494309189535f;
        r = r - rintf(r);
        s = __builtin_amdgcn_sinf(r);
        c = __builtin_amdgcn_cosf(r);
    } else {
        sincosf(x, &s, &c);
    }
}

// sin and cos of 2x from those of x (double-angle formulas).  Each step at
// most quadruples the absolute error of its inputs and adds a rounding; the
// encodings take at most two steps from a pe_sincos value, which keeps them
// within 16 times its error, far below the bf16 step they are rounded to.
__device__ __forceinline__ void pe_double(float s, float c, float& s2, float& c2) {
    s2 = 2.0f * s * c;
    c2 = c * c - s * s;
}

__device__ __forceinline__ float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// v for v > 0, else 0.01 v, as the larger of the two: one multiply and one
// v_maximum3_f32 (fmaxf of a matrix-core result adds a NaN-quieting max of its
// own).  Equal to the compare-and-select form for every finite v, +-0 and
// +-inf (a NaN stays a NaN).
__device__ __forceinline__ float lrelu(float v) { return __builtin_elementwise_maximum(v, 0.01f * v); }

// torch.nn.Softplus(beta=1, threshold=20)
__device__ __forceinline__ float softplus(float v) { return v > 20.0f ? v : log1pf(expf(v)); }

__device__ __forceinline__ bf16x8 load8(const uint16_t* p) {
    bf16x8 v;
    __builtin_memcpy(&v, p, sizeof(v));
    return v;
}

// The eights (a0, a1 | a2, a3) of which each lane half holds half (two packed
// registers each): half 0 gets the whole first eight, half 1 the second.
__device__ __forceinline__ bf16x8 swap_halves(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1) {
    const auto s0 = __builtin_amdgcn_permlane32_swap(a0, b0, false, false);
    const auto s1 = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
    return __builtin_bit_cast(bf16x8, make_uint4(s0[0], s1[0], s0[1], s1[1]));
}

// Copies outputs [n0, n0 + 64) of the weights W [N, 16 KS] to `buf`; complete
// after the next __syncthreads().  Each wave takes 16 rows, 64 bytes of them at
// a time (two steps of 16 inputs; of an odd last one, what follows it in memory
// or zeros, which nobody reads).  The load unit writes a lane's 16 bytes at
// slot `lane` of the instruction's 1024; the lane picks its piece of the row by
// a rotation (an exclusive or with half its row), so that the eight lanes of a
// read cycle, eight rows at one input step, find theirs on different banks.
// ALIGNED: W is 16-byte aligned; else the copies go through registers.
template <int KS, int N, bool ALIGNED>
struct Fetch {
    static constexpr int kSteps = (KS + 1) / 2;
    static constexpr int K = 16 * KS;
    const uint16_t* W;
    int at;      // the lane's first input
    uint4* dst;  // the wave's part of the buffer

    __device__ __forceinline__ Fetch(const uint16_t* w, int n0, uint4* buf) : W(w) {
        const int lane = threadIdx.x % kWave;
        const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
        at = (n0 + wave * 16 + lane / 4) * K + ((lane ^ (lane / 8)) & 3) * 8;
        dst = buf + wave * kSteps * kWave;
    }
    // the 64 bytes of steps 2 i and 2 i + 1
    __device__ __forceinline__ void step(int i) const {
        if (i >= kSteps) return;
        if (ALIGNED) {
            // a buffer load: one that goes through a flat address would make
            // every LDS read wait for all others
            const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(W), 0, N * K * 2, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(dst + i * kWave), 16,
                                                     2 * at, 64 * i, 0, 0);
        } else {
            uint4 v = make_uint4(0, 0, 0, 0);
            if (at + 32 * i < N * K) __builtin_memcpy(&v, W + at + 32 * i, sizeof(v));
            dst[i * kWave + threadIdx.x % kWave] = v;
        }
    }
    __device__ __forceinline__ void all() const {
#pragma unroll
        for (int i = 0; i < kSteps; ++i) step(i);
    }
};

struct NoFetch {
    static constexpr int kSteps = 0;
    __device__ __forceinline__ NoFetch(const uint16_t*, int, uint4*) {}
    __device__ __forceinline__ void step(int) const {}
};

// The lane's weight operand of tile t at step ks.
template <int KS>
__device__ __forceinline__ bf16x8 weight_operand(const uint4* w, int t, int ks) {
    const int lane = threadIdx.x % kWave;
    const int row = lane & 31;
    const int slot = (row & 15) * 4 + ((((ks & 1) << 1) + (lane >> 5)) ^ ((row >> 1) & 3));
    return __builtin_bit_cast(bf16x8, w[(row >> 4) * ((KS + 1) / 2 * kWave) + slot + (2 * t * ((KS + 1) / 2) + ks / 2) * kWave]);
}

// The accumulators of a piece of 64 outputs.
typedef f32x16 PieceAcc[kPieceTiles];

// Activation and conversion of a quarter (16 outputs) of a finished piece: an
// operand of the next layer.
__device__ __forceinline__ bf16x8 finish_quarter(const PieceAcc& acc, int c) {
    uint32_t p[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
        p[q] = pack_bf16(lrelu(acc[c / 2][8 * (c % 2) + 2 * q]), lrelu(acc[c / 2][8 * (c % 2) + 2 * q + 1]));
    return swap_halves(p[0], p[1], p[2], p[3]);
}
__device__ __forceinline__ void finish_piece(const PieceAcc& acc, bf16x8* y) {
#pragma unroll
    for (int c = 0; c < 4; ++c) y[c] = finish_quarter(acc, c);
}

// The biases of 64 outputs, where the accumulators start.
__device__ __forceinline__ void start_piece(PieceAcc& acc, const float* s_bias) {
    const int half = threadIdx.x % kWave >> 5;
#pragma unroll
    for (int t = 0; t < kPieceTiles; ++t) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 b = *reinterpret_cast<const float4*>(s_bias + 32 * t + 8 * q + 4 * half);
            acc[t][4 * q] = b.x;
            acc[t][4 * q + 1] = b.y;
            acc[t][4 * q + 2] = b.z;
            acc[t][4 * q + 3] = b.w;
        }
    }
}

// 64 outputs of a layer over the wave's rows, from the weight piece in `w`,
// onto the biases in acc; meanwhile the next piece is fetched, the piece
// before (`other`, if PREV) is finished into yprev, and its accumulators start
// at the next piece's biases (if NEXT).  The 32x32x16 operands: lane l
// holds A[l % 32][8 (l / 32) + v] and B[8 (l / 32) + v][l % 32], v < 8;
// accumulator register r of lane l is D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
// So the lane of row j holds outputs 4 h .. 4 h + 3 of every eight (h = l / 32),
// and a swap of halves between the eights 2 i and 2 i + 1 gives each half all of
// its eight.
//
// Two input steps (four products, 128 cycles) at a time: their weights were
// read from LDS during the two before, and between the products, which leave
// seven in eight issue slots free, go the reads for the next two, a step of the
// fetch and a quarter of the piece before.
template <int KS, bool PREV, bool NEXT, typename F>
__device__ __forceinline__ void piece(const bf16x8* x, PieceAcc& acc, PieceAcc& other, bf16x8* yprev, const uint4* w,
                                      const float* next_bias, const F& fetch) {
    constexpr int kPairs = (KS + 1) / 2;
    constexpr int kValu = 0x2, kMfma = 0x8, kVmemRead = 0x20, kDsRead = 0x100;
    static_assert(kPairs >= 4, "a quarter of the piece before in each of four pairs");
    static_assert(kPieceTiles == 2, "four products in a pair");
    bf16x8 a[2][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) a[0][j] = weight_operand<KS>(w, j % 2, j / 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kPairs; ++c) {
        if (c + 1 < kPairs) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (2 * (c + 1) + j / 2 < KS) a[(c + 1) % 2][j] = weight_operand<KS>(w, j % 2, 2 * (c + 1) + j / 2);
        }
        fetch.step(c);
        if (c + 1 == kPairs && F::kSteps > kPairs) fetch.step(kPairs);
        if (PREV && c < 4) yprev[c] = finish_quarter(other, c);
        if (NEXT && c + 1 == kPairs) start_piece(other, next_bias);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (2 * c + j / 2 < KS)
                acc[j % 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[c % 2][j], x[2 * c + j / 2], acc[j % 2], 0, 0, 0);
        __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kDsRead, 4, 0);
        __builtin_amdgcn_sched_group_barrier(kVmemRead, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kValu, 6, 0);
#pragma unroll
        for (int j = 1; j < 4; ++j) {
            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
            __builtin_amdgcn_sched_group_barrier(kValu, 6, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// A layer of 64 NP outputs over operands x[KS].  Its first piece's copy into
// w0 is under way and its biases are in acc0; each piece is multiplied while
// the next one's copy (after the last piece: the following layer's first, with
// NKS steps and as many outputs, if NKS) fills the other buffer, and while the
// piece before is finished: before this layer's first, the last of the layer
// before (its four operands x[XL ..], if XL >= 0).  NP is even, so that every
// layer starts at w0 and acc0; its last piece stays in acc1.  s_bias: of this
// layer, the following one's after it.  Every wave of the block calls it.
template <int KS, int NP, int NKS, int XL, bool ALIGNED, int P = 0>
__device__ __forceinline__ void layer(bf16x8* x, bf16x8* y, PieceAcc& acc0, PieceAcc& acc1, uint4* w0, uint4* w1,
                                      const uint16_t* W, const uint16_t* Wnext, const float* s_bias) {
    static_assert(NP % 2 == 0, "the next layer starts at w0");
    __syncthreads();  // this piece is there, and the other buffer has been read
    constexpr bool kSame = P + 1 < NP;
    using F = std::conditional_t<kSame, Fetch<KS, kPiece * NP, ALIGNED>,
                                 std::conditional_t<(NKS > 0), Fetch<NKS, kPiece * NP, ALIGNED>, NoFetch>>;
    const F fetch(kSame ? W : Wnext, kSame ? kPiece * (P + 1) : 0, P % 2 ? w0 : w1);
    constexpr bool kNext = P + 1 < NP || NKS > 0;
    const float* next_bias = s_bias + kPiece * (P + 1);
    if constexpr (P % 2 != 0) piece<KS, true, kNext>(x, acc1, acc0, y + 4 * (P - 1), w1, next_bias, fetch);
    else if constexpr (P > 0) piece<KS, true, kNext>(x, acc0, acc1, y + 4 * (P - 1), w0, next_bias, fetch);
    else piece<KS, (XL >= 0), kNext>(x, acc0, acc1, x + (XL >= 0 ? XL : 0), w0, next_bias, fetch);
    if constexpr (P + 1 < NP)
        layer<KS, NP, NKS, XL, ALIGNED, P + 1>(x, y, acc0, acc1, w0, w1, W, Wnext, s_bias);
}

struct PairArgs {
    const float* pc_xyz;   // [M, K, 3]
    const float* pc_rgb;   // [M, K, 3]
    const float* pc_dir;   // [M, K, 3]
    const float* pc_feat;  // [M, K, 32]
    const float* sp_xyz;   // [M, 3]
    const uint8_t* valid;  // [M, K]
    const float* rays_d;   // [M, 3]
    int64_t M;
    int K, ns;             // ns: samples of a block
    epcq_aggregator_params p;
    float* out_alpha;      // [M]
    uint16_t* xc;          // [M, 256] bf16 sums of the pairs' features
};

template <bool ALIGNED>
__global__ __launch_bounds__(kBlock, 2) void agg_pair_kernel(PairArgs a) {
    // two arrays, so that reading one needs no wait for the copies to the other
    __shared__ uint4 s_w0[kPieceBytes / 16];
    __shared__ uint4 s_w1[kPieceBytes / 16];
    __shared__ __align__(16) float s_bias[4 * kH];
    __shared__ __align__(16) float s_wa[kH];
    __shared__ float s_inv[kRows], s_alpha[kRows];
    const uint16_t* w1 = static_cast<const uint16_t*>(a.p.w1);
    const uint16_t* w2 = static_cast<const uint16_t*>(a.p.w2);
    const uint16_t* w3 = static_cast<const uint16_t*>(a.p.w3);
    const uint16_t* w4 = static_cast<const uint16_t*>(a.p.w4);
    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    const int lane = tid % kWave;
    const int row = lane & 31;
    const int half = lane >> 5;
    const int brow = wave * kWaveRows + row;  // row of the block
    const int64_t m0 = (int64_t)blockIdx.x * a.ns;
    const int s = brow / a.K;
    const int64_t m = m0 + s;
    const bool in_range = s < a.ns && m < a.M;
    const int64_t pair = m0 * a.K + brow;

    // ---- the rows' inputs: each lane half takes every other four features.
    // The loads of all rows are under way together, before the weights'; an
    // invalid pair's values are dropped afterwards.
    bool valid = false;
    float px = 0.0f, py = 0.0f, pz = 0.0f, sx = 0.0f, sy = 0.0f, sz = 0.0f;
    float rgb[3] = {0.0f, 0.0f, 0.0f}, dir[3] = {0.0f, 0.0f, 0.0f}, rd[3] = {0.0f, 0.0f, 0.0f};
    float4 fv[4] = {};
    if (in_range) {
        valid = a.valid[pair] != 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) fv[i] = reinterpret_cast<const float4*>(a.pc_feat + pair * kFeat)[2 * i + half];
        px = a.pc_xyz[3 * pair];
        py = a.pc_xyz[3 * pair + 1];
        pz = a.pc_xyz[3 * pair + 2];
        sx = a.sp_xyz[3 * m];
        sy = a.sp_xyz[3 * m + 1];
        sz = a.sp_xyz[3 * m + 2];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            rgb[i] = a.pc_rgb[3 * pair + i];
            dir[i] = a.pc_dir[3 * pair + i];
            rd[i] = a.rays_d[3 * m + i];
        }
    }
    Fetch<kX1 / 16, kH, ALIGNED>(w1, 0, s_w0).all();
    s_bias[tid] = a.p.b1[tid];
    s_bias[kH + tid] = a.p.b2[tid];
    s_bias[2 * kH + tid] = a.p.b3[tid];
    s_bias[3 * kH + tid] = a.p.b4[tid];
    s_wa[tid] = a.p.wa[tid];
    if (!valid) {
        px = py = pz = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) fv[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int i = 0; i < 3; ++i) rgb[i] = dir[i] = 0.0f;
    }
    // ---- x1, as operands
    const float* fs = reinterpret_cast<const float*>(fv);
    bf16x8 x[kX1 / 16], y[kX3 / 16];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float* f = fs + 8 * i;
        x[i] = swap_halves(pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7]));
    }
    // dist = p - s and distpow = p^2 - s^2; invalid pairs have p = 0 as the
    // reference's zero-filled gathers
    const float df[6] = {px - sx, py - sy, pz - sz, px * px - sx * sx, py * py - sy * sy, pz * pz - sz * sz};
    auto encode = [&](auto checked) {
        constexpr bool C = decltype(checked)::value;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // PE(f, 3): the lane's four features give 24 columns, three eights;
            // those of half 0 and half 1 follow each other
            uint32_t e[12];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float sn[3], cs[3];
                pe_sincos<C>(fs[4 * i + j], sn[0], cs[0]);
                pe_double(sn[0], cs[0], sn[1], cs[1]);
                pe_double(sn[1], cs[1], sn[2], cs[2]);
#pragma unroll
                for (int q = 0; q < 3; ++q) e[3 * j + q] = pack_bf16(sn[q], cs[q]);
            }
            // the six eights B0 B1 B2 (half 0), C0 C1 C2 (half 1) as operands
            // (B0 | B1), (B2 | C0), (C1 | C2): the middle one is in place, and
            // one swap of (B0 | C1) with (B1 | C2) gives the others
            uint32_t lo[4], mid[4], hi[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t d0 = half ? e[4 + q] : e[q];
                const uint32_t d1 = half ? e[8 + q] : e[4 + q];
                mid[q] = half ? e[q] : e[8 + q];
                const auto sw = __builtin_amdgcn_permlane32_swap(d0, d1, false, false);
                lo[q] = sw[0];
                hi[q] = sw[1];
            }
            x[2 + 3 * i] = __builtin_bit_cast(bf16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
            x[3 + 3 * i] = __builtin_bit_cast(bf16x8, make_uint4(mid[0], mid[1], mid[2], mid[3]));
            x[4 + 3 * i] = __builtin_bit_cast(bf16x8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
        }
        uint32_t e[32];
        e[30] = 0;  // columns 284..287
        e[31] = 0;
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            // frequencies 1 and 4 directly; 2, 8 and 16 by doubling
            float sn[5], cs[5];
            pe_sincos<C>(df[i], sn[0], cs[0]);
            pe_sincos<C>(df[i] * 4.0f, sn[2], cs[2]);
            pe_double(sn[0], cs[0], sn[1], cs[1]);
            pe_double(sn[2], cs[2], sn[3], cs[3]);
            pe_double(sn[3], cs[3], sn[4], cs[4]);
#pragma unroll
            for (int j = 0; j < 5; ++j) e[i * 5 + j] = pack_bf16(sn[j], cs[j]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t* l = e + 8 * i;
            x[14 + i] = __builtin_bit_cast(bf16x8, half ? make_uint4(l[4], l[5], l[6], l[7])
                                                        : make_uint4(l[0], l[1], l[2], l[3]));
        }
    };
    // one test for the wave: when every argument of its encodings is below
    // 1024 in magnitude (as it is for any features of ordinary scale) they
    // all take the hardware path without a branch each
    bool large = false;
#pragma unroll
    for (int i = 0; i < 16; ++i) large = large || !(fabsf(fs[i]) < 1024.0f);
#pragma unroll
    for (int i = 0; i < 6; ++i) large = large || !(fabsf(df[i] * 4.0f) < 1024.0f);
    if (__ballot(large) == 0) encode(std::false_type{});
    else encode(std::true_type{});
    // x3 = [h2, rgb, dir - d, dir . d, 0...]: its last operand
    float dot = dir[0] * rd[0];
    dot = dot + dir[1] * rd[1];
    dot = dot + dir[2] * rd[2];
    const uint4 tail = half ? make_uint4(0, 0, 0, 0)
                            : make_uint4(pack_bf16(rgb[0], rgb[1]), pack_bf16(rgb[2], dir[0] - rd[0]),
                                         pack_bf16(dir[1] - rd[1], dir[2] - rd[2]), pack_bf16(dot, 0.0f));
    if (__syncthreads_or(valid)) {  // the biases are there; blocks without a valid pair skip the layers
        PieceAcc acc0, acc1;
        start_piece(acc0, s_bias);
        constexpr int kLast = kH / 16 - 4;  // operands of a layer's last piece
        layer<kX1 / 16, 4, kH / 16, -1, ALIGNED>(x, y, acc0, acc1, s_w0, s_w1, w1, w2, s_bias);
        layer<kH / 16, 4, kX3 / 16, kLast, ALIGNED>(y, x, acc0, acc1, s_w0, s_w1, w2, w3, s_bias + kH);
        x[kH / 16] = __builtin_bit_cast(bf16x8, tail);
        layer<kX3 / 16, 4, kH / 16, kLast, ALIGNED>(x, y, acc0, acc1, s_w0, s_w1, w3, w4, s_bias + 2 * kH);
        layer<kH / 16, 4, 0, kLast, ALIGNED>(y, x, acc0, acc1, s_w0, s_w1, w4, nullptr, s_bias + 3 * kH);
        finish_piece(acc1, x + kLast);
    }
    __syncthreads();  // every wave has read its weights: the buffers take the rows

    auto lds_row = [&](int r) {
        uint16_t* base = reinterpret_cast<uint16_t*>(r < 2 * kWaveRows ? s_w0 : s_w1);
        return base + (r % (2 * kWaveRows)) * kLdsStride;
    };
    // ---- the rows for the reductions; an invalid pair's is zero
    uint16_t* xr = lds_row(brow);
    if (valid) {
#pragma unroll
        for (int i = 0; i < kH / 16; ++i) *reinterpret_cast<bf16x8*>(xr + 16 * i + 8 * half) = x[i];
    } else {
#pragma unroll
        for (int i = 0; i < kH / 16; ++i) *reinterpret_cast<bf16x8*>(xr + 16 * i + 8 * half) = bf16x8{};
    }
    // ---- per-pair alpha, each lane half over the columns that it holds
    // (fused multiply-adds: one rounding each)
    float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < kH / 16; ++i) {
        const uint4 h = __builtin_bit_cast(uint4, x[i]);
        const float4 wl = *reinterpret_cast<const float4*>(s_wa + 16 * i + 8 * half);
        const float4 wh = *reinterpret_cast<const float4*>(s_wa + 16 * i + 8 * half + 4);
        part[0] = __builtin_fmaf(wl.x, __uint_as_float(h.x << 16), part[0]);
        part[1] = __builtin_fmaf(wl.y, __uint_as_float(h.x & 0xffff0000u), part[1]);
        part[2] = __builtin_fmaf(wl.z, __uint_as_float(h.y << 16), part[2]);
        part[3] = __builtin_fmaf(wl.w, __uint_as_float(h.y & 0xffff0000u), part[3]);
        part[0] = __builtin_fmaf(wh.x, __uint_as_float(h.z << 16), part[0]);
        part[1] = __builtin_fmaf(wh.y, __uint_as_float(h.z & 0xffff0000u), part[1]);
        part[2] = __builtin_fmaf(wh.z, __uint_as_float(h.w << 16), part[2]);
        part[3] = __builtin_fmaf(wh.w, __uint_as_float(h.w & 0xffff0000u), part[3]);
    }
    const float sum4 = (part[0] + part[1]) + (part[2] + part[3]);
    const float dotv = sum4 + __shfl_xor(sum4, 32) + a.p.ba[0];
    // ---- inverse distances, for the weights
    const float dx = px - sx, dy = py - sy, dz = pz - sz;
    float nrm = dx * dx;
    nrm = nrm + dy * dy;
    nrm = nrm + dz * dz;
    if (half == 0) {
        s_inv[brow] = valid ? 1.0f / (sqrtf(nrm) + 1e-6f) : 0.0f;
        s_alpha[brow] = valid ? softplus(dotv - 1.0f) : 0.0f;
    }
    __syncthreads();

    // ---- per sample, one for each half of the wave and eight columns for each
    // lane: weights, alpha and the weighted feature sum, in the order of the
    // neighbours
    for (int i = 2 * wave + half; i < a.ns && m0 + i < a.M; i += 2 * kWaves) {
        const int r0 = i * a.K;
        float sum = 0.0f;
        for (int j = 0; j < a.K; ++j) sum += s_inv[r0 + j];
        sum += 1e-6f;
        float acc_a = 0.0f;
        float acc[8] = {};
        for (int j = 0; j < a.K; ++j) {
            const float wj = s_inv[r0 + j] / sum;
            acc_a = __builtin_fmaf(wj, s_alpha[r0 + j], acc_a);
            const uint4 h = *reinterpret_cast<const uint4*>(lds_row(r0 + j) + row * 8);
            const uint32_t hw[4] = {h.x, h.y, h.z, h.w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                acc[2 * q] = __builtin_fmaf(wj, __uint_as_float(hw[q] << 16), acc[2 * q]);
                acc[2 * q + 1] = __builtin_fmaf(wj, __uint_as_float(hw[q] & 0xffff0000u), acc[2 * q + 1]);
            }
        }
        const uint4 packed = make_uint4(pack_bf16(acc[0], acc[1]), pack_bf16(acc[2], acc[3]),
                                        pack_bf16(acc[4], acc[5]), pack_bf16(acc[6], acc[7]));
        reinterpret_cast<uint4*>(a.xc + (m0 + i) * kH)[row] = packed;
        if (row == 0) a.out_alpha[m0 + i] = acc_a;
    }
}

struct ColorArgs {
    const uint16_t* xc;  // [M, 256]
    const float* rays_d; // [M, 3]
    int64_t M;
    epcq_aggregator_params p;
    float* out_rgb;      // [M, 3]
};

template <bool ALIGNED>
__global__ __launch_bounds__(kBlock, 2) void agg_color_kernel(ColorArgs a) {
    __shared__ uint4 s_w0[kPieceBytes / 16];
    __shared__ uint4 s_w1[kPieceBytes / 16];
    __shared__ __align__(16) float s_bias[3 * kC];
    __shared__ __align__(16) float s_c4[3 * kC];
    const uint16_t* c1 = static_cast<const uint16_t*>(a.p.c1);
    const uint16_t* c2 = static_cast<const uint16_t*>(a.p.c2);
    const uint16_t* c3 = static_cast<const uint16_t*>(a.p.c3);
    Fetch<kXc / 16, kC, ALIGNED>(c1, 0, s_w0).all();
    const int tid = threadIdx.x;
    if (tid < kC) {
        s_bias[tid] = a.p.cb1[tid];
        s_bias[kC + tid] = a.p.cb2[tid];
        s_bias[2 * kC + tid] = a.p.cb3[tid];
#pragma unroll
        for (int j = 0; j < 3; ++j) s_c4[j * kC + tid] = a.p.c4[j * kC + tid];
    }
    const int lane = tid % kWave;
    const int half = lane >> 5;
    const int64_t m = (int64_t)blockIdx.x * kRows + tid / kWave * kWaveRows + (lane & 31);
    bf16x8 x[kXc / 16], y[kC / 16];
#pragma unroll
    for (int i = 0; i < kH / 16; ++i) x[i] = m < a.M ? load8(a.xc + m * kH + 16 * i + 8 * half) : bf16x8{};
    // PE(d, 4): half 0 takes d_x and d_z, half 1 d_y and the columns past it
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float d = m < a.M ? a.rays_d[3 * m + (i ? 2 : half)] : 0.0f;
        uint32_t e[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float sn, cs;
            pe_sincos(d * (float)(1 << j), sn, cs);
            e[j] = i && half ? 0 : pack_bf16(sn, cs);
        }
        x[kH / 16 + i] = __builtin_bit_cast(bf16x8, make_uint4(e[0], e[1], e[2], e[3]));
    }
    PieceAcc acc0, acc1;
    __syncthreads();
    start_piece(acc0, s_bias);
    constexpr int kLast = kC / 16 - 4;
    layer<kXc / 16, 2, kC / 16, -1, ALIGNED>(x, y, acc0, acc1, s_w0, s_w1, c1, c2, s_bias);
    layer<kC / 16, 2, kC / 16, kLast, ALIGNED>(y, x, acc0, acc1, s_w0, s_w1, c2, c3, s_bias + kC);
    layer<kC / 16, 2, 0, kLast, ALIGNED>(x, y, acc0, acc1, s_w0, s_w1, c3, nullptr, s_bias + 2 * kC);
    finish_piece(acc1, y + kLast);
    if (m >= a.M) return;
    // last layer (128 -> 3) in fp32, each half the columns that it holds
    float part[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < kC / 16; ++i) {
        const uint4 h = __builtin_bit_cast(uint4, y[i]);
        const float hv[8] = {__uint_as_float(h.x << 16), __uint_as_float(h.x & 0xffff0000u),
                             __uint_as_float(h.y << 16), __uint_as_float(h.y & 0xffff0000u),
                             __uint_as_float(h.z << 16), __uint_as_float(h.z & 0xffff0000u),
                             __uint_as_float(h.w << 16), __uint_as_float(h.w & 0xffff0000u)};
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const float* wq = s_c4 + j * kC + 16 * i + 8 * half;
#pragma unroll
            for (int v = 0; v < 8; ++v) part[j] += wq[v] * hv[v];
        }
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const float other = __shfl_xor(part[j], 32);
        const float v = (half ? other + part[j] : part[j] + other) + a.p.cb4[j];
        const float sig = 1.0f / (1.0f + expf(-v));
        if (half == 0) a.out_rgb[3 * m + j] = sig * (1.0f + 2.0f * 0.001f) - 0.001f;
    }
}

}  // namespace
}  // namespace epcq

using namespace epcq;

extern "C" size_t epcq_aggregator_workspace_size(int64_t M) {
    if (M <= 0) return 0;
    return (size_t)M * kH * sizeof(uint16_t);
}

extern "C" int epcq_aggregator_forward(const float* pc_xyz, const float* pc_rgb, const float* pc_dir,
                                       const float* pc_feat, const float* sp_xyz, const uint8_t* valid,
                                       const float* rays_d, int64_t M, int32_t K, int32_t F,
                                       const epcq_aggregator_params* params, float* out_alpha, float* out_rgb,
                                       void* workspace, size_t workspace_bytes, void* stream) {
    if (M < 0) return fail(EPCQ_ERR_INVALID, "aggregator: negative sample count");
    if (K < 1 || K > 32) return fail(EPCQ_ERR_INVALID, "aggregator: num_point_cloud_per_sp must be in [1, 32]");
    if (F != kFeat)
        return fail(EPCQ_ERR_INVALID, "aggregator: pc_feat must have 32 features (block1 takes 7F + 60 = 284 inputs)");
    if (!params) return fail(EPCQ_ERR_INVALID, "aggregator: missing parameters");
    if (M == 0) return EPCQ_OK;
    const size_t need = epcq_aggregator_workspace_size(M);
    if (workspace_bytes < need || !workspace) return fail(EPCQ_ERR_WORKSPACE, "aggregator: workspace too small");
    if ((reinterpret_cast<uintptr_t>(workspace) & 15u) != 0)
        return fail(EPCQ_ERR_INVALID, "aggregator: workspace must be 16-byte aligned");
    hipStream_t st = as_stream(stream);
    PairArgs pa;
    pa.pc_xyz = pc_xyz;
    pa.pc_rgb = pc_rgb;
    pa.pc_dir = pc_dir;
    pa.pc_feat = pc_feat;
    pa.sp_xyz = sp_xyz;
    pa.valid = valid;
    pa.rays_d = rays_d;
    pa.M = M;
    pa.K = K;
    pa.ns = kRows / K;
    pa.p = *params;
    pa.out_alpha = out_alpha;
    pa.xc = static_cast<uint16_t*>(workspace);
    const int64_t blocks = ceil_div(M, pa.ns);
    if (blocks > INT32_MAX) return fail(EPCQ_ERR_INVALID, "aggregator: too many samples");
    uintptr_t low = 0;  // the load unit's copies to LDS want 16-byte alignment
    for (const void* w : {params->w1, params->w2, params->w3, params->w4, params->c1, params->c2, params->c3})
        low |= reinterpret_cast<uintptr_t>(w);
    const bool aligned = (low & 15u) == 0;
    if (aligned) agg_pair_kernel<true><<<dim3((unsigned)blocks), dim3(kBlock), 0, st>>>(pa);
    else agg_pair_kernel<false><<<dim3((unsigned)blocks), dim3(kBlock), 0, st>>>(pa);
    if (int e = check_launch("aggregator/pairs")) return e;
    ColorArgs ca;
    ca.xc = pa.xc;
    ca.rays_d = rays_d;
    ca.M = M;
    ca.p = *params;
    ca.out_rgb = out_rgb;
    const dim3 cgrid((unsigned)ceil_div(M, kRows));
    if (aligned) agg_color_kernel<true><<<cgrid, dim3(kBlock), 0, st>>>(ca);
    else agg_color_kernel<false><<<cgrid, dim3(kBlock), 0, st>>>(ca);
    return check_launch("aggregator/colour");
}
