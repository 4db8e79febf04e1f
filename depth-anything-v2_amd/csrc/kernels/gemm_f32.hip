// fp32 and fp16 paths of the precision modes (DAV2_CREATE_FORCE_FP32 /
// FORCE_FP16): the linear and convolution GEMMs in float32 on the MFMA
// (v_mfma_f32_16x16x4_f32, or v_mfma_f32_16x16x32_bf16 on operands split in
// three), with the epilogues of the int8 GEMM, and the fp32 im2col that feeds
// convolutions.
//
// fp16 arithmetic comes in the reference's two forms. Cooperative-matrix
// linears (linear_coop_fp16.glsl via linear_fp16* with cooperative_matrix_fp16,
// src/operators.cpp:540-768): operands rounded to binary16, exact products,
// fp32 accumulation. The fp32 GEMM does this with half_operands: both operands
// are rounded to binary16 on their way from LDS to v_mfma_f32_16x16x4_f32, which
// multiplies them exactly and sums in fp32. Native binary16 shaders
// (prepare_tokens_fp16, project_tokens_fp16, conv_transpose_nonoverlap_fp16):
// every product is a binary16 multiplication, widened and added to an fp32 sum
// in k order; gemm_h16p_kernel does exactly that on the VALU, so its results
// match the oracle bit for bit.
//
// Reference: linear_tiled.glsl / linear_vec*.glsl (src/operators.cpp:882-955),
// conv2d (:1528-1676), conv_transpose_nonoverlap (:1807-1861),
// project_tokens (:1408-1452), gelu.glsl, add_scaled.glsl. The reference sums
// each dot product in its own tile order; fp32 results are compared within a
// tolerance, not bit for bit.
//
// K advances in stages of 32 floats copied straight from global memory into an
// LDS ring (global_load_lds_dwordx4), XOR-swizzled 128-byte rows as in the int8
// GEMM, one barrier per stage; the operands of the next 16 k are read from LDS
// while the present ones multiply. A lane's 16-byte fragment holds 4
// consecutive k of its row; the 4 MFMAs of a fragment take element e of every
// lane, so each MFMA sums k = 4g + e over the lane groups g and the four
// together cover 16 k. What bounds it: the fp32 MFMA (157 TFLOP/s), of which
// a chip full of tiles reaches 110 (the same loop without the copies: 135).

#include <type_traits>

#include "common.h"
#include "dav2_hip.h"

namespace {

using namespace dav2k;

constexpr int kBK = 32;  // floats per K step

struct F32Params {
    const float* a;
    uint64_t lda;
    const float* b;
    uint64_t ldb;
    uint32_t m, n, k;
    const float* bias;
    float* out;
    uint64_t out_row_offset, out_row_stride;
    const float* residual;
    const float* gamma;
    uint32_t relu_output;
    uint32_t convt_k, convt_w, convt_h, convt_c;
    uint32_t half_operands;  // round both operands to binary16
};

// Four consecutive weight rows n .. n + 3 of activation row m. Row-major
// epilogues write them as one float4 when `vec` (n % 4 == 0 rows and 16-byte
// aligned buffers); the channel-major ones run along m across the lanes.
template <int EPI>
DAV2_DEV void store_f32(const F32Params& g, uint32_t m, uint32_t n, const float (&acc)[4], bool vec) {
    if (EPI == DAV2_GEMM_EPI_CONVT || EPI == DAV2_GEMM_EPI_TRANSPOSED) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (n + r >= g.n) return;
            if (EPI == DAV2_GEMM_EPI_CONVT) {
                const uint32_t kidx = (n + r) / g.convt_c, oc = (n + r) - kidx * g.convt_c;
                const float v = acc[r] + (g.bias ? g.bias[oc] : 0.0f);
                const uint32_t k = g.convt_k;
                const uint32_t iy = m / g.convt_w, ix = m - iy * g.convt_w;
                const uint32_t ky = kidx / k, kx = kidx - ky * k;
                const uint32_t ow = g.convt_w * k, oh = g.convt_h * k;
                g.out[(static_cast<uint64_t>(oc) * oh + iy * k + ky) * ow + ix * k + kx] = v;
            } else {
                const uint64_t idx = static_cast<uint64_t>(n + r) * g.out_row_stride + m + g.out_row_offset;
                float o = acc[r] + (g.bias ? g.bias[n + r] : 0.0f);
                if (g.residual) o = o + g.residual[idx];
                if (g.relu_output) o = fmaxf(o, 0.0f);
                g.out[idx] = o;
            }
        }
        return;
    }
    const uint64_t idx = (static_cast<uint64_t>(m) + g.out_row_offset) * g.n + n;
    float v[4], res[4], gam[4];
    if (vec) {
        const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
        const float4 b = g.bias ? *reinterpret_cast<const float4*>(g.bias + n) : zero;
        v[0] = acc[0] + b.x, v[1] = acc[1] + b.y, v[2] = acc[2] + b.z, v[3] = acc[3] + b.w;
        if (EPI == DAV2_GEMM_EPI_ROW_LAYERSCALE) {
            const float4 s = *reinterpret_cast<const float4*>(g.gamma + n);
            const float4 x = *reinterpret_cast<const float4*>(g.residual + idx);
            gam[0] = s.x, gam[1] = s.y, gam[2] = s.z, gam[3] = s.w;
            res[0] = x.x, res[1] = x.y, res[2] = x.z, res[3] = x.w;
        }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bool in = n + r < g.n;
            v[r] = acc[r] + (g.bias && in ? g.bias[n + r] : 0.0f);
            if (EPI == DAV2_GEMM_EPI_ROW_LAYERSCALE) {
                gam[r] = in ? g.gamma[n + r] : 0.0f;
                res[r] = in ? g.residual[idx + r] : 0.0f;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (EPI == DAV2_GEMM_EPI_ROW_GELU) v[r] = gelu_erfcc(v[r]);
        if (EPI == DAV2_GEMM_EPI_ROW_LAYERSCALE) {
            const float scaled = v[r] * gam[r];  // add_scaled.glsl:26-30, no contraction
            v[r] = res[r] + scaled;
        }
    }
    if (vec) {
        *reinterpret_cast<float4*>(g.out + idx) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r < g.n) g.out[idx + r] = v[r];
    }
}

template <int EPI>
DAV2_DEV bool vector_rows(const F32Params& g) {
    if (EPI == DAV2_GEMM_EPI_CONVT || EPI == DAV2_GEMM_EPI_TRANSPOSED) return false;
    const uintptr_t any = reinterpret_cast<uintptr_t>(g.out) | reinterpret_cast<uintptr_t>(g.bias) |
                          reinterpret_cast<uintptr_t>(g.gamma) | reinterpret_cast<uintptr_t>(g.residual);
    return g.n % 4u == 0 && (any & 15u) == 0;
}

// First row and column of this workgroup's tile; false past the last row. Row
// tiles go to grid x, and on to z beyond kMaxRowTiles.
template <int BN, int BM>
DAV2_DEV bool tile_start(const F32Params& g, uint32_t& row0, uint32_t& col0) {
    uint32_t tm, tn;
    tile_of(tm, tn);
    const uint64_t row = (static_cast<uint64_t>(blockIdx.z) * gridDim.x + tm) * BM;
    row0 = static_cast<uint32_t>(row);
    col0 = tn * BN;
    return row < g.m;
}

// BN weight rows (operand P of the MFMA, whose four result registers are then
// consecutive output columns) x BM activation rows per workgroup, WN x WM
// waves.
template <int BN, int BM, int WN, int WM, int STAGES, bool HALF, int EPI>
__global__ __launch_bounds__(64 * WN * WM) void gemm_f32_kernel(F32Params g) {
    constexpr int NW = WN * WM, TN = BN / WN / 16, TM = BM / WM / 16;
    constexpr int COPIES = (BN + BM) / 8;  // 1 KiB global -> LDS copies (8 rows of 128 bytes) per stage
    constexpr int LPW = (COPIES + NW - 1) / NW;
    constexpr int STAGE_BYTES = (BN + BM) * 128;
    static_assert(TN * WN * 16 == BN && TM * WM * 16 == BM, "whole MFMA blocks per wave");
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave / WM, wm = wave % WM;
    uint32_t row0, col0;
    if (!tile_start<BN, BM>(g, row0, col0)) return;
    const int steps = static_cast<int>((g.k + kBK - 1) / kBK);

    // Copy c brings stage rows 8 c .. + 7, lane l row + l / 8 and the 16-byte
    // chunk that swz maps to l % 8; wave w takes copies i NW + w (past the
    // last one it repeats that one, the same bytes). Rows past the
    // matrix read its last row (never stored), chunks past K chunk 0 of the
    // row (masked below).
    const float* src[LPW];
    uint32_t chunk_k[LPW];
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
        const uint32_t srow = 8u * min(i * NW + wave, COPIES - 1) + (lane >> 3);
        chunk_k[i] = 4u * ((lane & 7) ^ ((srow >> 1) & 7u));
        src[i] = srow < static_cast<uint32_t>(BN)  // uniform per instruction (BN % 8 == 0)
                     ? g.b + min(col0 + srow, g.n - 1) * g.ldb
                     : g.a + min(row0 + srow - BN, g.m - 1) * g.lda;
    }
    auto issue = [&](int step) {
#pragma unroll
        for (int i = 0; i < LPW; ++i) {
            const uint32_t kk = static_cast<uint32_t>(step) * kBK + chunk_k[i];
            copy16_to_lds(src[i] + (kk < g.k ? kk : 0u),
                          smem + (step % STAGES) * STAGE_BYTES + min(i * NW + wave, COPIES - 1) * 1024);
        }
    };

    v4f acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int s = 0; s < STAGES; ++s)
        if (s < steps) issue(s);
    // Fragments of 16 k (two per stage) go through two register sets: one is
    // read from LDS while the other multiplies.
    const int fr = lane & 15, fg = lane >> 4;
    v4f pf[2][TN], qf[2][TM];
    auto read = [&](int step, auto half) {
        constexpr int h = decltype(half)::value;
        const int8_t* st = smem + (step % STAGES) * STAGE_BYTES;
#pragma unroll
        for (int i = 0; i < TN; ++i)
            pf[h][i] = *reinterpret_cast<const v4f*>(st + swz<128>(wn * (TN * 16) + i * 16 + fr, 4 * h + fg));
#pragma unroll
        for (int j = 0; j < TM; ++j)
            qf[h][j] = *reinterpret_cast<const v4f*>(st + swz<128>(BN + wm * (TM * 16) + j * 16 + fr, 4 * h + fg));
    };
    // Binary16 operands are rounded here; the fp32 MFMA's products of them are
    // exact, subnormal ones included (v_mfma_f32_16x16x32_f16 sums a subnormal
    // operand with the weight of one of 2^-14).
    auto operand = [](v4f v) {
        return HALF ? __builtin_convertvector(__builtin_convertvector(v, v4h), v4f) : v;
    };
    auto multiply = [&](auto half) {
        constexpr int h = decltype(half)::value;
        v4f p[TN], q[TM];
#pragma unroll
        for (int i = 0; i < TN; ++i) p[i] = operand(pf[h][i]);
#pragma unroll
        for (int j = 0; j < TM; ++j) q[j] = operand(qf[h][j]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[i][e], q[j][e], acc[i][j], 0, 0, 0);
    };
    const std::integral_constant<int, 0> h0;
    const std::integral_constant<int, 1> h1;
    wait_stages<STAGES - 1, LPW>(min(STAGES - 1, steps - 1));
    __builtin_amdgcn_s_barrier();
    read(0, h0);
    for (int step = 0; step + 1 < steps; ++step) {
        read(step, h1);
        // rounding and products of binary16 operands interleave freely
        // (1370 x 2304 x 768 70 -> 65 us)
        if constexpr (!HALF) __builtin_amdgcn_sched_barrier(0);
        multiply(h0);
        if constexpr (!HALF) __builtin_amdgcn_sched_barrier(0);
        // this wave's operands of the stage are in registers and its copies
        // of the next stage have landed; after the barrier every wave's have,
        // and the slot is free for the stage STAGES later
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        wait_stages<STAGES - 2, LPW>(min(STAGES - 2, steps - 2 - step));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (step + STAGES < steps) issue(step + STAGES);
        read(step + 1, h0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(h1);
    }
    read(steps - 1, h1);
    auto clear_past = [&](auto half) {  // k past K (whole chunks, K % 4 == 0): zeros
        constexpr int h = decltype(half)::value;
        if (static_cast<uint32_t>(steps - 1) * kBK + 16u * h + 4u * fg < g.k) return;
#pragma unroll
        for (int i = 0; i < TN; ++i) pf[h][i] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < TM; ++j) qf[h][j] = v4f{0.f, 0.f, 0.f, 0.f};
    };
    clear_past(h0);
    clear_past(h1);
    multiply(h0);
    multiply(h1);

    // 16x16 result layout: lane l holds rows 4 (l / 16) + r of column l % 16.
    const bool vec = vector_rows<EPI>(g);
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        const uint32_t m = row0 + wm * (TM * 16) + j * 16 + fr;
        if (m >= g.m) continue;
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            const uint32_t n = col0 + wn * (TN * 16) + i * 16 + 4 * fg;
            const float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            if (n < g.n) store_f32<EPI>(g, m, n, v, vec);
        }
    }
}

typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2b __attribute__((ext_vector_type(2)));

// Operands are split times 2^24: the parts of anything above 2^-126 are then
// normal bfloat16 values, and those of subnormal floats too. Past 2^103 they
// are infinite, as are sums past 2^80.
constexpr float kSplitScale = 16777216.0f;

// Four floats as three bfloat16 parts each, every part the value nearest to
// what is left (ties to even): x = part 0 + part 1 + part 2 exactly, |part 1| <=
// 2^-8 and |part 2| <= 2^-17 of the power of two at or below |x|.
DAV2_DEV void split_bf16(v4f x, v2u (&part)[3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const v2f pair = {x[2 * h], x[2 * h + 1]};
            const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, v2b));
            part[k][h] = u;
            if (k < 2) {
                x[2 * h] -= __uint_as_float(u << 16);
                x[2 * h + 1] -= __uint_as_float(u & 0xFFFF0000u);
            }
        }
    }
}

// fp32 operands on the bfloat16 MFMA: each operand is split into three parts
// on its way into LDS (global -> registers, two stages ahead -> three planes of
// BK values a row) and six products per element go to v_mfma_f32_16x16x32_bf16: 96
// matrix cycles for 32 k of a block where v_mfma_f32_16x16x4_f32 takes 256. The
// three left out (parts 1 and 2, twice, and 2 and 2) are at most (1 + 2^-10)
// 2^-24 of the element's product. Products of the same order (part numbers that
// add up to 0, 1, 2) have a sum of their own: the MFMA cuts off what lies below
// its accumulator, and the small products added to the large sum cost 10 times
// this error where all operands are positive. Relative error against 64 bits,
// fp32 MFMA -> this, K = 64 / 384 / 1024 / 4096: normal operands 1.4e-7 / 3.5e-7 /
// 5.7e-7 / 1.1e-6 -> 5.0e-8 / 1.1e-7 / 1.9e-7 / 4.0e-7, positive ones 1.2e-7 / 2.7e-7
// / 4.9e-7 / 9.9e-7 -> 5.2e-8 / 1.0e-7 / 1.8e-7 / 3.5e-7, mantissas of the largest
// left-out products 9.3e-8 / 2.1e-7 / 5.2e-7 / 8.8e-6 -> 6.2e-8 / 6.6e-8 / 6.2e-8 /
// 6.8e-8. What bounds it: LDS (four plane reads and one write for each product of
// a 32x32 wave block) and the VALU's splitting.
template <int BN, int BM, int WN, int WM, int BK, int EPI>
__global__ __launch_bounds__(64 * WN * WM) void gemm_split_kernel(F32Params g) {
    constexpr int NT = 64 * WN * WM, TN = BN / WN / 16, TM = BM / WM / 16;
    constexpr int ROWS = BN + BM, QK = BK / 4, LPT = (ROWS * QK + NT - 1) / NT;  // float4 loads per thread and stage
    constexpr int PLANE = ROWS * BK * 2, STAGE = 3 * PLANE;  // bytes
    static_assert(TN * WN * 16 == BN && TM * WM * 16 == BM && NT % QK == 0, "whole blocks and rows");
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave / WM, wm = wave % WM;
    const int fr = lane & 15, fg = lane >> 4;
    uint32_t row0, col0;
    if (!tile_start<BN, BM>(g, row0, col0)) return;
    const int steps = static_cast<int>((g.k + BK - 1) / BK);

    // Thread t's load i is float4 t % QK of stage row t / QK + i NT / QK (past
    // the last row that one again, the same bytes). Rows past the matrix read
    // its last row (never stored), k past K is zero.
    const uint32_t kq = 4u * (tid % QK);
    const float* src[LPT];
    uint32_t dst[LPT];
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
        const uint32_t r = min(tid / QK + i * (NT / QK), ROWS - 1);
        src[i] = (r < static_cast<uint32_t>(BN) ? g.b + min(col0 + r, g.n - 1) * g.ldb
                                                : g.a + min(row0 + r - BN, g.m - 1) * g.lda) + kq;
        dst[i] = swz<2 * BK>(r, (tid % QK) >> 1) + 8u * (tid & 1);
    }
    v4f next[2][LPT];
    auto load = [&](int step, auto set) {
        const bool in = static_cast<uint32_t>(step) * BK + kq < g.k;
#pragma unroll
        for (int i = 0; i < LPT; ++i) {
            next[decltype(set)::value][i] = *reinterpret_cast<const v4f*>(src[i] + (in ? step * BK : -static_cast<int>(kq)));
        }
    };
    auto stash = [&](int step, auto set) {
        const bool in = static_cast<uint32_t>(step) * BK + kq < g.k;
        int8_t* st = smem + decltype(set)::value * STAGE;
#pragma unroll
        for (int i = 0; i < LPT; ++i) {
            v2u part[3];
            split_bf16(in ? next[decltype(set)::value][i] * kSplitScale : v4f{0.f, 0.f, 0.f, 0.f}, part);
#pragma unroll
            for (int k = 0; k < 3; ++k) *reinterpret_cast<v2u*>(st + k * PLANE + dst[i]) = part[k];
        }
    };

    v4f acc[TN][TM], mid[TN][TM], low[TN][TM];  // sums of the products of order 0, 1, 2
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = mid[i][j] = low[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    const std::integral_constant<int, 0> h0;
    const std::integral_constant<int, 1> h1;
    load(0, h0);
    load(min(1, steps - 1), h1);
    stash(0, h0);
    load(min(2, steps - 1), h0);
    __syncthreads();
    auto stage = [&](int step, auto cur, auto nxt) {
        const int8_t* st = smem + decltype(cur)::value * STAGE;
        v8b pf[BK / 32][3][TN], qf[BK / 32][3][TM];
#pragma unroll
        for (int h = 0; h < BK / 32; ++h)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int8_t* plane = st + k * PLANE;
#pragma unroll
                for (int i = 0; i < TN; ++i)
                    pf[h][k][i] =
                        *reinterpret_cast<const v8b*>(plane + swz<2 * BK>((wn * TN + i) * 16 + fr, 4 * h + fg));
#pragma unroll
                for (int j = 0; j < TM; ++j)
                    qf[h][k][j] =
                        *reinterpret_cast<const v8b*>(plane + swz<2 * BK>(BN + (wm * TM + j) * 16 + fr, 4 * h + fg));
            }
        // unconditional (past the last stage it is loaded again and never
        // read), so that the waits count the other set's loads as in flight
        stash(step + 1, nxt);
        load(min(step + 3, steps - 1), nxt);
        constexpr int pp[6] = {2, 1, 0, 1, 0, 0}, qq[6] = {0, 0, 0, 1, 1, 2};
#pragma unroll
        for (int h = 0; h < BK / 32; ++h)
#pragma unroll
            for (int t = 0; t < 6; ++t)
#pragma unroll
                for (int i = 0; i < TN; ++i)
#pragma unroll
                    for (int j = 0; j < TM; ++j) {
                        const int order = pp[t] + qq[t];
                        v4f& sum = order == 0 ? acc[i][j] : order == 1 ? mid[i][j] : low[i][j];
                        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[h][pp[t]][i], qf[h][qq[t]][j], sum, 0, 0, 0);
                    }
        // this wave's reads of the stage and its writes of the next have
        // ended; after the barrier every wave's have
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
    };
    int step = 0;
    for (; step + 1 < steps; step += 2) {
        stage(step, h0, h1);
        stage(step + 1, h1, h0);
    }
    if (step < steps) stage(step, h0, h1);

    // Infinite and NaN operands, and operands and sums that the scale takes past
    // the largest float, end as infinities or NaN here: a wave with such a sum
    // computes its block again on the fp32 MFMA, operands straight from memory,
    // and takes those sums from there.
    auto infinite = [](float v) { return !(fabsf(v) <= 3.402823466e+38f); };
    bool again = false;
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[i][j][r] = (acc[i][j][r] + (mid[i][j][r] + low[i][j][r])) * (1.0f / (kSplitScale * kSplitScale));
                again |= infinite(acc[i][j][r]);
            }
    if (__any(again)) {
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j) mid[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        for (uint32_t k = 4u * fg; k < g.k + 4u * fg; k += 16u) {
            v4f p[TN], q[TM];
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const uint32_t n = min(col0 + wn * (TN * 16) + i * 16 + fr, g.n - 1);
                p[i] = k < g.k ? *reinterpret_cast<const v4f*>(g.b + n * g.ldb + k) : v4f{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                const uint32_t m = min(row0 + wm * (TM * 16) + j * 16 + fr, g.m - 1);
                q[j] = k < g.k ? *reinterpret_cast<const v4f*>(g.a + m * g.lda + k) : v4f{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TN; ++i)
#pragma unroll
                    for (int j = 0; j < TM; ++j)
                        mid[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[i][e], q[j][e], mid[i][j], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (infinite(acc[i][j][r])) acc[i][j][r] = mid[i][j][r];
    }

    // 16x16 result layout: lane l holds rows 4 (l / 16) + r of column l % 16.
    const bool vec = vector_rows<EPI>(g);
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        const uint32_t m = row0 + wm * (TM * 16) + j * 16 + fr;
        if (m >= g.m) continue;
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            const uint32_t n = col0 + wn * (TN * 16) + i * 16 + 4 * fg;
            const float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            if (n < g.n) store_f32<EPI>(g, m, n, v, vec);
        }
    }
}

// Native binary16 products: out[m][n] = sum over k = 0, 1, .. K-1 of
// float(fp16(h(a[m][k]) * h(b[n][k]))) in fp32, h = round to binary16, then
// the epilogue (+ bias): prepare_tokens_fp16.glsl:37-52,
// project_tokens_common.glsl (NATIVE_FP16) and
// conv_transpose_nonoverlap_common.glsl (NATIVE_FP16), whose sums run over
// the inner index in ascending order.
//
// Bounded by the VALU (a product is half a v_pk_mul_f16, two k at once, and a
// v_fma_mix_f32 that widens and adds it) and, since every sum is one chain over
// K, by the waves that hide its latency: small tiles, 32 R x 32 on four waves.
// A thread owns one row (or two, 32 apart) of 32 and four columns. K goes in
// chunks of 64, rounded on the way from registers (one chunk ahead) into one of
// two LDS buffers of 128-byte rows, whose 16-byte pieces (8 k) are XOR-swizzled
// so that the rows a wave reads at once fall on different banks. Past K both
// operands are zero: + 0 leaves a sum as it is.
// us at rows x N x K, 64x64 tiles of 4x4 a thread and the products widened and
// added separately -> this: 1369 x 768 x 588 131 -> 57, 1369 x 96 x 768 122 ->
// 21, 1369 x 768 x 768 166 -> 66, 5476 x 1024 x 1024 527 -> 331 (17 T
// products/s), 252 x 384 x 588 94 -> 18.
constexpr uint32_t kMaxGridY = 65535u;

template <int R, int EPI>
__global__ __launch_bounds__(256) void gemm_h16p_kernel(F32Params g) {
    constexpr int kRows = 32 * R + 32, kLoads = kRows * 16 / 256;  // columns (weights) first
    __shared__ __attribute__((aligned(16))) int8_t tile[2][kRows * 128];
    // channel-major epilogues store along the rows: there the lanes run over them
    constexpr bool kAlongRows = EPI == DAV2_GEMM_EPI_CONVT || EPI == DAV2_GEMM_EPI_TRANSPOSED;
    const uint32_t tid = threadIdx.x, tx = kAlongRows ? tid >> 5 : tid & 7u, ty = kAlongRows ? tid & 31u : tid >> 3;
    const uint32_t row0 = blockIdx.x * 32u * R, col0 = (blockIdx.z * kMaxGridY + blockIdx.y) * 32u;
    if (col0 >= g.n) return;
    auto piece = [](uint32_t r, uint32_t c) { return r * 128u + ((c ^ r ^ (r >> 2)) & 7u) * 16u; };

    // Thread t's load i is float4 t % 16 of tile row t / 16 + 16 i; rows past
    // the matrix read its last row (never stored).
    const uint32_t kq = 4u * (tid & 15u);
    const float* src[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const uint32_t r = (tid >> 4) + 16u * i;
        src[i] = i < 2 ? g.b + min(col0 + r, g.n - 1) * g.ldb : g.a + min(row0 + r - 32u, g.m - 1) * g.lda;
    }
    v4f next[kLoads];
    auto load = [&](uint32_t k0) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) next[i] = *reinterpret_cast<const v4f*>(src[i] + (k0 + kq < g.k ? k0 + kq : 0u));
    };
    auto stash = [&](uint32_t k0, int8_t* buf) {
        const bool in = k0 + kq < g.k;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const v4f v = in ? next[i] : v4f{0.f, 0.f, 0.f, 0.f};
            const v4h h = {static_cast<_Float16>(v[0]), static_cast<_Float16>(v[1]), static_cast<_Float16>(v[2]),
                           static_cast<_Float16>(v[3])};
            *reinterpret_cast<v4h*>(buf + piece((tid >> 4) + 16u * i, (tid & 15u) >> 1) + 8u * (tid & 1u)) = h;
        }
    };

    float s[R][4];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) s[r][c] = 0.0f;
    const float one = 1.0f;
    load(0);
    stash(0, tile[0]);
    load(64u);
    for (uint32_t k0 = 0, buf = 0; k0 < g.k; k0 += 64u, buf ^= 1u) {
        __syncthreads();  // this chunk is in LDS; every wave is done with the other buffer
        stash(k0 + 64u, tile[buf ^ 1u]);
        load(k0 + 128u);
        const int8_t* t = tile[buf];
#pragma unroll
        for (uint32_t c8 = 0; c8 < 8; ++c8) {
            uint4 av[R], bv[4];
#pragma unroll
            for (int r = 0; r < R; ++r) av[r] = *reinterpret_cast<const uint4*>(t + piece(32u + 32u * r + ty, c8));
#pragma unroll
            for (int c = 0; c < 4; ++c) bv[c] = *reinterpret_cast<const uint4*>(t + piece(4u * tx + c, c8));
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                auto word = [p](const uint4& v) { return p == 0 ? v.x : p == 1 ? v.y : p == 2 ? v.z : v.w; };
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    uint32_t prod[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) prod[c] = mul_half2(word(av[r]), word(bv[c]));
                    add_product_pairs(s[r], prod, one);
                }
            }
        }
    }
    const bool vec = vector_rows<EPI>(g);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t m = row0 + 32u * r + ty;
        const uint32_t n = col0 + 4u * tx;
        if (m < g.m && n < g.n) store_f32<EPI>(g, m, n, s[r], vec);
    }
}

// out[p][c] = input[ic][iy][ix] of tap c = ic k^2 + ky k + kx of output pixel
// p (zero outside the image, max(., 0) first with relu); columns K .. ld-1 zero.
__global__ __launch_bounds__(256) void im2col_f32_kernel(const float* __restrict__ input, uint32_t width,
                                                         uint32_t height, uint32_t channels, uint32_t out_width,
                                                         uint32_t kernel, uint32_t stride, int32_t padding,
                                                         uint32_t relu, uint64_t rows, uint32_t columns, uint32_t ld,
                                                         float* __restrict__ out) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x;
    if (i >= rows * ld) return;
    const uint64_t p = i / ld;
    const uint32_t c = static_cast<uint32_t>(i - p * ld);
    float v = 0.0f;
    if (c < columns) {
        const uint32_t kk = kernel * kernel;
        const uint32_t ic = c / kk, t = c - ic * kk, ky = t / kernel, kx = t - ky * kernel;
        const uint32_t oy = static_cast<uint32_t>(p / out_width), ox = static_cast<uint32_t>(p - uint64_t(oy) * out_width);
        const int32_t iy = static_cast<int32_t>(oy * stride + ky) - padding;
        const int32_t ix = static_cast<int32_t>(ox * stride + kx) - padding;
        if (iy >= 0 && ix >= 0 && iy < static_cast<int32_t>(height) && ix < static_cast<int32_t>(width)) {
            v = input[(static_cast<uint64_t>(ic) * height + iy) * width + ix];
            if (relu) v = fmaxf(v, 0.0f);
        }
    }
    out[i] = v;
}

// A launch holds fewer than 2^32 threads in x; the tiles have at most 640.
constexpr uint32_t kMaxRowTiles = 1u << 22;

template <int BN, int BM>
dim3 tile_grid(const F32Params& g) {
    const uint32_t rows = ceil_div(g.m, BM), x = min(rows, kMaxRowTiles);
    return dim3(x, ceil_div(g.n, BN), ceil_div(rows, x));
}

template <int BN, int BM, int WN, int WM, int STAGES, bool HALF, int EPI>
void launch_tile(const F32Params& g, hipStream_t s) {
    constexpr size_t lds = static_cast<size_t>(STAGES) * (BN + BM) * 128u;
    static_assert(lds <= 64u * 1024u, "no larger dynamic LDS is asked for");
    dispatch(gemm_f32_kernel<BN, BM, WN, WM, STAGES, HALF, EPI>, tile_grid<BN, BM>(g), dim3(64 * WN * WM), lds, s, g);
}

constexpr uint32_t kCus = 256;  // MI355X

// The fp32 MFMA bounds the time (157 TFLOP/s) and every workgroup of these
// grids is resident at once, so it goes as the output area of the busiest CU
// over the rate the tile reaches on a full chip (5480 x 3072 x 1024, TFLOP/s):
// 93 / 103 / 108 / 109 in the order below, on operands that are rounded to
// binary16 on the way 76 / 91 / 100 / 107. us by that order at 1370 rows, N x
// K, float32: 4096 x 1024 with GELU 127 / 121 / 132 / 123, 2304 x 768 55 / 57 /
// 58 / 66, 768 x 768 24 / 26 / 24 / 26, 768 x 3072 86 / 97 / 79 / 91; binary16:
// 4096 x 1024 158 / 130 / 138 / 122, 2304 x 768 73 / 65 / 66 / 71, 768 x 768 32 /
// 32 / 30 / 30, 768 x 3072 115 / 114 / 107 / 108.
template <bool HALF, int EPI>
void launch_tiles(const F32Params& g, hipStream_t s) {
    struct Tile {
        uint32_t bn, bm, rate;
    };
    constexpr Tile tiles[] = {{32, 32, HALF ? 76 : 93}, {64, 32, HALF ? 91 : 103}, {64, 80, HALF ? 100 : 108},
                              {64, 96, HALF ? 107 : 109}};
    int best = -1;
    double least = 0.0;
    for (int i = 0; i < 4; ++i) {
        if (ceil_div(g.n, tiles[i].bn) > 65535u) continue;  // grid limit; f32_params checked it for 64 columns
        const uint64_t count = static_cast<uint64_t>(ceil_div(g.n, tiles[i].bn)) * ceil_div(g.m, tiles[i].bm);
        const double cost = static_cast<double>(ceil_div(count, kCus)) * (tiles[i].bn * tiles[i].bm) / tiles[i].rate;
        if (best < 0 || cost < least) best = i, least = cost;
    }
    switch (best) {
        case 0: launch_tile<32, 32, 2, 2, HALF ? 4 : 3, HALF, EPI>(g, s); break;
        case 1: launch_tile<64, 32, 2, 2, 2, HALF, EPI>(g, s); break;
        case 2: launch_tile<64, 80, 4, 1, 2, HALF, EPI>(g, s); break;
        default: launch_tile<64, 96, 2, 2, 2, HALF, EPI>(g, s); break;
    }
}

template <int BN, int BM, int WN, int WM, int BK, int EPI>
void launch_split_tile(const F32Params& g, hipStream_t s) {
    constexpr size_t lds = 2u * 3u * (BN + BM) * BK * 2u;
    if constexpr (lds > 64u * 1024u) {
        static const hipError_t attr =
            hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_split_kernel<BN, BM, WN, WM, BK, EPI>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        (void)attr;
    }
    dispatch(gemm_split_kernel<BN, BM, WN, WM, BK, EPI>, tile_grid<BN, BM>(g), dim3(64 * WN * WM), lds, s, g);
}

// The tile of the split changes no bits. Its grid takes the time of one tile on
// a CU and less for each further one on the busiest CU, which fills what the
// first leaves idle (us at K = 1024 in the table below; 32x32 goes in stages of
// 64 k). us by its order, then the best of launch_tiles<false>, which is ahead by up to a
// tenth on the smallest grids only: 31 x 1024 x 1024 12.0 / 20 / 25 / 29, 11.4; 253 x
// 1024 x 1024 13 / 21 / 26 / 30, 12; 253 x 768 x 3072 31 / 56 / 69 / 81, 30; 545 x
// 3072 x 768 36 / 28 / 39 / 25, 33; 1370 x 768 x 768 27 / 27 / 22 / 25, 24; 1370 x
// 768 x 3072 92 / 93 / 70 / 81, 79; 1370 x 1024 x 4096 150 / 130 / 178 / 109, 119;
// 1370 x 4096 x 1024 148 / 106 / 130 / 87, 118; 5477 x 1024 x 4096 537 / 375 / 446 /
// 319, 437. A sched_barrier between the splitting and the products cost 128x64 20%
// (99 / 82 at 1370 x 4096 x 1024).
template <int EPI>
void launch_split(const F32Params& g, hipStream_t s) {
    struct Tile {
        uint32_t bn, bm;
        double first, more;
    };
    constexpr Tile tiles[] = {{32, 32, 12.5, 5.5}, {64, 64, 21.5, 17.0}, {64, 80, 25.5, 24.5}, {128, 64, 30.5, 24.5}};
    int best = -1;
    double least = 0.0;
    for (int i = 0; i < 4; ++i) {
        if (ceil_div(g.n, tiles[i].bn) > 65535u) continue;  // grid limit; f32_params checked it for 64 columns
        const uint64_t count = static_cast<uint64_t>(ceil_div(g.n, tiles[i].bn)) * ceil_div(g.m, tiles[i].bm);
        const double cost = tiles[i].first + tiles[i].more * static_cast<double>(ceil_div(count, kCus) - 1u);
        if (best < 0 || cost < least) best = i, least = cost;
    }
    switch (best) {
        case 0: launch_split_tile<32, 32, 2, 2, 64, EPI>(g, s); break;
        case 1: launch_split_tile<64, 64, 4, 2, 32, EPI>(g, s); break;
        case 2: launch_split_tile<64, 80, 2, 5, 32, EPI>(g, s); break;
        default: launch_split_tile<128, 64, 4, 2, 32, EPI>(g, s); break;
    }
}

// Which arithmetic sums a row depends on K alone, so that a row's bits do not
// depend on the rows that come with it (an image's on its batch). Below K = 64
// the products the split leaves out can cost more than the sums of the fp32
// MFMA: 6.2e-8 against 3.3e-8 / 6.1e-8 / 7.7e-8 / 9.3e-8 at K = 8 / 32 / 48 / 64 for
// operands chosen for it.
constexpr uint32_t kSplitDepth = 64;

template <int EPI>
void launch(const F32Params& g, hipStream_t s) {
    if (g.half_operands)
        launch_tiles<true, EPI>(g, s);
    else if (g.k < kSplitDepth)
        launch_tiles<false, EPI>(g, s);
    else
        launch_split<EPI>(g, s);
}

template <int EPI>
void launch_h16p(const F32Params& g, hipStream_t s) {
    const uint32_t nt = ceil_div(g.n, 32);
    const dim3 cols(0, min(nt, kMaxGridY), ceil_div(nt, kMaxGridY));
    // Two rows a thread halve the LDS reads of a product, one row gives twice
    // the waves. us, two / one, by 64x32 tiles: 66 (1369 x 96 x 768) 34 / 20, 264
    // (1369 x 384 x 768) 49 / 40, 528 (1369 x 768 x 768) 68 / 60; between 696 and
    // 2080 within 6% either way by how the last round of workgroups falls (704,
    // 1369 x 1024 x 768, 68 / 70; 1032, 2738 x 768 x 768, 105 / 100; 1760, 3480 x
    // 1024 x 768, 145 / 152; 2064, 5476 x 768 x 768, 181 / 182); 2752 (5476 x 1024 x
    // 768) 220 / 232
    if (static_cast<uint64_t>(ceil_div(g.m, 64)) * nt >= 8u * kCus)
        dispatch(gemm_h16p_kernel<2, EPI>, dim3(ceil_div(g.m, 64), cols.y, cols.z), dim3(256), 0, s, g);
    else
        dispatch(gemm_h16p_kernel<1, EPI>, dim3(ceil_div(g.m, 32), cols.y, cols.z), dim3(256), 0, s, g);
}

// Checks a dav2_gemm_f32_args and fills the kernel parameters; false if the
// call is invalid.
bool f32_params(const dav2_gemm_f32_args* a, F32Params& g) {
    if (!a || !a->a || !a->b || !a->out || a->m == 0 || a->n == 0 || a->k == 0 || a->k % 4u || a->lda < a->k ||
        a->ldb < a->k || a->lda % 4u || a->ldb % 4u || (reinterpret_cast<uintptr_t>(a->a) & 15u) ||
        (reinterpret_cast<uintptr_t>(a->b) & 15u) || ceil_div(a->n, 64) > 65535u || a->half_operands > 1u)
        return false;
    const uint32_t e = a->epilogue;
    if (e != DAV2_GEMM_EPI_ROW && e != DAV2_GEMM_EPI_ROW_GELU && e != DAV2_GEMM_EPI_ROW_LAYERSCALE &&
        e != DAV2_GEMM_EPI_TRANSPOSED && e != DAV2_GEMM_EPI_CONVT)
        return false;
    if (e == DAV2_GEMM_EPI_ROW_LAYERSCALE && (!a->residual || !a->gamma)) return false;
    if (e == DAV2_GEMM_EPI_TRANSPOSED && a->out_row_stride < a->m + a->out_row_offset) return false;
    if (e == DAV2_GEMM_EPI_CONVT &&
        (a->convt_kernel == 0 || a->convt_channels == 0 || a->n != a->convt_kernel * a->convt_kernel * a->convt_channels ||
         a->m != a->convt_width * a->convt_height))
        return false;
    if ((a->relu_output || (a->residual && e != DAV2_GEMM_EPI_ROW_LAYERSCALE)) && e != DAV2_GEMM_EPI_TRANSPOSED)
        return false;
    g = F32Params{};
    g.a = a->a;
    g.lda = a->lda;
    g.b = a->b;
    g.ldb = a->ldb;
    g.m = a->m;
    g.n = a->n;
    g.k = a->k;
    g.bias = a->bias;
    g.out = a->out;
    g.out_row_offset = a->out_row_offset;
    g.out_row_stride = a->out_row_stride;
    g.residual = a->residual;
    g.gamma = a->gamma;
    g.relu_output = a->relu_output;
    g.convt_k = a->convt_kernel;
    g.convt_w = a->convt_width;
    g.convt_h = a->convt_height;
    g.convt_c = a->convt_channels;
    g.half_operands = a->half_operands;
    return true;
}

}  // namespace

extern "C" {

int dav2_hip_gemm_f32(const dav2_gemm_f32_args* a, void* stream) {
    F32Params g;
    if (!f32_params(a, g)) return hipErrorInvalidValue;
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (a->epilogue) {
        case DAV2_GEMM_EPI_ROW: launch<DAV2_GEMM_EPI_ROW>(g, s); break;
        case DAV2_GEMM_EPI_ROW_GELU: launch<DAV2_GEMM_EPI_ROW_GELU>(g, s); break;
        case DAV2_GEMM_EPI_ROW_LAYERSCALE: launch<DAV2_GEMM_EPI_ROW_LAYERSCALE>(g, s); break;
        case DAV2_GEMM_EPI_TRANSPOSED: launch<DAV2_GEMM_EPI_TRANSPOSED>(g, s); break;
        default: launch<DAV2_GEMM_EPI_CONVT>(g, s); break;
    }
    return hipGetLastError();
}

int dav2_hip_gemm_h16_products(const dav2_gemm_f32_args* a, void* stream) {
    F32Params g;
    if (!f32_params(a, g)) return hipErrorInvalidValue;
    const uint32_t e = a->epilogue;
    if ((e != DAV2_GEMM_EPI_ROW && e != DAV2_GEMM_EPI_TRANSPOSED && e != DAV2_GEMM_EPI_CONVT) || a->residual ||
        a->relu_output)
        return hipErrorInvalidValue;
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (e) {
        case DAV2_GEMM_EPI_ROW: launch_h16p<DAV2_GEMM_EPI_ROW>(g, s); break;
        case DAV2_GEMM_EPI_TRANSPOSED: launch_h16p<DAV2_GEMM_EPI_TRANSPOSED>(g, s); break;
        default: launch_h16p<DAV2_GEMM_EPI_CONVT>(g, s); break;
    }
    return hipGetLastError();
}

int dav2_hip_im2col_f32(const float* input, uint32_t input_width, uint32_t input_height, uint32_t input_channels,
                        uint32_t output_width, uint32_t output_height, uint32_t kernel, uint32_t stride,
                        int32_t padding, uint32_t relu, float* out, uint32_t ld, void* stream) {
    const uint64_t rows = static_cast<uint64_t>(output_width) * output_height;
    const uint64_t columns = static_cast<uint64_t>(input_channels) * kernel * kernel;
    if (rows == 0) return hipSuccess;
    if (!input || !out || kernel == 0 || stride == 0 || padding < 0 || ld < columns || columns >= (1u << 24) ||
        rows * ld >= (1ull << 38))
        return hipErrorInvalidValue;
    dispatch(im2col_f32_kernel, dim3(ceil_div(rows * ld, 256)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), input, input_width, input_height, input_channels,
                       output_width, kernel, stride, padding, relu, rows, static_cast<uint32_t>(columns), ld, out);
    return hipGetLastError();
}

}  // extern "C"
