// Head-64 fp32 attention on the matrix cores, for the fp32 precision mode
// (FORCE_FP32): softmax((0.125 q) k^T) v on v_mfma_f32_16x16x4_f32, fused
// (flash_f32_kernel, the model's path), or as three public launchers over
// materialised scores, which no mode uses. fp32 products and sums, in the
// matrix core's order, so within tolerance of the reference
// (src/operators.cpp:1169-1208, bmm.glsl, softmax_lastdim.glsl), not bit for
// bit; the reference-order kernels are in attention_ref.hip.
//
// Layouts: qkv [batch*T][3*H*64]; scores [batch][H][T][T].

#include <type_traits>

#include "common.h"
#include "dav2_hip.h"

using namespace dav2k;

namespace {

// ---------------------------------------------------------------------------
// Scores. Workgroup tile 64 (queries) x 64 (keys), 4 waves in 2x2, each wave
// 32x32 = 2x2 MFMA blocks. Q and K tiles are staged through LDS with the
// 0.125 query scale applied first (bmm.glsl:57-63).
constexpr int kScoreStride = 65;  // padded LDS row length (floats)

__global__ __launch_bounds__(256) void attention_scores_kernel(const float* __restrict__ qkv,
                                                               float* __restrict__ scores, uint32_t tokens,
                                                               uint32_t heads) {
    constexpr int S = kScoreStride;
    __shared__ __attribute__((aligned(16))) float qt[64 * S];
    __shared__ __attribute__((aligned(16))) float kt[64 * S];

    const uint32_t bh = blockIdx.z;
    const uint32_t b = bh / heads, h = bh - b * heads;
    const uint32_t D = heads * 64u;
    const uint32_t i0 = blockIdx.y * 64u, j0 = blockIdx.x * 64u;
    const float* base = qkv + static_cast<uint64_t>(b) * tokens * 3u * D + h * 64u;
    const int tid = threadIdx.x;

    // 64 rows x 64 features = 1024 float4 loads per tile, 4 per thread.
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int c = tid + it * 256;
        const int r = c >> 4, f4 = (c & 15) * 4;
        float4 qv = make_float4(0.f, 0.f, 0.f, 0.f), kv = qv;
        if (i0 + r < tokens)
            qv = *reinterpret_cast<const float4*>(base + static_cast<uint64_t>(i0 + r) * 3u * D + f4);
        if (j0 + r < tokens)
            kv = *reinterpret_cast<const float4*>(base + static_cast<uint64_t>(j0 + r) * 3u * D + D + f4);
        float* qd = qt + r * S + f4;
        float* kd = kt + r * S + f4;
        qd[0] = qv.x * 0.125f;
        qd[1] = qv.y * 0.125f;
        qd[2] = qv.z * 0.125f;
        qd[3] = qv.w * 0.125f;
        kd[0] = kv.x;
        kd[1] = kv.y;
        kd[2] = kv.z;
        kd[3] = kv.w;
    }
    __syncthreads();

    const int lane = tid & 63, wave = tid >> 6;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    const int fr = lane & 15, g = lane >> 4;
    v4f acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[a][c] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) {
        float af[2], bf[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) af[a] = qt[(wr + a * 16 + fr) * S + ks * 4 + g];
#pragma unroll
        for (int c = 0; c < 2; ++c) bf[c] = kt[(wc + c * 16 + fr) * S + ks * 4 + g];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int c = 0; c < 2; ++c)
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[a], bf[c], acc[a][c], 0, 0, 0);
    }

    const uint64_t plane = static_cast<uint64_t>(bh) * tokens;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const uint32_t j = j0 + wc + c * 16 + fr;
            if (j >= tokens) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t i = i0 + wr + a * 16 + 4 * g + r;
                if (i < tokens) scores[(plane + i) * tokens + j] = acc[a][c][r];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Softmax over rows, in place, one wave per row, the whole row in VGPRs
// (CH values per lane; CH = 0 streams the row three times instead): max,
// e = exp(x - max), sum, e * (1 / max(sum, 1e-20)) as softmax_lastdim.glsl,
// with the lanes and the butterfly in this kernel's own order.
template <int CH>
__global__ __launch_bounds__(256) void softmax_kernel(void* data, uint64_t rows, uint32_t columns,
                                                      uint32_t row_stride) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t row = static_cast<uint64_t>(blockIdx.x) * 4u + (threadIdx.x >> 6);
    if (row >= rows) return;
    float* fr = static_cast<float*>(data) + row * row_stride;
    float v[CH > 0 ? CH : 1];
    float maximum = -3.402823466e+38f;
    if (CH > 0) {
#pragma unroll
        for (int j = 0; j < (CH > 0 ? CH : 1); ++j) {
            const uint32_t c = lane + 64u * j;
            v[j] = c < columns ? fr[c] : -3.402823466e+38f;
            maximum = fmaxf(maximum, v[j]);
        }
    } else {
        for (uint32_t c = lane; c < columns; c += 64u) maximum = fmaxf(maximum, fr[c]);
    }
    maximum = wave_max(maximum);
    float sum = 0.0f;
    if (CH > 0) {
#pragma unroll
        for (int j = 0; j < (CH > 0 ? CH : 1); ++j) {
            const uint32_t c = lane + 64u * j;
            if (c < columns) {
                const float e = expf(v[j] - maximum);
                sum = sum + e;
                v[j] = e;
            }
        }
    } else {
        for (uint32_t c = lane; c < columns; c += 64u) {
            const float e = expf(fr[c] - maximum);
            sum = sum + e;
            fr[c] = e;
        }
    }
    // Every lane holds a complete (though differently associated) sum.
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum = sum + __shfl_xor(sum, o, kWave);
    const float inverse = 1.0f / fmaxf(sum, 1.0e-20f);
    if (CH > 0) {
#pragma unroll
        for (int j = 0; j < (CH > 0 ? CH : 1); ++j) {
            const uint32_t c = lane + 64u * j;
            if (c < columns) fr[c] = v[j] * inverse;
        }
    } else {
        for (uint32_t c = lane; c < columns; c += 64u) fr[c] = fr[c] * inverse;
    }
}

// ---------------------------------------------------------------------------
// out = P v. Workgroup: 128 query rows x 64 features of one (batch, head);
// wave w owns rows 32w..32w+31 (2x4 MFMA blocks). The key axis advances 32
// tokens per step; P (128x32) and v^T (64x32) are staged through LDS.
__global__ __launch_bounds__(256) void attention_values_kernel(const float* __restrict__ probabilities,
                                                               const float* __restrict__ qkv,
                                                               float* __restrict__ out, uint32_t tokens,
                                                               uint32_t heads) {
    constexpr int PS = 33, VS = 33;  // padded LDS row lengths (floats)
    __shared__ __attribute__((aligned(16))) float pt[128 * PS];
    __shared__ __attribute__((aligned(16))) float vt[64 * VS];

    const uint32_t bh = blockIdx.z;
    const uint32_t b = bh / heads, h = bh - b * heads;
    const uint32_t D = heads * 64u;
    const uint32_t i0 = blockIdx.x * 128u;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int fr = lane & 15, g = lane >> 4;
    const float* vbase = qkv + static_cast<uint64_t>(b) * tokens * 3u * D + 2u * D + h * 64u;
    const uint64_t plane = static_cast<uint64_t>(bh) * tokens;

    v4f acc[2][4];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[a][c] = v4f{0.f, 0.f, 0.f, 0.f};

    for (uint32_t j0 = 0; j0 < tokens; j0 += 32u) {
        // Stage v[j0..j0+32)[0..64) transposed: 2048 values, 8 per thread.
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int c = tid + it * 256;  // 512 float4 chunks
            const int jr = c >> 4, f4 = (c & 15) * 4;
            float4 vv = make_float4(0.f, 0.f, 0.f, 0.f);
            if (j0 + jr < tokens)
                vv = *reinterpret_cast<const float4*>(vbase + static_cast<uint64_t>(j0 + jr) * 3u * D + f4);
            vt[(f4 + 0) * VS + jr] = vv.x;
            vt[(f4 + 1) * VS + jr] = vv.y;
            vt[(f4 + 2) * VS + jr] = vv.z;
            vt[(f4 + 3) * VS + jr] = vv.w;
        }
        // Stage P[i0..i0+128)[j0..j0+32): 4096 values, 16 per thread.
#pragma unroll
        for (int it = 0; it < 16; ++it) {
            const int c = tid + it * 256;
            const int ir = c >> 5, jc = c & 31;
            const uint32_t i = i0 + ir, j = j0 + jc;
            pt[ir * PS + jc] = i < tokens && j < tokens ? probabilities[(plane + i) * tokens + j] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            float af[2], bf[4];
#pragma unroll
            for (int a = 0; a < 2; ++a) af[a] = pt[(wave * 32 + a * 16 + fr) * PS + ks * 4 + g];
#pragma unroll
            for (int c = 0; c < 4; ++c) bf[c] = vt[(c * 16 + fr) * VS + ks * 4 + g];
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[a], bf[c], acc[a][c], 0, 0, 0);
        }
        __syncthreads();
    }

#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t i = i0 + wave * 32 + a * 16 + 4 * g + r;
            if (i >= tokens) continue;
            float* o = out + (static_cast<uint64_t>(b) * tokens + i) * D + h * 64u;
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c * 16 + fr] = acc[a][c][r];
        }
    }
}

// ---------------------------------------------------------------------------
// Fused: workgroup = 32 query rows of one (batch, head) as 2 groups of 16 x 2
// halves of the keys, one wave each. The two waves of a half share its key
// blocks of 32, copied straight into a ring of three 8 KB LDS slots (keys and
// values of a block take one slot each), 48 KB per workgroup, so three
// workgroups share a CU; one barrier per slot.
//
// Scores are computed transposed (keys x queries): lane l then holds, for
// query l % 16, keys 4 (l / 16) + r of a 16-key group in register r, which is
// the B operand of the value product over keys {4 g + r : g = 0..3} as it
// stands. Which feature a matrix row stands for is free as well: a lane's
// 16-byte piece of a key row serves four score MFMAs (features 16 s + 4 g + e),
// and its 16-byte piece of a value row four output blocks (features 4 m + c),
// so every operand is one ds_read_b128 and lane l ends with the 16 consecutive
// features 16 (l / 16) .. of its query.
//
// Softmax online, in fp32: running maximum per query, the sums rescaled only
// where a maximum grew, p = exp(s - max) / 2^n by expf; the division comes last.
// Bounded by the fp32 MFMA (157 TFLOP/s). ViT-B 686x518 (T = 1814, 12
// heads, 10.1 GFLOP): 495 us as scores + softmax + values (365 of them the
// values) -> 134 us (76 TFLOP/s); 1370 tokens, 16 heads 372 -> 103; 5477 tokens,
// 16 heads 3857 -> 1259 (98 TFLOP/s). Relative error against 64 bits 7.5e-7
// where the three kernels had 9.2e-7 (T = 1814).
constexpr uint32_t kFlashRows = 32, kFlashKeys = 32;
constexpr int kFlashSlot = kFlashKeys * 256;  // bytes
constexpr int kFlashSlots = 3;
constexpr float kLowest = -3.402823466e+38f;

// max / sum over the four lanes l, l ^ 16, l ^ 32, l ^ 48
template <typename Op>
DAV2_DEV float across_groups(float v, Op op) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = op(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void flash_f32_kernel(
    float* __restrict__ out, const float* __restrict__ qkv, uint32_t tokens, uint32_t heads, uint32_t row_blocks) {
    __shared__ __attribute__((aligned(16))) int8_t smem[2 * kFlashSlots * kFlashSlot];  // [key half][slot]
    // XCD-banded order: each of the 8 XCDs takes a contiguous run of (head,
    // row block) items, so a head's keys and values stay in one L2.
    const uint32_t total = gridDim.x, xcd = blockIdx.x & 7u, per = total >> 3, extra = total & 7u;
    const uint32_t work = xcd * per + min(xcd, extra) + (blockIdx.x >> 3);
    const uint32_t bh = work / row_blocks, rb = work - bh * row_blocks;
    const uint32_t b = bh / heads, h = bh - b * heads;
    const uint32_t D = heads * 64u;
    const uint64_t ld = 3u * static_cast<uint64_t>(D);
    const float* base = qkv + b * ld * tokens + h * 64u;
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t group = wave & 1u, half = wave >> 1;
    const uint32_t fr = lane & 15u, fg = lane >> 4;
    const uint32_t blocks = (tokens + kFlashKeys - 1u) / kFlashKeys;
    const uint32_t mine = (blocks + 1u) >> 1;  // blocks per half; past the last one every key is masked
    const uint32_t first = half * mine;
    int8_t* const ring = smem + half * kFlashSlots * kFlashSlot;

    // Item 2 i holds the keys of the half's block i, item 2 i + 1 its values;
    // item n sits in slot n % 3. Copy c of a slot (1 KiB) is rows 4 c .. + 3,
    // lane l row + l / 16, chunk l % 16; the wave's group takes copies
    // 4 group .. + 3. Key rows are stored with chunk c at c ^ (row % 16), so
    // that the 16 rows of an operand read fall on different banks. Rows past
    // the last token repeat it.
    auto issue = [&](uint32_t item) {
        const uint32_t j0 = (first + (item >> 1)) * kFlashKeys;
        const bool values = item & 1u;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t row = 16u * group + 4u * i + fg;
            const uint32_t chunk = values ? fr : fr ^ (row & 15u);
            copy16_to_lds(base + min(j0 + row, tokens - 1u) * ld + (values ? 2u * D : D) + 4u * chunk,
                          ring + (item % kFlashSlots) * kFlashSlot + (4u * group + i) * 1024u);
        }
    };

    // B operand of the score MFMAs: 0.125 q (bmm.glsl:57-63); rows past the
    // last token compute on its copy and are not stored.
    const uint32_t query = rb * kFlashRows + group * 16u + fr;
    v4f q[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        q[s] = *reinterpret_cast<const v4f*>(base + min(query, tokens - 1u) * ld + 16 * s + 4u * fg);
#pragma unroll
        for (int e = 0; e < 4; ++e) q[s][e] *= 0.125f;
    }

    v4f acc[4];  // output block c, register r: feature 16 fg + 4 r + c
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = v4f{0.f, 0.f, 0.f, 0.f};
    float maximum = kLowest, sum = 0.0f;  // sum: this lane's keys only
    // Weights are exp / 2^n, 2^n >= tokens: no sum of weighted values passes the
    // largest value (T = 5477, 16 heads 1247 -> 1256 us; the same bits elsewhere).
    const float share = __uint_as_float((95u + __clz(tokens - 1u)) << 23);
    v4f p[2];

    issue(0);
    issue(1);
    // Slot of item n free for item n + 2: its readers have passed the barrier
    // of item n + 1. The wait leaves the next item's four copies in flight.
    auto next = [&](uint32_t item) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        if (item + 1u < 2u * mine) DAV2_WAIT_VMCNT(4);
        else DAV2_WAIT_VMCNT(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (item + 2u < 2u * mine) issue(item + 2u);
    };
    auto scores = [&](uint32_t i, auto masked) {
        const int8_t* kt = ring + ((2u * i) % kFlashSlots) * kFlashSlot;
        v4f kf[2][4];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                kf[t][s] = *reinterpret_cast<const v4f*>(kt + (16 * t + fr) * 256u + (((4 * s + fg) ^ fr) << 4));
#pragma unroll
        for (int t = 0; t < 2; ++t) p[t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    p[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][s][e], q[s][e], p[t], 0, 0, 0);
        if constexpr (decltype(masked)::value) {
            const uint32_t j0 = (first + i) * kFlashKeys + 4u * fg;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (j0 + 16 * t + r >= tokens) p[t][r] = -__builtin_inff();
        }
        float top = maximum;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) top = fmaxf(top, p[t][r]);
        top = across_groups(top, [](float x, float y) { return fmaxf(x, y); });
        if (__any(top > maximum)) {
            const float scale = expf(maximum - top);
            sum *= scale;
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[c][r] *= scale;
            maximum = top;
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) p[t][r] = expf(p[t][r] - maximum) * share;
        sum += ((p[0][0] + p[0][1]) + (p[0][2] + p[0][3])) + ((p[1][0] + p[1][1]) + (p[1][2] + p[1][3]));
    };
    auto values = [&](uint32_t i, auto masked) {
        const int8_t* vt = ring + ((2u * i + 1u) % kFlashSlots) * kFlashSlot;
        v4f vf[2][4];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t row = 16u * t + 4u * fg + r;
                vf[t][r] = *reinterpret_cast<const v4f*>(vt + row * 256u + fr * 16u);
                // a masked key's weight is 0; its value must not be infinite or NaN
                if constexpr (decltype(masked)::value)
                    if ((first + i) * kFlashKeys + row >= tokens) vf[t][r] = v4f{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[t][r][c], p[t][r], acc[c], 0, 0, 0);
    };
    const uint32_t whole = min(mine, max(tokens / kFlashKeys, first) - first);  // blocks without a masked key
    for (uint32_t i = 0; i < mine; ++i) {
        next(2u * i);
        if (i < whole) scores(i, std::false_type{});
        else scores(i, std::true_type{});
        next(2u * i + 1u);
        if (i < whole) values(i, std::false_type{});
        else values(i, std::true_type{});
    }

    // The second half's maxima, sums and outputs through LDS to the first.
    sum = across_groups(sum, [](float x, float y) { return x + y; });
    __syncthreads();
    float* const hand = reinterpret_cast<float*>(smem) + group * 18u * 64u + lane;  // [18][lane]
    if (half == 1u) {
        hand[0] = maximum;
        hand[64] = sum;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) hand[(2 + 4 * c + r) * 64] = acc[c][r];
    }
    __syncthreads();
    if (half == 1u || query >= tokens) return;
    const float other = hand[0], top = fmaxf(maximum, other);
    const float s0 = expf(maximum - top), s1 = expf(other - top);
    const float inverse = 1.0f / fmaxf(sum * s0 + hand[64] * s1, 1.0e-20f);
    float* o = out + (static_cast<uint64_t>(b) * tokens + query) * D + h * 64u + 16u * fg;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
            v[c] = (acc[c][r] * s0 + hand[(2 + 4 * c + r) * 64] * s1) * inverse;
        *reinterpret_cast<float4*>(o + 4 * r) = make_float4(v[0], v[1], v[2], v[3]);
    }
}

void launch_softmax(void* data, uint64_t rows, uint32_t columns, uint32_t stride, hipStream_t s) {
    const unsigned grid = ceil_div(rows, 4);
    const uint32_t ch = (columns + 63u) / 64u;
#define DAV2_SM_CASE(N) \
    dispatch((softmax_kernel<N>), dim3(grid), dim3(256), 0, s, data, rows, columns, stride)
    if (ch <= 4) DAV2_SM_CASE(4);
    else if (ch <= 8) DAV2_SM_CASE(8);
    else if (ch <= 16) DAV2_SM_CASE(16);
    else if (ch <= 24) DAV2_SM_CASE(24);
    else if (ch <= 32) DAV2_SM_CASE(32);
    else if (ch <= 48) DAV2_SM_CASE(48);
    else if (ch <= 64) DAV2_SM_CASE(64);
    else if (ch <= 96) DAV2_SM_CASE(96);
    else DAV2_SM_CASE(0);
#undef DAV2_SM_CASE
}

}  // namespace

extern "C" {

// fp16 != 0 is rejected: binary16 attention is dav2_hip_attention_ref_*.
int dav2_hip_attention_scores(void* scores, const float* qkv, uint32_t tokens, uint32_t heads,
                              uint32_t batch, int fp16, void* stream) {
    if (fp16) return hipErrorInvalidValue;
    if (tokens == 0 || heads == 0 || batch == 0) return hipSuccess;
    if (!scores || !qkv || (reinterpret_cast<uintptr_t>(qkv) & 15) || heads > 65535u / batch)
        return hipErrorInvalidValue;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid(ceil_div(tokens, 64), ceil_div(tokens, 64), heads * batch);
    dispatch(attention_scores_kernel, grid, dim3(256), 0, s, qkv, static_cast<float*>(scores), tokens,
                       heads);
    return hipGetLastError();
}

int dav2_hip_softmax_rows(void* scores, uint64_t rows, uint32_t columns, uint32_t row_stride, int fp16,
                          void* stream) {
    if (fp16) return hipErrorInvalidValue;
    if (rows == 0) return hipSuccess;
    if (!scores || columns == 0 || row_stride < columns) return hipErrorInvalidValue;
    launch_softmax(scores, rows, columns, row_stride, static_cast<hipStream_t>(stream));
    return hipGetLastError();
}

int dav2_hip_attention_values(float* out, const void* probabilities, const float* qkv, uint32_t tokens,
                              uint32_t heads, uint32_t batch, int fp16, void* stream) {
    if (fp16) return hipErrorInvalidValue;
    if (tokens == 0 || heads == 0 || batch == 0) return hipSuccess;
    if (!out || !probabilities || !qkv || (reinterpret_cast<uintptr_t>(qkv) & 15) || heads > 65535u / batch)
        return hipErrorInvalidValue;
    const dim3 grid(ceil_div(tokens, 128), 1, heads * batch);
    dispatch(attention_values_kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const float*>(probabilities), qkv, out, tokens, heads);
    return hipGetLastError();
}

int dav2_hip_attention_f32(float* out, const float* qkv, uint32_t tokens, uint32_t heads, uint32_t batch,
                           void* stream) {
    if (tokens == 0 || heads == 0 || batch == 0) return hipSuccess;
    if (!out || !qkv || ((reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(out)) & 15))
        return hipErrorInvalidValue;
    const uint32_t row_blocks = ceil_div(tokens, kFlashRows);
    const uint64_t items = static_cast<uint64_t>(row_blocks) * heads * batch;
    if (items > 0x7fffffffull || tokens > 0x7fffffffu) return hipErrorInvalidValue;
    dispatch(flash_f32_kernel, dim3(static_cast<uint32_t>(items)), dim3(256), 0, static_cast<hipStream_t>(stream),
             out, qkv, tokens, heads, row_blocks);
    return hipGetLastError();
}

uint64_t dav2_hip_attention_scratch_bytes(uint32_t tokens, uint32_t heads, uint32_t batch, int fp16) {
    if (fp16) return 0;
    return static_cast<uint64_t>(batch) * heads * tokens * tokens * sizeof(float);
}

}  // extern "C"
