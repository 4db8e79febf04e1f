// Implicit-GEMM fp32 convolutions of the fp32 / fp16 modes: 3x3 (padding 1)
// and 1x1, stride 1, CHW in and out, on v_mfma_f32_16x16x4_f32, with the
// residual and ReLU fusions of the DPT residual units. Reference:
// conv2d (src/operators.cpp:1528-1676), add.glsl, relu.glsl; it sums each dot
// product in its own order, so results are compared within a tolerance.
//
// A workgroup owns BP consecutive pixels of the flattened map and BN output
// channels and walks the input channels in blocks of CB. A stage holds, per
// input channel, the KS row segments its pixels read (BP + 2 pixels each,
// unpadded: the segment of tap row ky starts (ky - 1) W - 1 pixels from the
// first output pixel) and the CB KS KS weights of each output channel, copied
// straight from global memory into one of two LDS slots while the other one
// multiplies. Each MFMA sums one tap over four input channels: lane l takes
// the weight of output channel l % 16 and the pixel l % 16, both of input
// channel l / 16. A tap that falls outside the image has some other pixel's
// value in its segment; a lane mask per tap turns it into zero.
//
// Bound: the fp32 MFMA (157 TFLOP/s). No im2col matrix is written and read
// back (9 times the input: 101 MB each way for 148x148x128), which took half
// to two thirds of the time of im2col + GEMM. us, im2col + GEMM (which
// reads the matrix on the bfloat16 split) / this: 148x148 128 -> 128 129 / 70 (93
// TFLOP/s), 74x74 128 -> 128 45 / 25, 296x296 128 -> 64 458 / 130 (99), 518x518 64
// -> 32 684 / 103 (96), 37x37 1024 -> 256 154 / 124; 1x1 296x296 128 -> 128 92 / 44.
// Three or four slots measured the same as two; reading each step's operands
// where they are used, 5% slower.

#include <type_traits>

#include "common.h"
#include "dav2_hip.h"

namespace {

using namespace dav2k;

struct ConvF32Params {
    const float* input;
    const float* weight;
    const float* bias;
    const float* residual;
    float* out;
    uint32_t width, height, pixels, channels, out_channels;
    uint32_t relu_input, relu_output;
    uint32_t n_tiles;
};

template <int KS>
struct ConvF32Stage {
    static constexpr int kTaps = KS * KS;
    static constexpr int kCB = KS == 3 ? 4 : 16;    // input channels per stage
    static constexpr int kRow = kCB * kTaps;        // weight floats per output channel, whole 16-byte chunks
};

// Floats per input channel of a stage: KS segments of BP + KS - 1, rounded up
// so that four channels start 16 banks apart.
template <int KS, int BP>
constexpr int channel_floats() {
    constexpr int used = KS * (BP + KS - 1);
    return (used + 47) / 64 * 64 + 16;
}

template <int KS, int BN, int BP>
__global__ __launch_bounds__(256) void conv_f32_kernel(ConvF32Params g) {
    using Stage = ConvF32Stage<KS>;
    constexpr int WN = 2, WP = 2, NW = WN * WP, TN = BN / WN / 16, TP = BP / WP / 16;
    constexpr int CB = Stage::kCB, TAPS = Stage::kTaps, ROW = Stage::kRow;
    constexpr int GROUP = KS == 3 ? 3 : 4;  // k steps (one tap over four channels each) whose operands are read together
    constexpr int SEG = BP + KS - 1, CH = channel_floats<KS, BP>();
    constexpr int IN_FLOATS = CB * CH, W_FLOATS = (BN * ROW + 255) / 256 * 256;  // whole copies
    constexpr int IN_COPIES = IN_FLOATS / 64, W_COPIES = W_FLOATS / 256;  // 64 x 4 and 64 x 16 bytes each
    constexpr int IN_PER_WAVE = (IN_COPIES + NW - 1) / NW, W_PER_WAVE = (W_COPIES + NW - 1) / NW;
    static_assert(IN_FLOATS % 64 == 0 && ROW % 4 == 0, "whole copies");
    static_assert(TN * WN * 16 == BN && TP * WP * 16 == BP, "whole MFMA blocks per wave");
    __shared__ __attribute__((aligned(16))) float lds[2][W_FLOATS + IN_FLOATS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave / WP, wp = wave % WP, fr = lane & 15, fg = lane >> 4;
    // each XCD (workgroup id % 8) takes one contiguous run of tiles, the
    // output channels of one pixel tile next to each other
    const uint32_t xcd = blockIdx.x & 7u, base = gridDim.x >> 3, extra = gridDim.x & 7u;
    const uint32_t tile = xcd * base + min(xcd, extra) + (blockIdx.x >> 3);
    const uint32_t n0 = tile % g.n_tiles * BN, p0 = tile / g.n_tiles * BP;
    const uint64_t plane = g.pixels;
    const uint32_t inner = g.channels * TAPS;
    const int stages = static_cast<int>(g.channels / CB);

    // Copies of this wave (i NW + wave; past the last one it repeats it).
    // Pixels outside the map and output channels past the last read a valid
    // element in their place: the former are masked, the latter not stored.
    const float* in_src[IN_PER_WAVE];
    const float* w_src[W_PER_WAVE];
#pragma unroll
    for (int i = 0; i < IN_PER_WAVE; ++i) {
        const uint32_t idx = 64u * min(i * NW + wave, IN_COPIES - 1) + lane;
        const uint32_t ch = idx / CH, at = idx - ch * CH;
        const uint32_t ky = min(at / SEG, KS - 1u), col = min(at - ky * SEG, SEG - 1u);
        int64_t p = static_cast<int64_t>(p0) + col;
        if (KS == 3) p += (static_cast<int64_t>(ky) - 1) * g.width - 1;
        p = p < 0 ? 0 : p >= static_cast<int64_t>(plane) ? static_cast<int64_t>(plane) - 1 : p;
        in_src[i] = g.input + ch * plane + p;
    }
#pragma unroll
    for (int i = 0; i < W_PER_WAVE; ++i) {
        const uint32_t chunk = 64u * min(i * NW + wave, W_COPIES - 1) + lane;
        const uint32_t row = chunk / (ROW / 4), c4 = chunk - row * (ROW / 4);
        w_src[i] = g.weight + static_cast<uint64_t>(min(n0 + row, g.out_channels - 1)) * inner + 4u * c4;
    }
    auto issue = [&](int s) {
        float* slot = lds[s & 1];
#pragma unroll
        for (int i = 0; i < W_PER_WAVE; ++i) {
            copy16_to_lds(w_src[i], slot + 256 * min(i * NW + wave, W_COPIES - 1));
            w_src[i] += ROW;
        }
#pragma unroll
        for (int i = 0; i < IN_PER_WAVE; ++i) {
            copy4_to_lds(in_src[i], slot + W_FLOATS + 64 * min(i * NW + wave, IN_COPIES - 1));
            in_src[i] += CB * plane;
        }
    };

    // inside[t][j]: tap t of this lane's pixel of block j lies in the image
    bool inside[TAPS][TP];
#pragma unroll
    for (int j = 0; j < TP; ++j) {
        const uint32_t p = p0 + wp * (TP * 16) + j * 16 + fr;
        const uint32_t y = p / g.width, x = p - y * g.width;
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
            const int ky = t / KS, kx = t % KS;
            inside[t][j] = KS == 1 || ((ky != 0 || y > 0) && (ky != 2 || y + 1 < g.height) && (kx != 0 || x > 0) &&
                                       (kx != 2 || x + 1 < g.width));
        }
    }

    float bias[TN][4];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            bias[i][r] = g.bias ? g.bias[min(n0 + wn * (TN * 16) + i * 16 + 4 * fg + r, g.out_channels - 1)] : 0.0f;

    v4f acc[TN][TP];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TP; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    auto walk = [&](auto relu) {
        issue(0);
        for (int s = 0; s < stages; ++s) {
            // this wave's copies of the stage have landed and its reads of the
            // other slot have ended (vmcnt(0) lgkmcnt(0)); after the barrier every
            // wave's have, and the other slot is free
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0x0070);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < stages) issue(s + 1);
            const float* w = lds[s & 1] + (wn * (TN * 16) + fr) * ROW + fg * TAPS;
            const float* in = lds[s & 1] + W_FLOATS + fg * CH + wp * (TP * 16) + fr;
            // operands of a group of k steps are read while the group before
            // it multiplies
            float wf[2][GROUP][TN], pf[2][GROUP][TP];
            auto read = [&](int group) {
#pragma unroll
                for (int e = 0; e < GROUP; ++e) {
                    const int c = (group * GROUP + e) / TAPS, t = (group * GROUP + e) % TAPS;
#pragma unroll
                    for (int i = 0; i < TN; ++i) wf[group & 1][e][i] = w[i * 16 * ROW + c * 4 * TAPS + t];
#pragma unroll
                    for (int j = 0; j < TP; ++j)
                        pf[group & 1][e][j] = in[c * 4 * CH + (t / KS) * SEG + j * 16 + t % KS];
                }
            };
            read(0);
#pragma unroll
            for (int group = 0; group < CB / 4 * TAPS / GROUP; ++group) {
                if (group + 1 < CB / 4 * TAPS / GROUP) read(group + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < GROUP; ++e) {
                    const int t = (group * GROUP + e) % TAPS;
#pragma unroll
                    for (int j = 0; j < TP; ++j) {
                        const float v = pf[group & 1][e][j];
                        const float u = decltype(relu)::value ? fmaxf(v, 0.0f) : v;
                        const float p = inside[t][j] ? u : 0.0f;
#pragma unroll
                        for (int i = 0; i < TN; ++i)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[group & 1][e][i], p, acc[i][j], 0, 0, 0);
                    }
                }
            }
        }
    };
    if (g.relu_input) walk(std::true_type{});
    else walk(std::false_type{});

    // lane l holds output channels 4 (l / 16) + r of pixel l % 16; the
    // residual of a block's pixels is loaded before any of them is stored
    auto store = [&](auto residual) {
#pragma unroll
        for (int j = 0; j < TP; ++j) {
            const uint32_t p = p0 + wp * (TP * 16) + j * 16 + fr;
            float res[TN][4];
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t n = min(n0 + wn * (TN * 16) + i * 16 + 4 * fg + r, g.out_channels - 1);
                    res[i][r] = decltype(residual)::value ? g.residual[n * plane + min(p, g.pixels - 1)] : 0.0f;
                }
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t n = n0 + wn * (TN * 16) + i * 16 + 4 * fg + r;
                    float v = acc[i][j][r] + bias[i][r];
                    if (decltype(residual)::value) v = v + res[i][r];
                    if (g.relu_output) v = fmaxf(v, 0.0f);
                    if (p < g.pixels && n < g.out_channels) g.out[n * plane + p] = v;
                }
        }
    };
    if (g.residual) store(std::true_type{});
    else store(std::false_type{});
}

template <int KS, int BN, int BP>
void launch_conv(ConvF32Params g, hipStream_t s) {
    g.n_tiles = ceil_div(g.out_channels, BN);
    dispatch(conv_f32_kernel<KS, BN, BP>, dim3(g.n_tiles * ceil_div(g.pixels, BP)), dim3(256), 0, s, g);
}

constexpr uint32_t kCus = 256;  // MI355X

// The time goes as the tiles of the busiest CU times their area over the rate
// of the tile (92 / 82 / 72 TFLOP/s on a full chip), plus 0.45 of a tile for
// what one tile alone on a CU leaves idle. us for 64x64 / 32x64 / 32x32 tiles
// (output channels x pixels): 148x148 128 -> 128 78 / 84 / 87, 74x74 128 -> 128
// 36 / 32 / 27, 74x74 256 -> 256 99 / 83 / 90, 296x296 128 -> 64 141 / 149 /
// 172, 518x518 64 -> 32 202 / 120 / 133, 37x37 1024 -> 256 246 / 159 / 127.
template <int KS>
void launch_conv_tile(const ConvF32Params& g, hipStream_t s) {
    auto cost = [&](uint32_t bn, uint32_t bp, double rate) {
        const uint64_t tiles = static_cast<uint64_t>(ceil_div(g.out_channels, bn)) * ceil_div(g.pixels, bp);
        return (ceil_div(tiles, kCus) + 0.45) * bn * bp / rate;
    };
    const double c64 = cost(64, 64, 92.0), c32 = cost(32, 64, 82.0), c1 = cost(32, 32, 72.0);
    if (c64 <= c32 && c64 <= c1)
        launch_conv<KS, 64, 64>(g, s);
    else if (c32 <= c1)
        launch_conv<KS, 32, 64>(g, s);
    else
        launch_conv<KS, 32, 32>(g, s);
}

}  // namespace

extern "C" {

int dav2_hip_conv2d_f32_supported(uint32_t width, uint32_t height, uint32_t channels, uint32_t out_channels,
                                  uint32_t kernel, uint32_t stride, uint32_t padding) {
    const uint64_t pixels = static_cast<uint64_t>(width) * height;
    if (pixels == 0 || channels == 0 || out_channels == 0 || stride != 1u || pixels > (1u << 30) ||
        static_cast<uint64_t>(channels) * 9u > 0xffffffffull ||
        static_cast<uint64_t>(ceil_div(out_channels, 32)) * ceil_div(pixels, 32) > 0x7fffffffull)
        return 0;
    if (kernel == 3u && padding == 1u) return channels % ConvF32Stage<3>::kCB == 0;
    if (kernel == 1u && padding == 0u) return channels % ConvF32Stage<1>::kCB == 0;
    return 0;
}

int dav2_hip_conv2d_f32(const dav2_conv_f32_args* a, void* stream) {
    if (!a || !a->input || !a->weight || !a->out || (reinterpret_cast<uintptr_t>(a->weight) & 15u) ||
        (a->flags & ~static_cast<uint32_t>(DAV2_CONV_RELU_INPUT | DAV2_CONV_RELU_OUTPUT)) ||
        !dav2_hip_conv2d_f32_supported(a->width, a->height, a->channels, a->out_channels, a->kernel, 1, a->kernel / 2))
        return hipErrorInvalidValue;
    ConvF32Params g{};
    g.input = a->input;
    g.weight = a->weight;
    g.bias = a->bias;
    g.residual = a->residual;
    g.out = a->out;
    g.width = a->width;
    g.height = a->height;
    g.pixels = a->width * a->height;
    g.channels = a->channels;
    g.out_channels = a->out_channels;
    g.relu_input = a->flags & DAV2_CONV_RELU_INPUT;
    g.relu_output = a->flags & DAV2_CONV_RELU_OUTPUT;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (a->kernel == 3)
        launch_conv_tile<3>(g, s);
    else
        launch_conv_tile<1>(g, s);
    return hipGetLastError();
}

}  // extern "C"
