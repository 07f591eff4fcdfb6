// 3x3 convolution with padding 1 on planar images in three-piece bf16 arithmetic (split_mfma.h):
//   out[n][co][y][x] = act^count(sum over ci, ky, kx of in[n][ci][y + ky - 1][x + kx - 1] * w[co][ci][ky][kx] + bias[co])
// (the three middle convolutions of the down-scaler, network/model.py:13-25 with ConvResBlock2D, network/layer.py, and
// with the weights turned round their data gradients), and the weight gradient (conv3x3_wgrad_k).
#include <type_traits>
#include <utility>
#include "spgt_device.h"
#include "spgt_host.h"
#include "split_mfma.h"

namespace spgt {

namespace {

constexpr int kConvCols = 32, kHaloCols = kConvCols + 2;           // output pixels of a workgroup: ROWS x 32
template <int ROWS>
constexpr int kHalo = (ROWS + 2) * kHaloCols;
constexpr int kConvOut = 48;                                        // output channels of a workgroup
constexpr int kStepUnits = 3 * 3 * 64;                              // operands of one step: channel block, piece, lane

// Steps of 32 products that `channels` input channels take: chunks of 32 channels are 36 (tap, eight channels) units in
// 9 steps of four, what is left is 9 * ceil(rest / 8) units.
__host__ __device__ inline int conv_steps(int channels) {
    return channels / 32 * 9 + (9 * ((channels % 32 + 7) / 8) + 3) / 4;
}

}  // namespace

// The weights as MFMA operands [output channel group][step][block of 16][piece][lane]: lane l of step s of a chunk with CG
// groups of eight channels holds unit u = 4 s + l / 16, which is tap u / CG, channels 8 (u % CG) .. + 7 of the chunk, of
// output channel l % 16.  TURNED: the weights of the data gradient, in and out exchanged and the taps reversed.
__global__ __launch_bounds__(256) void conv3x3_pack_k(const float* __restrict__ w, v4u* __restrict__ pack, int cin,
                                                      int cout, int turned, int steps, int total) {
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int lane = idx & 63;
    const int block = (idx >> 6) % 3;
    const int gs = (idx >> 6) / 3;
    const int step = gs % steps, group = gs / steps;
    const int full = cin / 32;
    const int chunk = min(step / 9, full);
    const int cg = chunk < full ? 4 : (cin % 32 + 7) / 8;
    const int u = 4 * (step - 9 * chunk) + (lane >> 4);
    const int tap = u / cg, c0 = 32 * chunk + 8 * (u % cg);
    const int co = kConvOut * group + 16 * block + (lane & 15);
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int c = c0 + j;
        const bool ok = tap < 9 && co < cout && c < cin;
        v[j] = !ok ? 0.f : turned ? w[((int64_t)c * cout + co) * 9 + 8 - tap] : w[((int64_t)co * cin + c) * 9 + tap];
    }
    const Split8 p = split8(v);
    v4u* o = pack + ((int64_t)gs * 3 + block) * 3 * 64 + lane;
    o[0] = __builtin_bit_cast(v4u, p.hi);
    o[64] = __builtin_bit_cast(v4u, p.mid);
    o[128] = __builtin_bit_cast(v4u, p.lo);
}

// A workgroup forms 8 x 32 (small inputs: 2 x 32) pixels of 48 output channels, 32 input channels at a time: its threads
// read the pixels with their halo, eight channels of one pixel per thread, and put the split values into LDS as 16-byte units
// [piece][eight channels][pixel].  A unit is what a lane of an MFMA 16x16x32 holds, so the nine taps read the
// same units at shifted pixels, and a step's four quarters of 32 products may be different taps.  Wave w takes a quarter
// of the pixels for all 48 channels; the weights stream from L2, a step of 72 MFMAs ahead.  Two workgroups share a CU,
// one's loads beside the other's products.
// What bounds it is the matrix pipe: 128 -> 42 channels take 36 steps of 1152 cycles for 256 pixels, against 44 KB of
// input per 32 channels and tile.  Four images of 363 x 364, packing included: 128 -> 42 channels 753 -> 309 us, 42 ->
// 44 275 -> 123, 42 -> 128 turned 584 -> 367; of 122 x 123: 93 -> 50, 40 -> 24, 40 -> 24; one image of 30 x 31, 42 ->
// 42 channels: 18 -> 13, 128 -> 42 17.5 -> 22.6 on the device and 34 -> 26 as a call (before: the convolution library's
// fp32 kernels); the error against 64-bit sums 2.2 .. 3.6e-7 -> 1.1 .. 2.0e-7 of the norm.  With a branch around each
// load 128 -> 42 took 603 us.
// A wave with sums that are not finite forms them again with fp32 MFMAs.
// grid (tiles * output channel groups, rounded up to a multiple of 8), block 256
template <int ROWS>
__global__ __launch_bounds__(256, 2) void conv3x3_split_k(const float* __restrict__ in, const v8bf* __restrict__ pack,
                                                          const float* __restrict__ w, const float* __restrict__ bias,
                                                          float* __restrict__ out, int cin, int cout, int H, int W,
                                                          int turned, int act, int act_count, int tx, int ty, int groups,
                                                          int steps, int total) {
    extern __shared__ __align__(16) v8bf tile[];  // [3][4][HALO]
    constexpr int HALO = kHalo<ROWS>, PLANE = 4 * HALO;
    constexpr int NB = ROWS / 2;  // blocks of 16 pixels of a wave: block i of the tile is row i / 2, columns 16 (i % 2) ..
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, quad = lane >> 4;
    // neighbouring tiles on one XCD: they share halo pixels
    const int per_xcd = gridDim.x >> 3;
    int id = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (id >= total) return;
    const int group = id % groups;
    id /= groups;
    const int x0 = id % tx * kConvCols;
    id /= tx;
    const int y0 = id % ty * ROWS;
    const int n = id / ty;
    const int64_t plane = (int64_t)H * W;
    const float* const src = in + (int64_t)n * cin * plane;  // N * channels alone may pass 2^31
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(src), 0, (uint32_t)cin * (uint32_t)plane * 4u, 0x00027000);

    v4f big[NB][3], small[NB][3];  // [16 pixels][16 channels]
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int c = 0; c < 3; ++c) big[b][c] = small[b][c] = v4f{0.f, 0.f, 0.f, 0.f};

    const v8bf* wp = pack + (int64_t)group * steps * kStepUnits + lane;
    v8bf wa[3][3], wb[3][3];
    auto load_w = [&](v8bf (&v)[3][3], int step) {
        const v8bf* s = wp + (int64_t)min(step, steps - 1) * kStepUnits;
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int p = 0; p < 3; ++p) v[c][p] = s[(c * 3 + p) * 64];
    };
    // products of step s of a chunk with cg groups of eight channels
    auto block_row = [&](int b) { return (NB * wave + b) >> 1; };
    auto block_col = [&](int b) { return 16 * ((NB * wave + b) & 1); };
    const int pixel = block_row(0) * kHaloCols + block_col(0) + l16;
    auto multiply = [&](const v8bf (&v)[3][3], int s, int cg) {
        const int u = min(4 * s + quad, 9 * cg - 1);  // past the last unit the weights are zeros
        const int tap = cg == 4 ? u >> 2 : cg == 2 ? u >> 1 : cg == 1 ? u : (u * 86) >> 8;
        const int dy = (tap * 11) >> 5;
        const v8bf* t = tile + (u - tap * cg) * HALO + pixel + dy * kHaloCols + tap - 3 * dy;
        v8bf xv[2][3];
        auto read = [&](v8bf (&x)[3], int b) {
#pragma unroll
            for (int p = 0; p < 3; ++p) x[p] = t[p * PLANE + (b >> 1) * kHaloCols + 16 * (b & 1)];
        };
        read(xv[0], 0);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (b + 1 < NB) read(xv[(b + 1) & 1], b + 1);  // under this block's MFMAs
            __builtin_amdgcn_sched_barrier(0);
            auto mul = [&](v4f (&acc)[3], int q, int p) {
#pragma unroll
                for (int c = 0; c < 3; ++c) acc[c] = mfma16_bf16(v[c][q], xv[b & 1][p], acc[c]);
            };
            mul(small[b], 2, 0);
            mul(big[b], 0, 0);
            mul(small[b], 0, 2);
            mul(small[b], 1, 1);
            mul(small[b], 1, 0);
            mul(small[b], 0, 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    load_w(wa, 0);
    for (int c0 = 0, step = 0; c0 < cin; c0 += 32) {
        const int cg = min(4, (cin - c0 + 7) / 8);
        if (c0 > 0) __syncthreads();  // the previous chunk consumed
        constexpr int TRIPS = (4 * HALO + 255) / 256;
        float v[TRIPS][8];
#pragma unroll
        for (int i = 0; i < TRIPS; ++i) {
            const int e = threadIdx.x + 256 * i;
            const int g = e / HALO, px = e - g * HALO;
            const int ry = px / kHaloCols, rx = px - ry * kHaloCols;
            const int y = y0 + ry - 1, x = x0 + rx - 1;
            const bool ok = g < cg && y >= 0 && y < H && x >= 0 && x < W;
            // pixels outside the image and channels past the last lie outside the buffer and read as zeros: straight-line
            // code, every load of the chunk is requested before the first is used
            const uint32_t off = ok ? 4u * ((uint32_t)(c0 + 8 * g) * (uint32_t)plane + (uint32_t)(y * W + x)) : 0x80000000u;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                v[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off + 4u * j * (uint32_t)plane, 0, 0));
        }
#pragma unroll
        for (int i = 0; i < TRIPS; ++i) {
            const int e = threadIdx.x + 256 * i;
            if (e < cg * HALO) {
                const Split8 s = split8(v[i]);
                tile[e] = s.hi;
                tile[e + PLANE] = s.mid;
                tile[e + 2 * PLANE] = s.lo;
            }
        }
        __syncthreads();
        const int chunk_steps = (9 * cg + 3) / 4;
        int s = 0;
        for (; s + 1 < chunk_steps; s += 2, step += 2) {
            load_w(wb, step + 1);
            multiply(wa, s, cg);
            load_w(wa, step + 2);
            multiply(wb, s + 1, cg);
        }
        if (s < chunk_steps) {  // an odd count: the next chunk starts with the operands in wa again
            load_w(wb, step + 1);
            multiply(wa, s, cg);
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int p = 0; p < 3; ++p) wa[c][p] = wb[c][p];
            ++step;
        }
    }

    bool bad = false;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
        for (int c = 0; c < 3; ++c) big[b][c] += small[b][c];
        bad = bad || not_finite(big[b]);
    }
    const int col = x0 + l16;
    float unscale = kSplitUnscale;
    if (__builtin_expect(__any(bad), 0)) {
        unscale = 1.f;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int c = 0; c < 3; ++c) big[b][c] = v4f{0.f, 0.f, 0.f, 0.f};
            for (int tap = 0; tap < 9; ++tap) {
                const int y = y0 + block_row(b) + tap / 3 - 1, x = col + block_col(b) + tap % 3 - 1;
                const bool ok = y >= 0 && y < H && x >= 0 && x < W;
                for (int c4 = 0; c4 < cin; c4 += 4) {
                    const int ci = c4 + quad;
                    const float xv = ok && ci < cin ? src[ci * plane + (int64_t)y * W + x] : 0.f;
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const int co = kConvOut * group + 16 * c + l16;
                        float wv = 0.f;
                        if (ci < cin && co < cout)
                            wv = turned ? w[((int64_t)ci * cout + co) * 9 + 8 - tap] : w[((int64_t)co * cin + ci) * 9 + tap];
                        big[b][c] = mfma16(wv, xv, big[b][c]);
                    }
                }
            }
        }
    }
    float* const dst = out + (int64_t)n * cout * plane;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const int co = kConvOut * group + 16 * c + 4 * quad;
        float b4[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) b4[r] = bias && co + r < cout ? bias[co + r] : 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int y = y0 + block_row(b), x = col + block_col(b);
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = fmaf(big[b][c][r], unscale, b4[r]);
            for (int i = 0; i < act_count; ++i) activate_all(v, act);
            if (y < H && x < W) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (co + r < cout) dst[(co + r) * plane + (int64_t)y * W + x] = v[r];
            }
        }
    }
}

}  // namespace spgt

using namespace spgt;

static int64_t conv_workgroups(int N, int out_channels, int H, int W, int rows) {
    return (int64_t)N * ceil_div(W, kConvCols) * ceil_div(H, rows) * ceil_div(out_channels, kConvOut);
}

// Workgroups of one launch: a grid counts its work-items in 32 bits.  Larger batches go out in several launches.
constexpr int64_t kConvMaxWorkgroups = ((int64_t)1 << 24) - 8;

extern "C" int spgt_conv3x3_supported(int N, int in_channels, int out_channels, int H, int W) {
    if (N <= 0 || H <= 0 || W <= 0 || spgt_conv3x3_workspace_bytes(in_channels, out_channels) == 0) return 0;
    return (int64_t)H * W <= INT32_MAX && (int64_t)in_channels * H * W <= (int64_t)1 << 28 &&
           conv_workgroups(1, out_channels, H, W, 8) <= kConvMaxWorkgroups;
}

static bool conv_few(int N, int out_channels, int H, int W) {
    return conv_workgroups(N, out_channels, H, W, 8) < device_cu_count() * 3 / 4;
}

// Microseconds on the device, the convolution library's fp32 kernels and this one (packing included).  Where tiles of
// eight rows fill the chip this one is the quicker up to 256 input channels; with more, whose serial chains of steps
// are longer, from one and a half workgroups per compute unit on (384 -> 64, 192 workgroups: 102 and 110; 512 -> 64 125
// and 145; 512 -> 512, 576 of them 750 and 535).  Where they do not, a chain's length decides: up to 64 input channels
// this one is the quicker (42 -> 42 of 30 x 31 17.8 and 13.1); up to 128 it takes longer on the device (128 -> 42 of 30
// x 31 17.5 and 22.6) but less than the 34 us or more that the library's call takes on the host, while two workgroups
// of two rows per compute unit hold it (128 -> 512 of 16 x 8 x 9, 704 of them: 35 and 49); 256 -> 64 of 30 x 31 take 23
// and 39.  with_gradient: a training step through the convolution.  From 2^28 products per tap or 12 Mi values on the
// kernels decide it (forward and backward: 64 -> 64 of 16 x 64 x 65 232 and 169, 64 -> 1 of 4 x 256 x 257 293 and 166);
// below, the host's time does, alike on both sides (42 -> 42 of 4 x 90 x 91 166 and 165, of 30 x 31 174 and 168), and those
// stay with the library.
extern "C" int spgt_conv3x3_pays(int N, int in_channels, int out_channels, int H, int W, int with_gradient) {
    if (!spgt_conv3x3_supported(N, in_channels, out_channels, H, W)) return 0;
    const int64_t pixels = (int64_t)N * H * W, cus = device_cu_count();
    if (with_gradient && pixels * (in_channels + out_channels) < (int64_t)12 << 20 &&
        (double)pixels * in_channels * out_channels < (double)(1 << 28))
        return 0;
    if (!conv_few(N, out_channels, H, W))
        return in_channels <= 256 || 2 * conv_workgroups(N, out_channels, H, W, 8) >= 3 * cus;
    return in_channels <= 64 || (in_channels <= 128 && conv_workgroups(N, out_channels, H, W, 2) <= 2 * cus);
}

extern "C" size_t spgt_conv3x3_workspace_bytes(int in_channels, int out_channels) {
    if (in_channels <= 0 || out_channels <= 0 || in_channels > 4096 || out_channels > 4096) return 0;
    return (size_t)ceil_div(out_channels, kConvOut) * conv_steps(in_channels) * kStepUnits * 16;
}

extern "C" int spgt_conv3x3_forward(const float* input, const float* weight, const float* bias, float* out, int N,
                                    int in_channels, int out_channels, int H, int W, int turned, int activation,
                                    int act_count, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    if (!input || !weight || !out) return fail(SPGT_ERR_INVALID_ARGUMENT, "conv3x3_forward: null pointer argument");
    const size_t need = spgt_conv3x3_workspace_bytes(in_channels, out_channels);
    if (N <= 0 || H <= 0 || W <= 0 || need == 0)
        return fail(SPGT_ERR_INVALID_ARGUMENT, "conv3x3_forward: sizes must be positive, at most 4096 channels");
    if (activation != SPGT_ACT_NONE && activation != SPGT_ACT_RELU && activation != SPGT_ACT_SILU)
        return fail(SPGT_ERR_INVALID_ARGUMENT, "conv3x3_forward: unknown activation");
    if (act_count < 0 || (turned != 0 && turned != 1))
        return fail(SPGT_ERR_INVALID_ARGUMENT, "conv3x3_forward: negative act_count, or turned neither 0 nor 1");
    if (!aligned4(input) || !aligned4(weight) || !aligned4(out) || (bias && !aligned4(bias)))
        return fail(SPGT_ERR_INVALID_ARGUMENT, "conv3x3_forward: misaligned pointer");
    if (input == out) return fail(SPGT_ERR_INVALID_ARGUMENT, "conv3x3_forward: out must not alias the input");
    if (!workspace || !aligned16(workspace) || workspace_bytes < need)
        return fail(SPGT_ERR_WORKSPACE, "conv3x3_forward: workspace missing, misaligned or too small");
    const int steps = conv_steps(in_channels), groups = ceil_div(out_channels, kConvOut);
    // tiles of two rows while those of eight would leave a quarter of the compute units idle: 8 workgroups of eight rows
    // 41 us against 22, 128 of them 44 against 36; 144 and 192 equal; 256 of them 48 against 58
    const bool few = conv_few(N, out_channels, H, W);
    const int tx = ceil_div(W, kConvCols), ty = ceil_div(H, few ? 2 : 8);
    const int64_t per_image = (int64_t)tx * ty * groups;
    if (per_image > kConvMaxWorkgroups) return fail(SPGT_ERR_INVALID_ARGUMENT, "conv3x3_forward: too many pixels");
    if ((int64_t)H * W > INT32_MAX || (int64_t)in_channels * H * W > (int64_t)1 << 28)
        return fail(SPGT_ERR_INVALID_ARGUMENT, "conv3x3_forward: an image of 1 GB at most");
    const int operands = groups * steps * 3 * 64;
    hipLaunchKernelGGL(conv3x3_pack_k, dim3(ceil_div(operands, 256)), dim3(256), 0, stream, weight,
                       static_cast<v4u*>(workspace), in_channels, out_channels, turned, steps, operands);
    const size_t lds = (size_t)3 * 4 * (few ? kHalo<2> : kHalo<8>) * 16;
    auto launch = [&](auto kernel) {
        (void)allow_dynamic_lds(kernel, lds);
        const int64_t plane = (int64_t)H * W, images = kConvMaxWorkgroups / per_image;
        for (int64_t n = 0; n < N; n += images) {
            const int64_t total = std::min<int64_t>(images, N - n) * per_image;
            hipLaunchKernelGGL(kernel, dim3((unsigned)(ceil_div(total, (int64_t)8) * 8)), dim3(256), lds, stream,
                               input + n * in_channels * plane, static_cast<const v8bf*>(workspace), weight, bias,
                               out + n * out_channels * plane, in_channels, out_channels, H, W, turned, activation,
                               activation == SPGT_ACT_NONE ? 0 : act_count, tx, ty, groups, steps, (int)total);
        }
    };
    if (few) launch(conv3x3_split_k<2>);
    else launch(conv3x3_split_k<8>);
    return check_launch("conv3x3_forward");
}

// ---- weight gradient ----

namespace spgt {

namespace {

constexpr int kGradCols = 32;  // pixels of a step: one row of a column strip

// f(0) .. f(N - 1) with the index as a constant (a loop this long is unrolled too late for its arrays to become registers)
template <typename F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
    each_of(f, std::make_integer_sequence<int, N>{});
}

struct WeightGradPlan {
    int ci_tiles, ni, groups;            // 16 input channels and ni blocks of 16 output channels per wave
    int strips, ranges, rows, items;     // an item: `rows` rows of a strip of one image
    int chunks;                          // waves per (ci tile, group), each a run of items
};

}  // namespace

// Partial sums of dw[co][ci][ky][kx] = sum over n, y, x of g[n][co][y][x] * in[n][ci][y + ky - 1][x + kx - 1], and of g per
// channel, in three-piece bf16 arithmetic.  A wave takes 16 input channels, NI blocks of 16 output channels and all nine
// taps, and walks down column strips 32 pixels wide: the contraction runs along the pixels of a row, which both planar
// operands hold side by side, so a lane's eight of them are two 16-byte loads and nothing goes through LDS.  Three rows of
// the input stay in registers as operands for the three shifts along x (the odd pairs by v_alignbit from the even ones),
// so a step splits one new row and one of g for 54 NI MFMAs; the loads run two steps ahead, the splitting between the
// MFMAs of the step before.  First taps of the oldest row: its registers take the next one.  Strips at the ends of a row
// read on into the next row and clear those values; where a row or an image ends the buffer they load value by value, those
// outside at offsets outside the buffer, which read as zeros.
// The matrix pipe and the issue of one wave per SIMD bound it.  With the sums over the waves and the bias, microseconds on
// the device, the convolution library's (transposes and bias sums included) and this one's: 4 x 363 x 364 pixels, 128 -> 42
// channels 1039 and 402, 42 -> 42 567 and 130; 4 x 122 x 123, 42 -> 42 91 and 35; 16 x 64 x 65, 64 -> 64 97 and 56; one
// image of 30 x 31, 42 -> 42 41 and 18; the error against 64-bit sums 2.7 .. 8.9e-7 -> 0.8 .. 1.7e-7 of the norm.  Ends of
// rows value by value 159 for 130, splitting whole pairs behind one MFMA 133, at least 24 rows an item 84 for 30 at 90 x 91.
// grid (waves / 4, rounded up to a multiple of 8), block 256; one wave per SIMD, for 54 NI + 230 registers
template <int NI>
__global__ __launch_bounds__(256, 1) void conv3x3_wgrad_k(const float* __restrict__ in, const float* __restrict__ grad,
                                                          float4* __restrict__ partial, float* __restrict__ bias_partial,
                                                          int cin, int cout, int H, int W, WeightGradPlan p) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, quad = lane >> 4;
    // waves of one chunk read the same pixels: neighbours, on one XCD
    const int per_xcd = gridDim.x >> 3;
    const int id = ((blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3)) * 4 + wave;
    const int blocks = p.ci_tiles * p.groups;
    if (id >= blocks * p.chunks) return;
    const int ct = id % p.ci_tiles, group = id / p.ci_tiles % p.groups, chunk = id / blocks;
    const int first = (int)((int64_t)chunk * p.items / p.chunks), end = (int)((int64_t)(chunk + 1) * p.items / p.chunks);
    const uint32_t plane = (uint32_t)H * (uint32_t)W;
    constexpr uint32_t kOutside = 0x80000000u;  // past any descriptor below
    const int cx = 16 * ct + l16;

    v4f big[9][NI], small[9][NI];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int c = 0; c < NI; ++c) big[t][c] = small[t][c] = v4f{0.f, 0.f, 0.f, 0.f};
    float colsum[NI] = {};
    v4u xf[3][2][3];     // [row slot][shift to the left, to the right][piece]
    v4u xm[3];           // the row in the middle position, formed where it is used
    v4u gf[2][NI][3];    // [parity][block][piece]
    float rx[2][10], rg[2][NI][8];

    for (int item = first; item < end; ++item) {
        const int range = item % p.ranges, col = item / p.ranges;
        const int x0 = kGradCols * (col % p.strips), n = col / p.strips;
        const int y0 = range * p.rows, rows = min(p.rows, H - y0);
        const float* const xs = in + (int64_t)n * cin * plane;
        const float* const gs = grad + (int64_t)n * cout * plane;
        const bool interior = x0 >= 1 && x0 + kGradCols < W;
        // (a 16-byte load that starts in a row of 4 values ends in the next one at the latest)
        const bool wide_ends = W >= 4;
        const int px = x0 + 8 * quad;
        // row y of all channels, from the value before its first pixel on; nothing where there is no such row
        auto row_of = [&](const float* base, int channels, int y, bool ok) __attribute__((always_inline)) {
            return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base + (int64_t)y * W - 1), 0,
                                                     ok ? ((uint32_t)channels * plane - (uint32_t)y * (uint32_t)W) * 4u + 4u : 0u,
                                                     0x00027000);
        };
        const uint32_t xo = cx < cin ? 4u * ((uint32_t)cx * plane + (uint32_t)px) : kOutside;
        auto fetch_x = [&](float (&v)[10], int y) __attribute__((always_inline)) {
            const __amdgpu_buffer_rsrc_t r = row_of(xs, cin, y, y >= 0 && y < H);
            if (interior || (wide_ends && y > 0 && y < H - 1)) {
                const v4f a = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, xo, 0, 0));
                const v4f b = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, xo + 16u, 0, 0));
                const v2f c = __builtin_bit_cast(v2f, __builtin_amdgcn_raw_buffer_load_b64(r, xo + 32u, 0, 0));
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = a[j], v[4 + j] = b[j];
                v[8] = c[0], v[9] = c[1];
            } else {
#pragma unroll
                for (int j = 0; j < 10; ++j) {
                    const uint32_t o = (uint32_t)(px + j - 1) < (uint32_t)W && cx < cin ? xo + 4u * j : kOutside;
                    v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0));
                }
            }
        };
        auto fetch_g = [&](float (&v)[NI][8], int y) __attribute__((always_inline)) {
            const __amdgpu_buffer_rsrc_t r = row_of(gs, cout, y, y < y0 + rows);
#pragma unroll
            for (int c = 0; c < NI; ++c) {
                const int co = 16 * (NI * group + c) + l16;
                const uint32_t go = co < cout ? 4u * ((uint32_t)co * plane + (uint32_t)px) + 4u : kOutside;
                if (interior || (wide_ends && y < H - 1)) {
                    const v4f a = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, go, 0, 0));
                    const v4f b = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, go + 16u, 0, 0));
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[c][j] = a[j], v[c][4 + j] = b[j];
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const uint32_t o = px + j < W && co < cout ? go + 4u * j : kOutside;
                        v[c][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0));
                    }
                }
            }
        };
        // Pairs in two halves, the second with what the first left: so no MFMA's shadow has more than it covers.
        // values 2 j - 1 and 2 j of the lane's eight: pair j of the shift to the left, pair j - 1 of that to the right
        uint32_t piece_hi;
        float left_a, left_b;
        auto half_x = [&](v4u (&f)[2][3], float (&v)[10], int j, bool second) __attribute__((always_inline)) {
            if (!second) {
                if (!interior) {
#pragma unroll
                    for (int e = 2 * j; e < 2 * j + 2; ++e) v[e] = (uint32_t)(px + e - 1) < (uint32_t)W ? v[e] : 0.f;
                }
                left_a = v[2 * j], left_b = v[2 * j + 1];
                split_first(left_a, left_b, piece_hi);
                return;
            }
            uint32_t q[3] = {piece_hi, 0, 0};
            split_rest(left_a, left_b, q[1], q[2]);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                if (j < 4) f[0][k][j] = q[k];
                if (j > 0) f[1][k][j - 1] = q[k];
            }
        };
        auto half_g = [&](v4u (&f)[NI][3], float (&v)[NI][8], int c, int j, bool second) __attribute__((always_inline)) {
            if (!second) {
                if (!interior) {
#pragma unroll
                    for (int e = 2 * j; e < 2 * j + 2; ++e) v[c][e] = px + e < W ? v[c][e] : 0.f;
                }
                left_a = v[c][2 * j], left_b = v[c][2 * j + 1];
                split_first(left_a, left_b, piece_hi);
                return;
            }
            f[c][0][j] = piece_hi;
            uint32_t m, l;
            split_rest(left_a, left_b, m, l);
            f[c][1][j] = m, f[c][2][j] = l;
        };
        auto split_x = [&](v4u (&f)[2][3], float (&v)[10], int j) __attribute__((always_inline)) {
            half_x(f, v, j, false), half_x(f, v, j, true);
        };
        auto split_g = [&](v4u (&f)[NI][3], float (&v)[NI][8], int c, int j) __attribute__((always_inline)) {
            half_g(f, v, c, j, false), half_g(f, v, c, j, true);
        };
        auto middle_x = [&](const v4u (&f)[2][3]) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < 3; ++k)
#pragma unroll
                for (int j = 0; j < 4; ++j) xm[k][j] = __builtin_amdgcn_alignbit(f[1][k][j], f[0][k][j], 16);
        };
        auto add_column = [&](const float (&v)[NI][8], int c) __attribute__((always_inline)) {
            colsum[c] += ((v[c][0] + v[c][1]) + (v[c][2] + v[c][3])) + ((v[c][4] + v[c][5]) + (v[c][6] + v[c][7]));
        };
        {
            float before[10], at[10];
            fetch_x(before, y0 - 1);
            fetch_x(at, y0);
            fetch_x(rx[0], y0 + 1);
            fetch_g(rg[0], y0);
            fetch_x(rx[1], y0 + 2);
            fetch_g(rg[1], y0 + 1);
#pragma unroll
            for (int j = 0; j < 5; ++j) split_x(xf[0], before, j), split_x(xf[1], at, j), split_x(xf[2], rx[0], j);
#pragma unroll
            for (int c = 0; c < NI; ++c) {
#pragma unroll
                for (int j = 0; j < 4; ++j) split_g(gf[0], rg[0], c, j);
                add_column(rg[0], c);
            }
        }
        // step s: row y0 + s of g; the raw values of step s + 1 (row y0 + s + 2 of the input) are in parity (s + 1) % 2
        auto step = [&](auto k_, int s) __attribute__((always_inline)) {
            constexpr int K = decltype(k_)::value, SLOT = K % 3, D = K % 2;
            fetch_x(rx[D], y0 + s + 3);
            fetch_g(rg[D], y0 + s + 2);
            __builtin_amdgcn_sched_barrier(0);
            constexpr int XP[6] = {2, 0, 0, 1, 1, 0}, GP[6] = {0, 0, 2, 1, 0, 1};  // pieces of the six products
            constexpr int SHIFT[3] = {0, -1, 1};
            constexpr int PAIRS = 5 + 4 * NI;
            each<54>([&](auto i_) __attribute__((always_inline)) {
                constexpr int I = decltype(i_)::value, T = I / 6, Q = I % 6, ROW = (SLOT + T / 3) % 3;
                v4f (&acc)[NI] = Q == 1 ? big[T] : small[T];
                const v4u (&x)[3] = SHIFT[T % 3] < 0 ? xm : xf[ROW][SHIFT[T % 3] & 1];
#pragma unroll
                for (int c = 0; c < NI; ++c)
                    acc[c] = mfma16_bf16(__builtin_bit_cast(v8bf, x[XP[Q]]), __builtin_bit_cast(v8bf, gf[D][c][GP[Q]]),
                                         acc[c]);
                if constexpr (T % 3 == 0 && Q == 5) middle_x(xf[ROW]);
                // 18 .. 51: the next step's operands (the oldest row's registers are free)
                constexpr int FROM = (I - 18) * 2 * PAIRS / 34, TO = (I - 17) * 2 * PAIRS / 34;
                if constexpr (I >= 18 && I < 52 && TO > FROM) {
                    constexpr int P = FROM / 2;
                    if constexpr (P < 5) half_x(xf[SLOT], rx[D ^ 1], P, FROM % 2);
                    else half_g(gf[D ^ 1], rg[D ^ 1], (P - 5) / 4, (P - 5) % 4, FROM % 2);
                }
                if constexpr (I == 53) {
#pragma unroll
                    for (int c = 0; c < NI; ++c) add_column(rg[D ^ 1], c);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        for (int s = 0; s < rows; s += 6) {
            step(std::integral_constant<int, 0>{}, s);
            if (s + 1 < rows) step(std::integral_constant<int, 1>{}, s + 1);
            if (s + 2 < rows) step(std::integral_constant<int, 2>{}, s + 2);
            if (s + 3 < rows) step(std::integral_constant<int, 3>{}, s + 3);
            if (s + 4 < rows) step(std::integral_constant<int, 4>{}, s + 4);
            if (s + 5 < rows) step(std::integral_constant<int, 5>{}, s + 5);
        }
    }

    bool bad = false;
#pragma unroll
    for (int t = 0; t < 9; ++t) {
#pragma unroll
        for (int c = 0; c < NI; ++c) big[t][c] += small[t][c];
        bad = bad || not_finite(big[t]);
    }
    float unscale = kSplitUnscale;
    if (__builtin_expect(__any(bad), 0)) {
        unscale = 1.f;
#pragma unroll
        for (int t = 0; t < 9; ++t) {
#pragma unroll
            for (int c = 0; c < NI; ++c) big[t][c] = v4f{0.f, 0.f, 0.f, 0.f};
            for (int item = first; item < end; ++item) {
                const int range = item % p.ranges, col = item / p.ranges;
                const int x0 = kGradCols * (col % p.strips), n = col / p.strips;
                const int y0 = range * p.rows, y1 = min(y0 + p.rows, H);
                const float* const xs = in + ((int64_t)n * cin + cx) * plane;
                const float* const gs = grad + (int64_t)n * cout * plane;
                for (int y = y0; y < y1; ++y)
                    for (int x4 = x0; x4 < min(x0 + kGradCols, W); x4 += 4) {
                        const int x = x4 + quad, yi = y + t / 3 - 1, xi = x + t % 3 - 1;
                        const bool ok = cx < cin && x < W && yi >= 0 && yi < H && xi >= 0 && xi < W;
                        const float a = ok ? xs[(int64_t)yi * W + xi] : 0.f;
#pragma unroll
                        for (int c = 0; c < NI; ++c) {
                            const int co = 16 * (NI * group + c) + l16;
                            const float b = ok && co < cout ? gs[co * (int64_t)plane + (int64_t)y * W + x] : 0.f;
                            big[t][c] = mfma16(a, b, big[t][c]);
                        }
                    }
            }
        }
    }
    float4* const dst = partial + ((int64_t)chunk * blocks + group * p.ci_tiles + ct) * (9 * NI * 64) + lane;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int c = 0; c < NI; ++c) {
            const v4f v = big[t][c] * unscale;
            dst[(t * NI + c) * 64] = make_float4(v[0], v[1], v[2], v[3]);
        }
    if (ct == 0) {
#pragma unroll
        for (int c = 0; c < NI; ++c) {
            float v = colsum[c];
            v += __shfl_xor(v, 16);
            v += __shfl_xor(v, 32);
            if (quad == 0) bias_partial[((int64_t)chunk * p.groups + group) * (16 * NI) + 16 * c + l16] = v;
        }
    }
}

// The sums over the chunks, in sixteen interleaved chains and a fixed tree, in the weight's layout; the last `groups`
// workgroups sum the bias gradient.
// grid (ci tiles * groups * 9 NI + groups), block 1024
__global__ __launch_bounds__(1024) void conv3x3_wgrad_reduce_k(const float4* __restrict__ partial,
                                                               const float* __restrict__ bias_partial,
                                                               float* __restrict__ dw, float* __restrict__ db, int cin,
                                                               int cout, WeightGradPlan p) {
    __shared__ float4 sums[16][64];
    const int lane = threadIdx.x & 63, chain = threadIdx.x >> 6;
    const int tiles = p.ci_tiles * p.groups * 9 * p.ni;
    const bool is_bias = (int)blockIdx.x >= tiles;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    if (is_bias) {
        const int width = 16 * p.ni;
        const float* src = bias_partial + ((int)blockIdx.x - tiles) * width + min(lane, width - 1);
        for (int k = chain; k < p.chunks; k += 16) s.x += src[(int64_t)k * p.groups * width];
    } else {
        const float4* src = partial + (int64_t)blockIdx.x * 64 + lane;
#pragma unroll 4
        for (int k = chain; k < p.chunks; k += 16) {
            const float4 v = src[(int64_t)k * tiles * 64];
            s.x += v.x, s.y += v.y, s.z += v.z, s.w += v.w;
        }
    }
    sums[chain][lane] = s;
    for (int half = 8; half > 0; half >>= 1) {
        __syncthreads();
        if (chain < half) {
            const float4 o = sums[chain + half][lane];
            s.x += o.x, s.y += o.y, s.z += o.z, s.w += o.w;
            sums[chain][lane] = s;
        }
    }
    if (chain > 0) return;
    if (is_bias) {
        const int co = 16 * p.ni * ((int)blockIdx.x - tiles) + lane;
        if (db && lane < 16 * p.ni && co < cout) db[co] = s.x;
        return;
    }
    const int tile = blockIdx.x % (9 * p.ni), block = blockIdx.x / (9 * p.ni);
    const int tap = tile / p.ni, co = 16 * (p.ni * (block / p.ci_tiles) + tile % p.ni) + (lane & 15);
    const int ci = 16 * (block % p.ci_tiles) + 4 * (lane >> 4);
    const float v[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (co < cout && ci + r < cin) dw[((int64_t)co * cin + ci + r) * 9 + tap] = v[r];
}

}  // namespace spgt

// As many waves as SIMDs, each a run of items; the split of the rows that gives the shortest longest run, counting four
// steps for what an item takes before its first and five (7 us) for the sums over as many chunks.
static WeightGradPlan wgrad_plan(int N, int cin, int cout, int H, int W) {
    WeightGradPlan p{};
    p.ci_tiles = ceil_div(cin, 16);
    const int blocks = ceil_div(cout, 16);
    p.ni = blocks % 3 == 0 || blocks > 4 ? 3 : blocks % 2 == 0 ? 2 : 1;
    if (p.ni == 3 && blocks % 2 == 0 && blocks % 3 != 0) p.ni = 2;
    p.groups = ceil_div(blocks, p.ni);
    p.strips = ceil_div(W, kGradCols);
    const int64_t columns = (int64_t)N * p.strips;
    const int most = std::max(1, 4 * device_cu_count() / (p.ci_tiles * p.groups));
    int64_t best = INT64_MAX;
    for (int r = 1; r <= std::min(64, ceil_div(H, 3)); ++r) {
        const int rows = ceil_div(H, r), ranges = ceil_div(H, rows);
        const int64_t items = columns * ranges;
        const int64_t cost = ceil_div(items, (int64_t)most) * (rows + 4) * most + 5 * std::min<int64_t>(items, most);
        if (cost < best) best = cost, p.rows = rows, p.ranges = ranges;
    }
    p.items = (int)(columns * p.ranges);
    p.chunks = (int)std::min<int64_t>(most, p.items);
    return p;
}

extern "C" int spgt_conv3x3_weight_grad_supported(int N, int in_channels, int out_channels, int H, int W) {
    if (N <= 0 || H <= 0 || W <= 0 || in_channels <= 0 || out_channels <= 0 || in_channels > 4096 || out_channels > 4096)
        return 0;
    return (int64_t)H * W <= INT32_MAX && (int64_t)std::max(in_channels, out_channels) * H * W <= (int64_t)1 << 28 &&
           (int64_t)N * ceil_div(W, kGradCols) * 64 <= INT32_MAX;
}

// The kernel's steps are rows of 32 columns, of which an image's fill W / (32 strips), and a strip's walk takes four steps before
// its first of H.  What is left of that decides on narrow and flat images, against a library kernel whose tiles need 128
// channels on both sides to be full.  Microseconds, the library's and this one's, at fractions below and above each line:
// more than 96 channels on both sides, 0.45: 256 -> 256 of 342 x 8 x 9 (0.19) 284 and 560, 97 x 16 x 16 (0.40) 272 and 318,
// 23 x 33 x 33 (0.46) 298 and 278, 49 x 4 x 128 (0.50) 278 and 225, 24 x 25 (0.67) 280 and 210; fewer on one, 0.2: 64 -> 64 of
// 8025 x 7 x 7 (0.14) 513 and 735, 5462 x 8 x 9 (0.19) 527 and 557, 2731 x 12 x 12 (0.28) 519 and 393; up to 48 x 48, 0.12:
// 42 -> 42 of 44939 x 4 x 5 (0.08) 996 and 1410, 18343 x 7 x 7 (0.14) 995 and 863.
extern "C" int spgt_conv3x3_weight_grad_pays(int N, int in_channels, int out_channels, int H, int W) {
    if (!spgt_conv3x3_weight_grad_supported(N, in_channels, out_channels, H, W)) return 0;
    const double used = (double)W / (kGradCols * ceil_div(W, kGradCols)) * H / (H + 4.0);
    const double line = std::min(in_channels, out_channels) > 96 ? 0.45 : in_channels * out_channels > 48 * 48 ? 0.2 : 0.12;
    return used >= line ? 1 : 0;
}

extern "C" size_t spgt_conv3x3_weight_grad_workspace_bytes(int N, int in_channels, int out_channels, int H, int W) {
    if (!spgt_conv3x3_weight_grad_supported(N, in_channels, out_channels, H, W)) return 0;
    const WeightGradPlan p = wgrad_plan(N, in_channels, out_channels, H, W);
    const size_t values = (size_t)p.ci_tiles * p.groups * 9 * p.ni * 256 + (size_t)p.groups * p.ni * 16;
    return p.chunks * values * sizeof(float);
}

extern "C" int spgt_conv3x3_weight_grad(const float* input, const float* grad, float* weight_grad, float* bias_grad, int N,
                                        int in_channels, int out_channels, int H, int W, void* workspace,
                                        size_t workspace_bytes, hipStream_t stream) {
    if (!input || !grad || !weight_grad) return fail(SPGT_ERR_INVALID_ARGUMENT, "conv3x3_weight_grad: null pointer argument");
    const size_t need = spgt_conv3x3_weight_grad_workspace_bytes(N, in_channels, out_channels, H, W);
    if (need == 0)
        return fail(SPGT_ERR_INVALID_ARGUMENT,
                    "conv3x3_weight_grad: sizes must be positive, at most 4096 channels and 1 GB an image");
    if (!aligned4(input) || !aligned4(grad) || !aligned4(weight_grad) || (bias_grad && !aligned4(bias_grad)))
        return fail(SPGT_ERR_INVALID_ARGUMENT, "conv3x3_weight_grad: misaligned pointer");
    if (!workspace || !aligned16(workspace) || workspace_bytes < need)
        return fail(SPGT_ERR_WORKSPACE, "conv3x3_weight_grad: workspace missing, misaligned or too small");
    const WeightGradPlan p = wgrad_plan(N, in_channels, out_channels, H, W);
    const int blocks = p.ci_tiles * p.groups;
    float4* const partial = static_cast<float4*>(workspace);
    float* const bias_partial = reinterpret_cast<float*>(partial + (size_t)p.chunks * blocks * 9 * p.ni * 64);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(ceil_div(ceil_div(blocks * p.chunks, 4), 8) * 8), dim3(256), 0, stream, input, grad,
                           partial, bias_partial, in_channels, out_channels, H, W, p);
    };
    if (p.ni == 3) launch(conv3x3_wgrad_k<3>);
    else if (p.ni == 2) launch(conv3x3_wgrad_k<2>);
    else launch(conv3x3_wgrad_k<1>);
    hipLaunchKernelGGL(conv3x3_wgrad_reduce_k, dim3(blocks * 9 * p.ni + p.groups), dim3(1024), 0, stream, partial, bias_partial,
                       weight_grad, bias_grad, in_channels, out_channels, p);
    return check_launch("conv3x3_weight_grad");
}
