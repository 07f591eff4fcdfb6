// 3x3 convolution with padding 1 on planar images in three-piece bf16 arithmetic (split_mfma.h):
//   out[n][co][y][x] = act^count(sum over ci, ky, kx of in[n][ci][y + ky - 1][x + kx - 1] * w[co][ci][ky][kx] + bias[co])
// (the three middle convolutions of the down-scaler, network/model.py:13-25 with ConvResBlock2D, network/layer.py, and
// with the weights turned round their data gradients).
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
// and 39.  with_gradient: a training step through the convolution, whose autograd function costs 45 us of host time
// more than the library's.  From 2^28 products per tap or 12 Mi values on the kernels outweigh it (forward and
// backward: 64 -> 64 of 16 x 64 x 65 247 and 226, 42 -> 42 of 4 x 256 x 257 608 and 429, 64 -> 1 of it 315 and 277;
// below, 42 -> 42 of 4 x 122 x 123 201 and 238, of 30 x 31 187 and 234).
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
