// Weight and bias gradients of a token-major Linear y = x W + b:
//   dW[k][n] = sum_t x[t][k] g[t][n]        db[n] = sum_t g[t][n]
// (reference: extension/bind/galerkin_attention.cu:41-46, where the two are a library GEMM on the
// transposed input and a library reduction).  The contraction runs over the tokens, tens of thousands
// to millions of them, against 128 x 128 results: a split over token chunks, each chunk's [K, N] tile
// accumulated in MFMA registers straight from global memory (both operands are read with lanes along
// the feature axis, 128-byte runs; no transpose of x is ever formed), then one deterministic
// second-stage sum over the chunks (tile_reduce), bias gradient included.
#include "spgt_device.h"
#include "spgt_host.h"
#include "spgt_kernels.h"
#include "split_mfma.h"

namespace spgt {

// partial[batch][chunk][k * N + n] = sum over the chunk's tokens of x[t][k] * g[t][n]
// partial[batch][chunk][K * N + n] = sum over the chunk's tokens of g[t][n]
// grid (nchunk, batch * nstrip, ceil(K / 128)), block 256: wave w takes rows k in [32 (4 z + w), +32) of the strip
// of NT * 32 columns.  MFMA 32x32x2 step kk contracts tokens 2 kk and 2 kk + 1 of the chunk (lane half = token),
// A = x[t][k0 + lane % 32], B = g[t][n0 + 32 nt + lane % 32].  Operand batches of BK steps are requested one
// batch ahead of the MFMAs that consume them.
// TSPLIT (for K <= 32, where three of the four waves would have no rows): the four waves take the same 32 rows and
// a quarter of the chunk's tokens each, and their tiles are added through LDS in a fixed order.
template <int NT, bool TSPLIT>
__global__ __launch_bounds__(256, 2) void xtg_partial_k(const float* __restrict__ X, int64_t ldx, int64_t x_batch,
                                                     const float* __restrict__ G, int64_t ldg, int64_t g_batch,
                                                     float* __restrict__ partial, int64_t T, int K, int N,
                                                     int tokens_per_chunk, int nstrip) {
    constexpr int BK = 8;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tk = lane & 31;
    const int kh = lane >> 5;
    const int chunk = blockIdx.x;
    const int nchunk = gridDim.x;
    const int b = blockIdx.y / nstrip;
    const int strip = blockIdx.y - b * nstrip;
    const int k0 = TSPLIT ? 0 : (blockIdx.z * 4 + wave) * 32;
    const int n0 = strip * NT * 32;
    const int E = K * N + N;
    if (!TSPLIT && k0 >= K) return;  // whole wave: no barrier follows
    const int64_t c0 = (int64_t)chunk * tokens_per_chunk;
    const int64_t c1 = min(T, c0 + tokens_per_chunk);
    const int64_t quarter = TSPLIT ? (tokens_per_chunk / 4) : 0;  // tokens_per_chunk is a multiple of 16
    const int64_t t0 = TSPLIT ? min(c1, c0 + wave * quarter) : c0;
    const int64_t t1 = TSPLIT ? min(c1, t0 + quarter) : c1;
    const int steps = (int)((t1 - t0 + 1) / 2);
    // clamped feature indices: rows past K and columns past N read valid memory and are masked to zero
    const bool kok = k0 + tk < K;
    const float* xp = X + b * x_batch + t0 * ldx + min(k0 + tk, K - 1);
    const float* gp = G + b * g_batch + t0 * ldg;
    uint32_t goff[NT];
    bool nok[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        nok[nt] = n0 + 32 * nt + tk < N;
        goff[nt] = (uint32_t)min(n0 + 32 * nt + tk, N - 1);
    }
    v16f acc[NT];
    float colsum[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        colsum[nt] = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[nt][r] = 0.f;
    }
    const int last = (int)(t1 - t0) - 1;  // last valid token of the chunk, relative
    float xa[BK], ga[NT][BK], xb[BK], gb[NT][BK];
    // fetch only requests (clamped addresses); the masks are applied when the values are used, so that a batch's
    // loads stay in flight under the previous batch's MFMAs
    auto fetch = [&](float (&xv)[BK], float (&gv)[NT][BK], int batch) {
#pragma unroll
        for (int u = 0; u < BK; ++u) {
            const int64_t tr = min(2 * (batch * BK + u) + kh, last);
            xv[u] = xp[tr * ldx];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) gv[nt][u] = gp[tr * ldg + goff[nt]];
        }
    };
    auto multiply = [&](const float (&xv)[BK], const float (&gv)[NT][BK], int batch) {
#pragma unroll
        for (int u = 0; u < BK; ++u) {
            const bool ok = 2 * (batch * BK + u) + kh <= last;
            const float xm = (ok && kok) ? xv[u] : 0.f;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const float gm = (ok && nok[nt]) ? gv[nt][u] : 0.f;
                acc[nt] = mfma32(xm, gm, acc[nt]);
                colsum[nt] += gm;
            }
        }
    };
    const int nbatch = (steps + BK - 1) / BK;  // steps past the chunk's end contribute zeros
    if (nbatch > 0) fetch(xa, ga, 0);
    for (int bt = 0; bt < nbatch; bt += 2) {
        if (bt + 1 < nbatch) fetch(xb, gb, bt + 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(xa, ga, bt);
        __builtin_amdgcn_sched_barrier(0);
        if (bt + 2 < nbatch) fetch(xa, ga, bt + 2);
        __builtin_amdgcn_sched_barrier(0);
        if (bt + 1 < nbatch) multiply(xb, gb, bt + 1);
        __builtin_amdgcn_sched_barrier(0);
    }
    float* out = partial + ((int64_t)b * nchunk + chunk) * E;
    if constexpr (TSPLIT) {
        // the four waves' tiles and column sums: waves 1..3 to LDS, wave 0 adds them in order
        __shared__ float red[3][NT * 17 * 64];
        if (wave > 0) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
                for (int r = 0; r < 16; ++r) red[wave - 1][(nt * 17 + r) * 64 + lane] = acc[nt][r];
                red[wave - 1][(nt * 17 + 16) * 64 + lane] = colsum[nt];
            }
        }
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int w = 0; w < 3; ++w)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[nt][r] += red[w][(nt * 17 + r) * 64 + lane];
                colsum[nt] += red[w][(nt * 17 + 16) * 64 + lane];
            }
    }
    // acc[nt][r] = dW[k0 + 8 (r / 4) + 4 kh + r % 4][n0 + 32 nt + tk]
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        if (nok[nt]) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int k = k0 + 8 * (r >> 2) + 4 * kh + (r & 3);
                if (k < K) out[(int64_t)k * N + n0 + 32 * nt + tk] = acc[nt][r];
            }
        }
        // bias gradient: the two token halves of a column meet; written once per strip, by the wave of rows 0..31
        const float cs = colsum[nt] + __shfl_xor(colsum[nt], 32, 64);
        if (k0 == 0 && kh == 0 && nok[nt]) out[(int64_t)K * N + n0 + 32 * nt + tk] = cs;
    }
}

// The same partial sums for 128 x 128 blocks of dW, in three-piece bf16 arithmetic (split_mfma.h).  Both operands of an
// MFMA 32x32x16 hold eight consecutive tokens of one feature per lane, while memory has a token's features side by
// side: a wave takes eight tokens of x (waves 0..3) or g (waves 4..7), a lane two neighbouring features of them, and
// the lane's values, cut into pieces, are two ready operands, which go to LDS as 16-byte units, features of one
// parity side by side.  Block (h, a) of 32 features is then 2 (32 h + i) + a, i = 0 .. 31.  Wave w forms the rows of block
// (w & 1, w / 2 & 1) and the columns 64 (w / 4) .. +63.
// Tiles of 32 tokens, two LDS buffers, the raw rows of two tiles in flight.  What bounds it is memory: 32 KB per tile
// and CU against 1536 matrix cycles, and the 64 KB of partial sums per unit, which on short inputs are not hidden (the
// counters show 67 + 17 MB in 24 us at 65k tokens, 365 + 17 in 90 at 356k: 3.5 and 4.2 TB/s, a copy reaches 5.3).
// 65536 tokens of 128 x 128 with the sum over the chunks: 41 -> 27.5 us, 128 x 256 61 -> 41, three planes 83 -> 58, 16384
// tokens 27.7 -> 18.4 (before: fp32 MFMAs straight from global memory, 16 accumulators per wave); the error against
// 64-bit sums 1.78e-7 -> 1.29e-7 of the norm.
// A wave whose sums are not finite forms them again with fp32 MFMAs.
// grid (nchunk, batch * nstrip, ceil(K / 128)), block 512, one workgroup per compute unit.
// Requires N a multiple of 128, K a multiple of 4 and at least 128 (the rows of the last block past K are read from
// the row's last piece, used as zeros and not stored), ldx and ldg multiples of 4, 16-byte aligned x and g.
constexpr int kXtgTile = 32;
constexpr size_t kXtgLds = (size_t)2 * 3 * 2 * 4 * 128 * 16;  // [buffer][piece][x, g][eight tokens][parity][64] units

__global__ __launch_bounds__(512, 2) void xtg_partial_split_k(const float* __restrict__ X, int64_t ldx, int64_t x_batch,
                                                              const float* __restrict__ G, int64_t ldg,
                                                              int64_t g_batch, float* __restrict__ partial, int64_t T,
                                                              int K, int N, int tokens_per_chunk, int nstrip) {
    extern __shared__ __align__(16) v8bf units[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i32 = lane & 31;
    const int kh = lane >> 5;
    const int chunk = blockIdx.x;
    const int nchunk = gridDim.x;
    const int b = blockIdx.y / nstrip;
    const int strip = blockIdx.y - b * nstrip;
    const int k0 = blockIdx.z * 128;
    const int n0 = strip * 128;
    const int E = K * N + N;
    const int64_t t0 = (int64_t)chunk * tokens_per_chunk;
    const int last = (int)(min(T, t0 + tokens_per_chunk) - t0) - 1;
    const int tiles = (last + kXtgTile) / kXtgTile;
    const float* const xc = X + b * x_batch + t0 * ldx;
    const float* const gc = G + b * g_batch + t0 * ldg;

    // ---- this thread's share of a tile: eight tokens of two features
    const bool is_g = wave >= 4;
    const int eight = wave & 3;
    const bool feature_ok = is_g || k0 + 2 * lane < K;  // K is a multiple of 4: a pair lies inside the row or past it
    const float* const src = is_g ? gc + n0 + 2 * lane : xc + min(k0 + 2 * lane, K - 2);
    const int64_t ld = is_g ? ldg : ldx;
    float2 raw[2][8];
    auto fetch = [&](float2 (&v)[8], int tile) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            v[j] = *reinterpret_cast<const float2*>(src + (int64_t)min(tile * kXtgTile + 8 * eight + j, last) * ld);
    };
    float colsum[2] = {0.f, 0.f};
    auto split_store = [&](const float2 (&v)[8], int tile, int buf) {
        float even[8], odd[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bool ok = feature_ok && tile * kXtgTile + 8 * eight + j <= last;
            even[j] = ok ? v[j].x : 0.f;
            odd[j] = ok ? v[j].y : 0.f;
        }
        // eight tokens in pairs before they join the chain, which is then an eighth as long (error of the bias gradient at
        // 65k tokens of 128 columns, zero mean: 1.83e-7 of the norm token by token, 1.31e-7 this way)
        auto sum8 = [](const float (&u)[8]) { return ((u[0] + u[1]) + (u[2] + u[3])) + ((u[4] + u[5]) + (u[6] + u[7])); };
        colsum[0] += sum8(even);
        colsum[1] += sum8(odd);
        v8bf* d = units + ((buf * 3 * 2 + is_g) * 4 + eight) * 128 + lane;
        const Split8 e = split8(even), o = split8(odd);
        d[0] = e.hi, d[64] = o.hi;
        d[1024] = e.mid, d[1024 + 64] = o.mid;
        d[2048] = e.lo, d[2048 + 64] = o.lo;
    };

    // ---- this wave's block: 32 rows, 64 columns (two parities of 32)
    const int row_unit = ((wave >> 1) & 1) * 64 + 32 * (wave & 1) + i32;
    const int col_unit = 32 * (wave >> 2) + i32;
    v16f big[2], small[2];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) big[c][r] = small[c][r] = 0.f;
    auto multiply = [&](int buf) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const v8bf* u = units + (buf * 3 * 2 * 4 + 2 * s + kh) * 128;
            v8bf xv[3], gv[2][3];
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                xv[p] = u[p * 1024 + row_unit];
                gv[0][p] = u[p * 1024 + 512 + col_unit];
                gv[1][p] = u[p * 1024 + 512 + 64 + col_unit];
            }
            auto mul = [&](v16f (&acc)[2], int xp, int gp) {
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv[xp], gv[c][gp], acc[c], 0, 0, 0);
            };
            mul(small, 2, 0);
            mul(big, 0, 0);
            mul(small, 0, 2);
            mul(small, 1, 1);
            mul(small, 1, 0);
            mul(small, 0, 1);
        }
    };
    if (tiles > 0) {
        fetch(raw[0], 0);
        fetch(raw[1], 1);  // past the end: the last row again, used as zeros
        split_store(raw[0], 0, 0);
        __syncthreads();
        for (int it = 0; it < tiles; it += 2) {
#pragma unroll
            for (int d = 0; d < 2; ++d) {  // a tile past the end contributes zeros
                fetch(raw[d], it + d + 2);
                __builtin_amdgcn_sched_barrier(0);
                multiply(d);
                split_store(raw[d ^ 1], it + d + 1, d ^ 1);
                __syncthreads();
            }
        }
    }
    bool bad = false;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        float t = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            big[c][r] += small[c][r];
            t = fmaf(big[c][r], 0.f, t);
        }
        bad = bad || t != t;
    }
    const int krow = 2 * (32 * (wave & 1) + i32) + ((wave >> 1) & 1);  // of this lane as a row index, from k0 on
    float unscale = kSplitUnscale;
    if (__builtin_expect(__any(bad), 0)) {
        unscale = 1.f;
        const bool kok = k0 + krow < K;
        const float* xp = xc + min(k0 + krow, K - 1);
        const float* gp = gc + n0 + 2 * col_unit;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) big[c][r] = 0.f;
        for (int t = 0; t <= last; t += 2) {
            const int tr = min(t + kh, last);
            const bool ok = t + kh <= last;
            const float xk = ok && kok ? xp[tr * ldx] : 0.f;
            const float2 gn = ok ? *reinterpret_cast<const float2*>(gp + tr * ldg) : make_float2(0.f, 0.f);
            big[0] = mfma32(xk, gn.x, big[0]);
            big[1] = mfma32(xk, gn.y, big[1]);
        }
    }
    float* out = partial + ((int64_t)b * nchunk + chunk) * E;
    // big[c][r] = dW[k0 + 2 (32 (wave & 1) + i) + parity][n0 + 2 col_unit + c], i = 8 (r / 4) + 4 kh + r % 4
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int k = k0 + 2 * (32 * (wave & 1) + 8 * (r >> 2) + 4 * kh + (r & 3)) + ((wave >> 1) & 1);
        if (k < K)
            *reinterpret_cast<float2*>(out + (int64_t)k * N + n0 + 2 * col_unit) =
                make_float2(big[0][r] * unscale, big[1][r] * unscale);
    }
    if (blockIdx.z == 0) {
        // bias gradient: the four waves' column sums in a fixed order (the last barrier freed the buffers)
        float* colsm = reinterpret_cast<float*>(units);  // [4][128]
        if (is_g) {
            colsm[eight * 128 + 2 * lane] = colsum[0];
            colsm[eight * 128 + 2 * lane + 1] = colsum[1];
        }
        __syncthreads();
        if (threadIdx.x < 128) {
            const int n = threadIdx.x;
            out[(int64_t)K * N + n0 + n] = (colsm[n] + colsm[128 + n]) + (colsm[256 + n] + colsm[384 + n]);
        }
    }
}

// out = residual + dropout(y) on [rows, cols] (cols a multiple of 4; residual may be null): the reference's
// F.dropout followed by the residual add (network/sp_layer.py:76, 100-103; network/layer.py:173) in one pass, with
// the keep decisions of dropout_site / dropout_apply (spgt_device.h).  The same call on a gradient with the
// forward's seed is the backward of the dropout.  A thread takes 16-byte pieces, grid-stride.
__global__ __launch_bounds__(256) void dropout_add_k(const float* __restrict__ y, const float* __restrict__ residual,
                                                     float* __restrict__ out, int64_t pieces, int cols4,
                                                     const uint32_t* __restrict__ seed, float p, uint32_t site) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < pieces; e += stride) {
        const int64_t row = e / cols4;
        const uint32_t col = 4u * (uint32_t)(e - row * cols4);
        const DropoutSite ds = dropout_site(seed, site, row, p);
        const float4 v = reinterpret_cast<const float4*>(y)[e];
        float4 o = make_float4(dropout_apply(ds, col, v.x), dropout_apply(ds, col + 1, v.y),
                               dropout_apply(ds, col + 2, v.z), dropout_apply(ds, col + 3, v.w));
        if (residual) {
            const float4 r = reinterpret_cast<const float4*>(residual)[e];
            o.x += r.x, o.y += r.y, o.z += r.z, o.w += r.w;
        }
        reinterpret_cast<float4*>(out)[e] = o;
    }
}

}  // namespace spgt

using namespace spgt;

namespace {

struct WgradPlan {
    int nt, nstrip, kz, tpc, nchunk;
    bool wide;
};

// The plan depends on the sizes only (the workspace query has nothing else): the wide kernel serves N a multiple
// of 128 with K a multiple of 4 from 128 up and is chosen then; a call whose strides or alignment do not fit it
// runs the kernel above on the same chunks.
WgradPlan wgrad_plan(int64_t T, int K, int N, int batch) {
    WgradPlan p;
    p.wide = K % 4 == 0 && K >= 128 && N % 128 == 0;
    p.nt = N >= 128 ? 4 : (N > 32 ? 2 : 1);
    p.nstrip = ceil_div(N, p.nt * 32);
    p.kz = ceil_div(K, 128);
    // about two workgroups per compute unit (one for the wide kernel: its two LDS buffers take 96 of 160 KB), at most
    // as many chunks as tile_reduce sums, at least 64 tokens each
    const int per = std::max(1, (p.wide ? 1 : 2) * device_cu_count() / std::max(1, batch * p.nstrip * p.kz));
    int64_t nchunk = std::min<int64_t>(std::min(per, kReduceChains * kReduceMaxPerChain), std::max<int64_t>(1, T / 64));
    int64_t tpc = ceil_div(ceil_div(T, nchunk), (int64_t)16) * 16;
    p.tpc = (int)tpc;
    p.nchunk = (int)ceil_div(T, tpc);
    return p;
}

}  // namespace

extern "C" size_t spgt_linear_weight_grad_workspace_bytes(int64_t tokens, int in_features, int out_features,
                                                          int batch) {
    if (tokens <= 0 || in_features <= 0 || out_features <= 0 || batch <= 0 || out_features % 4 != 0) return 0;
    if (tokens > ((int64_t)1 << 31) - 1024 || (int64_t)in_features * out_features + out_features > INT32_MAX) return 0;
    const WgradPlan p = wgrad_plan(tokens, in_features, out_features, batch);
    return (size_t)batch * p.nchunk * ((size_t)in_features * out_features + out_features) * sizeof(float);
}

extern "C" int spgt_linear_weight_grad(const float* x, int64_t ldx, int64_t x_batch_stride, const float* grad,
                                       int64_t ldg, int64_t grad_batch_stride, float* out, void* workspace,
                                       size_t workspace_bytes, int64_t tokens, int in_features, int out_features,
                                       int batch, hipStream_t stream) {
    if (!x || !grad || !out || !workspace)
        return fail(SPGT_ERR_INVALID_ARGUMENT, "linear_weight_grad: null pointer argument");
    const size_t need = spgt_linear_weight_grad_workspace_bytes(tokens, in_features, out_features, batch);
    if (need == 0)
        return fail(SPGT_ERR_INVALID_ARGUMENT,
                    "linear_weight_grad: sizes must be positive, out_features a multiple of 4, tokens below 2^31");
    if (ldx < in_features || ldg < out_features)
        return fail(SPGT_ERR_INVALID_ARGUMENT, "linear_weight_grad: row strides shorter than the rows");
    const int64_t E = (int64_t)in_features * out_features + out_features;
    if (workspace_bytes < need || !aligned16(workspace))
        return fail(SPGT_ERR_WORKSPACE, "linear_weight_grad: workspace missing, misaligned or too small");
    if (!aligned4(x) || !aligned4(grad) || !aligned16(out))
        return fail(SPGT_ERR_INVALID_ARGUMENT, "linear_weight_grad: out must be 16-byte aligned");
    const WgradPlan p = wgrad_plan(tokens, in_features, out_features, batch);
    if ((int64_t)batch * p.nstrip > 65535 || p.kz > 65535)
        return fail(SPGT_ERR_INVALID_ARGUMENT, "linear_weight_grad: too many column strips or row blocks");
    float* partial = static_cast<float*>(workspace);
    const dim3 grid(p.nchunk, batch * p.nstrip, p.kz);
#define SPGT_XTG(NT)                                                                                               \
    if (in_features <= 32)                                                                                         \
        hipLaunchKernelGGL((xtg_partial_k<NT, true>), grid, dim3(256), 0, stream, x, ldx, x_batch_stride, grad, ldg, \
                           grad_batch_stride, partial, tokens, in_features, out_features, p.tpc, p.nstrip);        \
    else                                                                                                           \
        hipLaunchKernelGGL((xtg_partial_k<NT, false>), grid, dim3(256), 0, stream, x, ldx, x_batch_stride, grad, ldg, \
                           grad_batch_stride, partial, tokens, in_features, out_features, p.tpc, p.nstrip)
    const bool wide_ok = p.wide && ldx % 4 == 0 && ldg % 4 == 0 && x_batch_stride % 4 == 0 &&
                         grad_batch_stride % 4 == 0 && aligned16(x) && aligned16(grad);
    if (wide_ok) (void)allow_dynamic_lds(xtg_partial_split_k, kXtgLds);
    if (wide_ok)
        hipLaunchKernelGGL(xtg_partial_split_k, grid, dim3(512), kXtgLds, stream, x, ldx, x_batch_stride, grad, ldg,
                           grad_batch_stride, partial, tokens, in_features, out_features, p.tpc, p.nstrip);
    else if (p.nt == 4) { SPGT_XTG(4); }
    else if (p.nt == 2) { SPGT_XTG(2); }
    else { SPGT_XTG(1); }
#undef SPGT_XTG
    hipLaunchKernelGGL(tile_reduce, dim3(ceil_div((int)E, 256), batch), dim3(1024), 0, stream, partial, out, (int)E,
                       p.nchunk, 1.0f);
    return check_launch("linear_weight_grad");
}

extern "C" int spgt_dropout_add(const float* y, const float* residual, float* out, int64_t rows, int cols,
                                const uint32_t* seed, float droprate, int site, hipStream_t stream) {
    if (!y || !out || !seed) return fail(SPGT_ERR_INVALID_ARGUMENT, "dropout_add: null pointer argument");
    if (rows < 0 || cols <= 0 || cols % 4 != 0)
        return fail(SPGT_ERR_INVALID_ARGUMENT, "dropout_add: cols must be a positive multiple of 4");
    if (!(droprate >= 0.f && droprate < 1.f)) return fail(SPGT_ERR_INVALID_ARGUMENT, "dropout_add: the rate must lie in [0, 1)");
    if (!aligned16(y) || !aligned16(out) || (residual && !aligned16(residual)) || !aligned8(seed))
        return fail(SPGT_ERR_INVALID_ARGUMENT, "dropout_add: tensors must be 16-byte aligned, the seed 8-byte aligned");
    if (rows == 0) return SPGT_OK;
    const int64_t pieces = rows * (cols / 4);
    const unsigned grid = (unsigned)std::min<int64_t>(ceil_div(pieces, (int64_t)256), (int64_t)16 * device_cu_count());
    hipLaunchKernelGGL(dropout_add_k, dim3(grid), dim3(256), 0, stream, y, residual, out, pieces, cols / 4, seed, droprate,
                       (uint32_t)site);
    return check_launch("dropout_add");
}
