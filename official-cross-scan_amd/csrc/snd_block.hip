// The passes of a VSS block around its scan: token LayerNorm, depthwise convolution + SiLU, the step-size projection, output
// LayerNorm + gate, and the weight gradients of the two projections.  What they move is
// read once from memory (halos and second passes come from the L2) and written once, in the layout its reader wants - tokens by
// channels for the linear layers, channels by pixels for the scan - with the transposition done in LDS on the way.  None is at the
// rate of memory yet: the convolution's bytes at a copy's rate take 6 / 8 of its 19 / 49 us, the gate's backward's 14 of 39.
// Measured on a block of width 96 (inner 192, rank 6) at 8 x 56 x 56, bf16, us forward / backward, against the torch layers
// they replace: convolution + SiLU 90 / 420 -> 19 / 49 (layout copies, im2col per image for the weight), projections 100 / 400
// -> 35 / 95 (products with one long side, copies into and out of their layout), output norm + gate 60 / 150 -> 21 / 39,
// token norm 33 / 70 -> 6 / 13 each, weight gradient of a linear layer 93 + 20 -> 16; the block's training step 2940 -> 1340.
#include <algorithm>
#include <initializer_list>
#include <type_traits>

#include "snd_block.h"
#include "snd_device.h"

namespace snd {
namespace {

__device__ __forceinline__ float silu(float x) { return x / (1.f + expf(-x)); }
__device__ __forceinline__ float dsilu(float x) {
    const float s = 1.f / (1.f + expf(-x));
    return s * fmaf(x, 1.f - s, 1.f);
}
// The value as a tensor of type T holds it.  Parameters and intermediate results are rounded where the chain of torch layers
// these passes stand for rounds them under autocast, so that both compute with the same numbers.
template <typename T> __device__ __forceinline__ float rnd(float x) {
    T v;
    stg(&v, 0, x);
    return ldg(&v, 0);
}

// ---------------------------------------------------------------- LayerNorm over tokens
// GL lanes per token (16 up to 256 channels: no lane is idle at a width of 96, and the sums over a token stay inside one DPP
// row; 64 beyond), the token's channels in registers, CPL per lane.  TX: type of x and dx, TY: of y and dy.
template <int GL> __device__ __forceinline__ float token_sum(float v) {
    v = group_sum<16>(v);
    if (GL == 64) {
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
    }
    return v;
}
template <typename TX, typename TY, int GL, int CPL>
__global__ __launch_bounds__(256) void norm_fwd_kernel(const TX *x, const float *gamma, const float *beta, float eps, int64_t tokens, int C, TY *y,
                                                       float *stats) {
    const int l = threadIdx.x % GL;
    const int64_t tok = (int64_t)blockIdx.x * (256 / GL) + threadIdx.x / GL, tc = min(tok, tokens - 1);
    const bool tin = tok < tokens;
    float v[CPL], sum = 0.f, var = 0.f;
#pragma unroll
    for (int k = 0; k < CPL; ++k) v[k] = ldg(x + tc * C, min(l + GL * k, C - 1));
#pragma unroll
    for (int k = 0; k < CPL; ++k) {
        v[k] = l + GL * k < C ? v[k] : 0.f;
        sum += v[k];
    }
    const float mean = token_sum<GL>(sum) / (float)C;
#pragma unroll
    for (int k = 0; k < CPL; ++k) {
        v[k] = l + GL * k < C ? v[k] - mean : 0.f;
        var = fmaf(v[k], v[k], var);
    }
    const float rstd = rsqrtf(token_sum<GL>(var) / (float)C + eps);
#pragma unroll
    for (int k = 0; k < CPL; ++k) {
        const int c = l + GL * k;
        if (tin && c < C) stg(y + tc * C, c, fmaf(v[k] * rstd, gamma[c], beta[c]));
    }
    if (stats && tin && l == 0) *(float2 *)(stats + 2 * tc) = make_float2(mean, rstd);
}
// A lane group takes every NG * gridDim.x-th token and keeps its channels' dgamma, dbeta in registers.  Every block ends in an
// atomic per channel, all blocks to the same few lines, one after the other: with blocks of 16 waves (where their sums fit in LDS)
// there are 256 of them (25088 x 96: 26 -> 12 us).
constexpr int norm_threads(int GL) { return GL == 16 ? 1024 : 256; }
template <typename TX, typename TY, int GL, int CPL>
__global__ __launch_bounds__(norm_threads(GL)) void norm_bwd_kernel(const TY *dy, const TX *x, const float *gamma, const float *stats, int64_t tokens, int C, TX *dx,
                                                       float *dgamma, float *dbeta) {
    constexpr int NT = norm_threads(GL), NG = NT / GL, CW = GL * CPL, NW = NT / 64;
    __shared__ float sG[NW][CW], sB[NW][CW];
    const int l = threadIdx.x % GL, wave = threadIdx.x >> 6;
    float g[CPL], dg[CPL], db[CPL];
#pragma unroll
    for (int k = 0; k < CPL; ++k) {
        g[k] = gamma[min(l + GL * k, C - 1)];
        dg[k] = db[k] = 0.f;
    }
    for (int64_t t0 = (int64_t)blockIdx.x * NG; t0 < tokens; t0 += (int64_t)gridDim.x * NG) {
        const int64_t tok = t0 + threadIdx.x / GL, tc = min(tok, tokens - 1);
        const bool tin = tok < tokens;
        const float2 st = *(const float2 *)(stats + 2 * tc);
        float xh[CPL], d[CPL], m1 = 0.f, m2 = 0.f;
#pragma unroll
        for (int k = 0; k < CPL; ++k) {
            xh[k] = ldg(x + tc * C, min(l + GL * k, C - 1));
            d[k] = ldg(dy + tc * C, min(l + GL * k, C - 1));
        }
#pragma unroll
        for (int k = 0; k < CPL; ++k) {
            const bool in = tin && l + GL * k < C;
            xh[k] = in ? (xh[k] - st.x) * st.y : 0.f;
            d[k] = in ? d[k] : 0.f;
            dg[k] = fmaf(d[k], xh[k], dg[k]);
            db[k] += d[k];
            d[k] *= g[k];
            m1 += d[k];
            m2 = fmaf(d[k], xh[k], m2);
        }
        m1 = token_sum<GL>(m1) / (float)C;
        m2 = token_sum<GL>(m2) / (float)C;
#pragma unroll
        for (int k = 0; k < CPL; ++k) {
            const int c = l + GL * k;
            if (tin && c < C) stg(dx + tc * C, c, st.y * (d[k] - m1 - xh[k] * m2));
        }
    }
#pragma unroll
    for (int k = 0; k < CPL; ++k) {
        if (GL == 16) {                             // over the wave's four tokens
            dg[k] += __shfl_xor(dg[k], 16);
            dg[k] += __shfl_xor(dg[k], 32);
            db[k] += __shfl_xor(db[k], 16);
            db[k] += __shfl_xor(db[k], 32);
        }
        if ((threadIdx.x & 63) < GL) { sG[wave][l + GL * k] = dg[k]; sB[wave][l + GL * k] = db[k]; }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < C; c += NT) {
        float a = 0.f, b = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) { a += sG[w][c]; b += sB[w][c]; }
        glb_add(dgamma + c, a);
        glb_add(dbeta + c, b);
    }
}

// ---------------------------------------------------------------- depthwise 3x3 + SiLU
// A block takes 32 channels of 4 rows x 32 columns.  The 6 x 34 pixels around them go through LDS, channels innermost at an
// odd pitch, so that both sides of the transposition (lanes along channels of a token, along pixels of a channel) are free of
// bank conflicts.
// Bound by instructions, most of them for the staging's addresses, and by how many blocks a CU holds: with tiles as fp32 in LDS and
// indices divided out per element 33 us forward and 64 backward at 8 x 56 x 56, 192 channels, bf16; tiles in 16 bits 22 and 51; rows
// as scalar bases, all of a thread's loads at once, 19 and 49.
constexpr int kCvC = 32, kCvR = 4, kCvX = 32, kCvP = kCvC + 1, kCvRow = (kCvX + 2) * kCvP, kCvTile = (kCvR + 2) * kCvRow;
// A tile is kept in LDS in the tensors' type: what is staged are its values, or results that are rounded to it.  A thread's loads are
// requested together, at valid addresses (clamped coordinates): a row's is the scalar base, a column's and channel's an offset that
// all rows share (below 2^32 bytes in an image that the scan takes); what lies outside the image becomes zero afterwards.
constexpr int kCvS = kCvR + 2, kCvJ = (kCvX + 2 + 7) / 8;            // staged rows; staged columns per thread (tokens, channels along lanes)
template <typename T> struct ConvX {
    T v[kCvS][kCvJ];
    __device__ __forceinline__ void load(const T *xb, int h0, int w0, int c0, int H, int W, int Di) {
        uint32_t off[kCvJ];
#pragma unroll
        for (int j = 0; j < kCvJ; ++j) off[j] = (uint32_t)min(max(w0 + (int)(threadIdx.x >> 5) + 8 * j - 1, 0), W - 1) * (2 * Di) + min(c0 + (int)(threadIdx.x & 31), Di - 1);
#pragma unroll
        for (int r = 0; r < kCvS; ++r) {
            const T *const row = xb + (int64_t)min(max(h0 + r - 1, 0), H - 1) * W * 2 * Di;
#pragma unroll
            for (int j = 0; j < kCvJ; ++j) v[r][j] = row[off[j]];
        }
    }
    __device__ __forceinline__ void put(T *sX, int h0, int w0, int c0, int H, int W, int Di) const {
        const int ch = threadIdx.x & 31, x0 = threadIdx.x >> 5;
#pragma unroll
        for (int j = 0; j < kCvJ; ++j) {
            const int x = x0 + 8 * j, q = w0 + x - 1;
            const bool in = q >= 0 && q < W && c0 + ch < Di;
            if (x < kCvX + 2)
#pragma unroll
                for (int r = 0; r < kCvS; ++r) sX[r * kCvRow + x * kCvP + ch] = in && h0 + r - 1 >= 0 && h0 + r - 1 < H ? v[r][j] : T{};
        }
    }
};
// du and pre (from the planes of channel c0), staged as dpre = du * silu'(pre): lanes along 32 columns, four channels per thread, and the
// last two columns by themselves
template <typename T> struct ConvD {
    T v[kCvS][4], a[kCvS][4], ve[2], ae[2];
    __device__ __forceinline__ static void edge(int k, int &r, int &x, int &ch) {
        r = min((int)(threadIdx.x >> 6) + 4 * k, kCvS - 1);
        x = kCvX + (threadIdx.x & 1);
        ch = (threadIdx.x >> 1) & 31;
    }
    __device__ __forceinline__ void load(const T *du, const T *pre, int h0, int w0, int c0, int H, int W, int Di) {
        const uint32_t HW = (uint32_t)H * W;
        uint32_t off[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) off[k] = (uint32_t)min((int)(threadIdx.x >> 5) + 8 * k, Di - 1 - c0) * HW + min(max(w0 + (int)(threadIdx.x & 31) - 1, 0), W - 1);
#pragma unroll
        for (int r = 0; r < kCvS; ++r) {
            const int64_t row = (int64_t)min(max(h0 + r - 1, 0), H - 1) * W;
#pragma unroll
            for (int k = 0; k < 4; ++k) { v[r][k] = (du + row)[off[k]]; a[r][k] = (pre + row)[off[k]]; }
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            int r, x, ch;
            edge(k, r, x, ch);
            const uint32_t o = (uint32_t)min(ch, Di - 1 - c0) * HW + (uint32_t)min(max(h0 + r - 1, 0), H - 1) * W + min(w0 + x - 1, W - 1);
            ve[k] = du[o];
            ae[k] = pre[o];
        }
    }
    __device__ __forceinline__ void put(T *sD, int h0, int w0, int c0, int H, int W, int Di) const {
        auto store = [&](int r, int x, int ch, const T &d, const T &p) {
            const int h = h0 + r - 1, q = w0 + x - 1;
            stg(sD, r * kCvRow + x * kCvP + ch, h >= 0 && h < H && q >= 0 && q < W && c0 + ch < Di ? ldg(&d, 0) * dsilu(ldg(&p, 0)) : 0.f);
        };
#pragma unroll
        for (int r = 0; r < kCvS; ++r)
#pragma unroll
            for (int k = 0; k < 4; ++k) store(r, threadIdx.x & 31, (threadIdx.x >> 5) + 8 * k, v[r][k], a[r][k]);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            int r, x, ch;
            edge(k, r, x, ch);                      // (rows beyond the last: the last once more)
            store(r, x, ch, ve[k], ae[k]);
        }
    }
};

template <typename T>
__global__ __launch_bounds__(256) void conv_fwd_kernel(snd_block_shape s, const T *xz, const float *w, const float *bias, T *pre, T *u) {
    __shared__ T sX[kCvTile];
    const int H = s.nrows, W = s.ncols, Di = s.inner, t = threadIdx.x;
    const int nX = (W + kCvX - 1) / kCvX, h0 = (blockIdx.x / nX) * kCvR, w0 = (blockIdx.x % nX) * kCvX, c0 = blockIdx.y * kCvC, b = blockIdx.z;
    const T *xb = xz + (int64_t)b * H * W * 2 * Di;
    ConvX<T> cx;
    cx.load(xb, h0, w0, c0, H, W, Di);
    cx.put(sX, h0, w0, c0, H, W, Di);
    __syncthreads();
    const int x = t & 31;
    if (w0 + x >= W) return;
#pragma unroll
    for (int ch = t >> 5; ch < kCvC; ch += 8) {
        const int c = c0 + ch;
        if (c >= Di) break;
        float wt[9], acc[kCvR];
#pragma unroll
        for (int k = 0; k < 9; ++k) wt[k] = rnd<T>(w[c * 9 + k]);
        const float bv = bias ? rnd<T>(bias[c]) : 0.f;
#pragma unroll
        for (int r = 0; r < kCvR; ++r) acc[r] = 0.f;
#pragma unroll
        for (int r = 0; r < kCvR + 2; ++r)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const float v = ldg(sX, r * kCvRow + (x + j) * kCvP + ch);
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    if (r - i >= 0 && r - i < kCvR) acc[r - i < 0 ? 0 : r - i < kCvR ? r - i : 0] = fmaf(wt[i * 3 + j], v, acc[r - i < 0 ? 0 : r - i < kCvR ? r - i : 0]);
            }
        const int64_t o = ((int64_t)b * Di + c) * H * W + w0 + x;
#pragma unroll
        for (int r = 0; r < kCvR; ++r)
            if (h0 + r < H) {
                const float v = rnd<T>(rnd<T>(acc[r]) + bv);
                if (pre) stg(pre + o + (int64_t)(h0 + r) * W, 0, v);
                stg(u + o + (int64_t)(h0 + r) * W, 0, silu(v));
            }
    }
}
template <typename T>
__global__ __launch_bounds__(256) void conv_bwd_kernel(snd_block_shape s, const T *du, const T *pre, const T *xz, const float *w, T *dxz, float *dw,
                                                       float *dbias) {
    __shared__ __align__(16) T sX[kCvTile];
    __shared__ T sD[kCvTile];
    static_assert(sizeof(sX) >= 8 * 10 * 32 * sizeof(float), "the block's sums take the place of the staged x");
    const int H = s.nrows, W = s.ncols, Di = s.inner, t = threadIdx.x;
    const int nX = (W + kCvX - 1) / kCvX, h0 = (blockIdx.x / nX) * kCvR, w0 = (blockIdx.x % nX) * kCvX, c0 = blockIdx.y * kCvC, b = blockIdx.z;
    const T *xb = xz + (int64_t)b * H * W * 2 * Di;
    const int64_t plane = ((int64_t)b * Di + c0) * H * W;
    ConvX<T> cx;
    ConvD<T> cd;
    cx.load(xb, h0, w0, c0, H, W, Di);
    cd.load(du + plane, pre + plane, h0, w0, c0, H, W, Di);
    cx.put(sX, h0, w0, c0, H, W, Di);
    cd.put(sD, h0, w0, c0, H, W, Di);
    __syncthreads();
    const int ch = t & 31, c = c0 + ch;
    float wt[9], gw[9], gb = 0.f;
#pragma unroll
    for (int k = 0; k < 9; ++k) { wt[k] = c < Di ? rnd<T>(w[c * 9 + k]) : 0.f; gw[k] = 0.f; }
    for (int x = t >> 5; x < kCvX; x += 8) {
        float dx[kCvR] = {};
#pragma unroll
        for (int r = 0; r < kCvR + 2; ++r)
#pragma unroll
            for (int j = 0; j < 3; ++j) {           // dx[h, q] = sum w[i][j] dpre[h - i + 1, q - j + 1]
                const float d = ldg(sD, r * kCvRow + (x + 2 - j) * kCvP + ch);
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const int o = r - 2 + i;        // r = o + 2 - i
                    if (o >= 0 && o < kCvR) dx[o < 0 ? 0 : o < kCvR ? o : 0] = fmaf(wt[i * 3 + j], d, dx[o < 0 ? 0 : o < kCvR ? o : 0]);
                }
            }
        float d[kCvR];
#pragma unroll
        for (int r = 0; r < kCvR; ++r) { d[r] = ldg(sD, (r + 1) * kCvRow + (x + 1) * kCvP + ch); gb += d[r]; }
#pragma unroll
        for (int r = 0; r < kCvR + 2; ++r)
#pragma unroll
            for (int j = 0; j < 3; ++j) {           // dw[i][j] = sum dpre[h, q] x[h + i - 1, q + j - 1]
                const float v = ldg(sX, r * kCvRow + (x + j) * kCvP + ch);
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    if (r - i >= 0 && r - i < kCvR) gw[i * 3 + j] = fmaf(d[r - i < 0 ? 0 : r - i < kCvR ? r - i : 0], v, gw[i * 3 + j]);
            }
        if (w0 + x < W && c < Di)
#pragma unroll
            for (int r = 0; r < kCvR; ++r)
                if (h0 + r < H) stg(dxz + (((int64_t)b * H + h0 + r) * W + w0 + x) * 2 * Di, c, dx[r]);
    }
    __syncthreads();
    float *red = (float *)sX;                       // [8][10][32]
#pragma unroll
    for (int k = 0; k < 9; ++k) red[((t >> 5) * 10 + k) * 32 + ch] = gw[k];
    red[((t >> 5) * 10 + 9) * 32 + ch] = gb;
    __syncthreads();
    for (int i = t; i < 320; i += 256) {
        float v = 0.f;
#pragma unroll
        for (int p = 0; p < 8; ++p) v += red[p * 320 + i];
        const int k = i >> 5, cc = c0 + (i & 31);
        if (cc < Di) {
            if (k < 9) glb_add(dw + cc * 9 + k, v);
            else if (dbias) glb_add(dbias + cc, v);
        }
    }
}

// ---------------------------------------------------------------- output LayerNorm + gate
// A block of 8 waves takes 64 pixels of an image with all their channels: y is read along pixels (twice for mean and variance, then in
// tiles of 32 channels that LDS turns to channels along lanes), z and out along channels.
constexpr int kGtT = 512, kGtP = 64, kGtPitch = kGtP + 1, kGtK = 4;    // threads; pixels; values per thread of a 32-channel tile
__device__ __forceinline__ void gate_tile(const float *yb, int64_t HW, int c0, int Di, int px, float *sY) {
#pragma unroll
    for (int k = 0; k < kGtK; ++k) {
        const int ch = (threadIdx.x >> 6) + 8 * k;
        sY[ch * kGtPitch + px] = yb[(int64_t)min(c0 + ch, Di - 1) * HW];    // (channels and pixels beyond the edge: never used)
    }
}
template <typename T>
__global__ __launch_bounds__(kGtT) void gate_fwd_kernel(snd_block_shape s, const float *y, const T *xz, const float *gamma, const float *beta, float eps,
                                                       T *out, float *stats) {
    __shared__ float sY[32 * kGtPitch], sR[8][kGtP], sMean[kGtP], sStd[kGtP];
    const int64_t HW = (int64_t)s.nrows * s.ncols;
    const int Di = s.inner, t = threadIdx.x, px = t & 63, cg = t >> 6, b = blockIdx.y;
    const int64_t p0 = (int64_t)blockIdx.x * kGtP;
    const bool pin = p0 + px < HW;
    const float *yb = y + (int64_t)b * Di * HW + (pin ? p0 + px : 0);
    float a = 0.f;
#pragma unroll 8
    for (int c = cg; c < Di; c += 8) a += yb[(int64_t)c * HW];
    sR[cg][px] = a;
    __syncthreads();
    const float mean = (((sR[0][px] + sR[1][px]) + (sR[2][px] + sR[3][px])) + ((sR[4][px] + sR[5][px]) + (sR[6][px] + sR[7][px]))) / (float)Di;
    __syncthreads();
    a = 0.f;
#pragma unroll 8
    for (int c = cg; c < Di; c += 8) {
        const float d = yb[(int64_t)c * HW] - mean;
        a = fmaf(d, d, a);
    }
    sR[cg][px] = a;
    __syncthreads();
    const float rstd = rsqrtf((((sR[0][px] + sR[1][px]) + (sR[2][px] + sR[3][px])) + ((sR[4][px] + sR[5][px]) + (sR[6][px] + sR[7][px]))) / (float)Di + eps);
    if (cg == 0) {
        sMean[px] = mean;
        sStd[px] = rstd;
        if (stats && pin) *(float2 *)(stats + 2 * (b * HW + p0 + px)) = make_float2(mean, rstd);
    }
    for (int c0 = 0; c0 < Di; c0 += 32) {
        __syncthreads();
        gate_tile(yb, HW, c0, Di, px, sY);
        __syncthreads();
        const int ch = t & 31, c = c0 + ch;
        if (c < Di) {
            const float g = gamma[c], be = beta[c];
            float z[kGtK];
#pragma unroll
            for (int k = 0; k < kGtK; ++k) z[k] = ldg(xz + (b * HW + min(p0 + (t >> 5) + 16 * k, HW - 1)) * 2 * Di + Di, c);
#pragma unroll
            for (int k = 0; k < kGtK; ++k) {
                const int q = (t >> 5) + 16 * k;
                const float nv = rnd<T>(fmaf((sY[ch * kGtPitch + q] - sMean[q]) * sStd[q], g, be));
                if (p0 + q < HW) stg(out + (b * HW + p0 + q) * Di, c, nv * rnd<T>(silu(z[k])));
            }
        }
    }
}
template <typename T>
__global__ __launch_bounds__(kGtT) void gate_bwd_kernel(snd_block_shape s, const T *dout, const float *y, const T *xz, const float *gamma,
                                                       const float *beta, const float *stats, float *dy, T *dxz, float *dgamma, float *dbeta) {
    __shared__ float sY[32 * kGtPitch], sMean[kGtP], sStd[kGtP], sM1[kGtP], sM2[kGtP], sG[16][32], sB[16][32];
    const int64_t HW = (int64_t)s.nrows * s.ncols;
    const int Di = s.inner, t = threadIdx.x, px = t & 63, b = blockIdx.y, ch = t & 31, pg = t >> 5;
    const int64_t p0 = (int64_t)blockIdx.x * kGtP;
    const bool pin = p0 + px < HW;
    const int64_t yo = (int64_t)b * Di * HW + (pin ? p0 + px : 0);
    if (t < kGtP) {
        const float2 st = pin ? *(const float2 *)(stats + 2 * (b * HW + p0 + px)) : make_float2(0.f, 0.f);
        sMean[px] = st.x;
        sStd[px] = st.y;
    }
    float m1[kGtK] = {}, m2[kGtK] = {};
    for (int c0 = 0; c0 < Di; c0 += 32) {           // the two means over channels the LayerNorm's gradient takes
        __syncthreads();
        gate_tile(y + yo, HW, c0, Di, px, sY);
        __syncthreads();
        const int c = c0 + ch;
        if (c < Di) {
            const float g = gamma[c];
            float z[kGtK], d[kGtK];
#pragma unroll
            for (int k = 0; k < kGtK; ++k) {
                const int64_t tok = b * HW + min(p0 + pg + 16 * k, HW - 1);
                z[k] = ldg(xz + tok * 2 * Di + Di, c);
                d[k] = ldg(dout + tok * Di, c);
            }
#pragma unroll
            for (int k = 0; k < kGtK; ++k) {
                const int q = pg + 16 * k;
                const float dn = rnd<T>(d[k] * rnd<T>(silu(z[k]))) * g;
                m1[k] += dn;
                m2[k] = fmaf(dn, (sY[ch * kGtPitch + q] - sMean[q]) * sStd[q], m2[k]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < kGtK; ++k) {
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) { m1[k] += __shfl_xor(m1[k], o); m2[k] += __shfl_xor(m2[k], o); }
        if (ch == 0) { sM1[pg + 16 * k] = m1[k] / (float)Di; sM2[pg + 16 * k] = m2[k] / (float)Di; }
    }
    for (int c0 = 0; c0 < Di; c0 += 32) {
        __syncthreads();
        gate_tile(y + yo, HW, c0, Di, px, sY);
        __syncthreads();
        const int c = c0 + ch;
        float gg = 0.f, gb = 0.f;
        if (c < Di) {
            const float g = gamma[c], be = beta[c];
            float z[kGtK], d[kGtK];
#pragma unroll
            for (int k = 0; k < kGtK; ++k) {
                const int64_t tok = b * HW + min(p0 + pg + 16 * k, HW - 1);
                z[k] = ldg(xz + tok * 2 * Di + Di, c);
                d[k] = ldg(dout + tok * Di, c);
            }
#pragma unroll
            for (int k = 0; k < kGtK; ++k) {
                const int q = pg + 16 * k;
                const float yh = (sY[ch * kGtPitch + q] - sMean[q]) * sStd[q], dn = rnd<T>(d[k] * rnd<T>(silu(z[k])));
                if (p0 + q < HW) {
                    stg(dxz + (b * HW + p0 + q) * 2 * Di + Di, c, rnd<T>(d[k] * rnd<T>(fmaf(yh, g, be))) * dsilu(z[k]));
                    gg = fmaf(dn, yh, gg);
                    gb += dn;
                }
                sY[ch * kGtPitch + q] = sStd[q] * (dn * g - sM1[q] - yh * sM2[q]);
            }
        }
        sG[pg][ch] = gg;
        sB[pg][ch] = gb;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int cc = (t >> 6) + 8 * k;
            if (pin && c0 + cc < Di) dy[yo + (int64_t)(c0 + cc) * HW] = sY[cc * kGtPitch + px];
        }
        if (t < 64 && c0 + ch < Di) {
            float v = 0.f;
#pragma unroll
            for (int p = 0; p < 16; ++p) v += t < 32 ? sG[p][ch] : sB[p][ch];
            glb_add((t < 32 ? dgamma : dbeta) + c0 + ch, v);
        }
    }
}

// ---------------------------------------------------------------- step-size projection (a product with one side of `rank`)
// The weights of up to kDtW channels at a time in LDS, padded to RP per channel and read by all lanes at one address; two
// pixels per thread where rows of the maps start on even elements (V), so that a store covers 4 bytes of 16-bit values.
constexpr int kDtFloats = 4096;
template <typename T, int V> __device__ __forceinline__ void ld_px(const T *p, float (&o)[V]) {
    if constexpr (V == 2 && sizeof(T) == 2) {
        const uint32_t r = *(const uint32_t *)p;
        o[0] = raw_to_f32((const T *)nullptr, r & 0xffffu);
        o[1] = raw_to_f32((const T *)nullptr, r >> 16);
    } else {
#pragma unroll
        for (int v = 0; v < V; ++v) o[v] = ldg(p, v);
    }
}
template <typename T, int V> __device__ __forceinline__ void st_px(T *p, const float (&x)[V]) {
    if constexpr (V == 2 && sizeof(T) == 2) {
        T a[2];
        stg(a, 0, x[0]);
        stg(a, 1, x[1]);
        *(uint32_t *)p = __builtin_bit_cast(uint32_t, a);
    } else {
#pragma unroll
        for (int v = 0; v < V; ++v) stg(p, v, x[v]);
    }
}
template <typename T, int RP> __device__ __forceinline__ void dt_stage(float *sW, const float *w, int d0, int n, int R) {
    for (int i = threadIdx.x; i < n * RP; i += 256) {
        const int d = i / RP, r = i - d * RP;
        const float v = w[(int64_t)(d0 + d) * R + min(r, R - 1)];
        sW[i] = r < R ? rnd<T>(v) : 0.f;
    }
}
// blockIdx.z takes a share of the channels
template <typename T, int RP, int V>
__global__ __launch_bounds__(256) void dt_fwd_kernel(snd_block_shape s, const T *proj, const float *w, T *delta) {
    __shared__ __align__(16) float sW[kDtFloats];
    const int64_t HW = (int64_t)s.nrows * s.ncols, p = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V, pc = min(p, HW - V);
    const int Di = s.inner, R = s.rank, bg = blockIdx.y, g = bg % s.n_groups;
    const T *src = proj + (int64_t)bg * (R + 2 * s.dstate) * HW + pc;
    float x[RP][V];
#pragma unroll
    for (int r = 0; r < RP; ++r) ld_px<T, V>(src + (int64_t)min(r, R - 1) * HW, x[r]);     // (the weights of r >= R are 0)
    const int per = (Di + gridDim.z - 1) / gridDim.z, d1 = min((int)(blockIdx.z + 1) * per, Di);
    T *dst = delta + (int64_t)bg * Di * HW + pc;
    for (int d0 = blockIdx.z * per; d0 < d1; d0 += kDtFloats / RP) {
        const int n = min(kDtFloats / RP, d1 - d0);
        __syncthreads();
        dt_stage<T, RP>(sW, w + (int64_t)g * Di * R, d0, n, R);
        __syncthreads();
#pragma unroll 4
        for (int d = 0; d < n; ++d) {
            float acc[V] = {};
#pragma unroll
            for (int r = 0; r < RP; ++r)
#pragma unroll
                for (int v = 0; v < V; ++v) acc[v] = fmaf(sW[d * RP + r], x[r][v], acc[v]);
            if (p < HW) st_px<T, V>(dst + (int64_t)(d0 + d) * HW, acc);
        }
    }
}
// 64 * V pixels per block, the channels dealt to its four waves.
template <typename T, int RP, int V>
__global__ __launch_bounds__(256) void dt_bwd_kernel(snd_block_shape s, const T *ddelta, const T *dB, const T *dC, const float *w, T *dproj) {
    __shared__ __align__(16) float sW[kDtFloats], sA[4][8][64 * V];
    const int64_t HW = (int64_t)s.nrows * s.ncols;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t p = ((int64_t)blockIdx.x * 64 + lane) * V, pc = min(p, HW - V);
    const int Di = s.inner, R = s.rank, N = s.dstate, bg = blockIdx.y, g = bg % s.n_groups;
    float acc[RP][V] = {};
    const T *src = ddelta + (int64_t)bg * Di * HW + pc;
    for (int d0 = 0; d0 < Di; d0 += kDtFloats / RP) {
        const int n = min(kDtFloats / RP, Di - d0);
        __syncthreads();
        dt_stage<T, RP>(sW, w + (int64_t)g * Di * R, d0, n, R);
        __syncthreads();
#pragma unroll 8
        for (int d = wave; d < n; d += 4) {
            float v[V];
            ld_px<T, V>(src + (int64_t)(d0 + d) * HW, v);
#pragma unroll
            for (int r = 0; r < RP; ++r)
#pragma unroll
                for (int k = 0; k < V; ++k) acc[r][k] = fmaf(sW[d * RP + r], v[k], acc[r][k]);
        }
    }
    T *dst = dproj + (int64_t)bg * (R + 2 * N) * HW + pc;
#pragma unroll
    for (int r0 = 0; r0 < RP; r0 += 8) {            // the waves' sums, eight rows at a time
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int k = 0; k < V; ++k) sA[wave][r][lane * V + k] = acc[r0 + r][k];
        __syncthreads();
        for (int r = wave; r < 8 && r0 + r < R; r += 4) {
            float v[V];
#pragma unroll
            for (int k = 0; k < V; ++k) v[k] = sA[0][r][lane * V + k] + sA[1][r][lane * V + k] + sA[2][r][lane * V + k] + sA[3][r][lane * V + k];
            if (p < HW) st_px<T, V>(dst + (int64_t)(r0 + r) * HW, v);
        }
    }
    const int64_t o = (int64_t)bg * N * HW + pc;
#pragma unroll 4
    for (int n = wave; n < N; n += 4) {
        float vb[V], vc[V];
        ld_px<T, V>(dB + o + (int64_t)n * HW, vb);
        ld_px<T, V>(dC + o + (int64_t)n * HW, vc);
        if (p < HW) {
            st_px<T, V>(dst + (int64_t)(R + n) * HW, vb);
            st_px<T, V>(dst + (int64_t)(R + N + n) * HW, vc);
        }
    }
}

// ---------------------------------------------------------------- weight gradients
// Both operands have the summed axis (pixels) innermost, which is the layout of either operand of a matrix instruction: a
// lane holds 8 (fp32: 4) consecutive pixels of one row, and rows come straight from memory in 64-byte runs.  The sum is
// long and the result small (a few thousand values), so the pixels are split over the grid and the parts added with atomics.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
template <typename T> struct Frag { typedef uint16_t E; E v[8]; static constexpr int K = 8; };
template <> struct Frag<float> { typedef float E; E v[4]; static constexpr int K = 4; };
__device__ __forceinline__ f32x4 mma(const Frag<float> &a, const Frag<float> &b, f32x4 c) {
#pragma unroll
    for (int k = 0; k < 4; ++k) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[k], b.v[k], c, 0, 0, 0);
    return c;
}
__device__ __forceinline__ f32x4 mma(const Frag<bf16_t> &a, const Frag<bf16_t> &b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma(const Frag<f16_t> &a, const Frag<f16_t> &b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
// VEC: rows start on 16-byte boundaries and hold whole fragments
template <typename T, bool VEC> __device__ __forceinline__ void ld_frag(Frag<T> &f, const T *row, int64_t k, int64_t K) {
    typedef typename Frag<T>::E E;
    const E *src = (const E *)row;
    if (VEC) {
        const uint4 v = k < K ? *(const uint4 *)(src + k) : make_uint4(0, 0, 0, 0);
        __builtin_memcpy(f.v, &v, 16);
    } else {
#pragma unroll
        for (int j = 0; j < Frag<T>::K; ++j) f.v[j] = k + j < K ? src[k + j] : (E)0;
    }
}
// MT x NT tiles of 16 x 16 per wave, WM x WN waves; blockIdx.x: tiles, y: image and share of its pixels, z: group
template <typename T, int MT, int NT, int WM, int WN, bool VEC>
__global__ __launch_bounds__(256) void wgrad_kernel(const T *a, int64_t ab, int64_t ag, const T *c, int64_t cb, int64_t cg, int M, int N, int64_t P,
                                                    int splits, float *out) {
    constexpr int STEP = 4 * Frag<T>::K, UNROLL = VEC ? 2 : 1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nN = (N + 16 * NT * WN - 1) / (16 * NT * WN), mt = blockIdx.x / nN, nt = blockIdx.x - mt * nN;
    const int m0 = (mt * WM + wave / WN) * 16 * MT, n0 = (nt * WN + wave % WN) * 16 * NT;
    const int b = blockIdx.y / splits, sp = blockIdx.y - b * splits, g = blockIdx.z;
    const int64_t per = ((P + splits - 1) / splits + STEP - 1) / STEP * STEP, k0 = sp * per, k1 = min(k0 + per, P);
    const T *ar[MT], *cr[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) ar[i] = a + b * ab + g * ag + (int64_t)min(m0 + 16 * i + (lane & 15), M - 1) * P;
#pragma unroll
    for (int i = 0; i < NT; ++i) cr[i] = c + b * cb + g * cg + (int64_t)min(n0 + 16 * i + (lane & 15), N - 1) * P;
    f32x4 acc[MT][NT] = {};
    if (m0 < M && n0 < N && k0 < k1) {
#pragma unroll UNROLL
        for (int64_t k = k0; k < k1; k += STEP) {
            const int64_t kl = k + (lane >> 4) * Frag<T>::K;
            Frag<T> fa[MT], fc[NT];
#pragma unroll
            for (int i = 0; i < MT; ++i) ld_frag<T, VEC>(fa[i], ar[i], kl, k1);
#pragma unroll
            for (int i = 0; i < NT; ++i) ld_frag<T, VEC>(fc[i], cr[i], kl, k1);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = mma(fa[i], fc[j], acc[i][j]);
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int m = m0 + 16 * i + (lane >> 4) * 4 + e, n = n0 + 16 * j + (lane & 15);
                    if (m < M && n < N) glb_add(out + ((int64_t)g * M + m) * N + n, acc[i][j][e]);
                }
    }
}

// The weight gradient of a linear layer on 16-bit tokens: out[m][n] += sum_t a[t][m] * c[t][n], and bias[m] += sum_t a[t][m].
// Here the summed axis is the outer one, so stages of 64 tokens x 64 channels of either operand are transposed on their way
// into LDS: a thread takes two channels of two tokens, swaps the inner halves, and stores two token pairs.  Threads are
// dealt 8 channel pairs x 8 token pairs to a wave: 32-byte runs of memory, and both the stores and the fragment reads
// (16 bytes at a pitch of 36 words) spread over all LDS banks.  The library's product has M * N / 4096 blocks and walks all
// tokens in each (25088 x 384 x 96: 93 us); here the tokens are split over the grid.
// Bound by one trip to memory per stage, and by how often the operands cross from the memory side into an L2: the blocks of one
// split, which read the same tokens, are dealt to one XCD where there are eight splits to deal, and the loads of two stages are in
// flight during a third's products.  Against neighbouring blocks on eight XCDs and one stage ahead, bf16, tokens x M x N, us: 25088 x 384 x
// 96 20.4 -> 16.1, 25088 x 96 x 192 16.0 -> 11.7, 6272 x 768 x 192 18.3 -> 15.8, 250000 x 96 x 96 54.0 -> 32.7, 12544 x 768 x 384 40.2 -> 29.0;
// by the second stage and cheaper addresses alone, fewer than eight splits not being placed: 32768 x 1024 x 768 215 -> 142.  (Halves of a
// block that take stages in turn and add up in LDS, half the atomics, 15 % slower and more; the splits % 8 that remain each on an XCD of its own
// too instead of spread, 12544 x 768 x 384 29 -> 39, or split counts rounded up, 32.)
template <typename T>
__global__ __launch_bounds__(256) void wgrad_tokens_kernel(const T *a, const T *c, int64_t tokens, int M, int N, int splits, float *out, float *bias) {
    constexpr int KT = 64, PW = KT / 2 + 4;         // tokens per stage; words per channel row
    __shared__ __align__(16) uint32_t sA[64 * PW], sC[64 * PW];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int nN = (N + 63) / 64, tiles = (M + 63) / 64 * nN;
    // blocks go to the eight XCDs in turn: eight splits at a time, each on an XCD of its own; the last splits % 8 spread over all
    const int whole = (splits & ~7) * tiles, i = blockIdx.x, rest = i - whole;
    const int tile = rest < 0 ? (i >> 3) % tiles : rest % tiles, split = rest < 0 ? (i >> 3) / tiles * 8 + (i & 7) : (splits & ~7) + rest / tiles;
    const int m0 = tile / nN * 64, n0 = tile % nN * 64;
    const int64_t per = ((tokens + splits - 1) / splits + KT - 1) / KT * KT, k0 = split * per, k1 = min(k0 + per, tokens);
    if (k0 >= k1) return;
    // item k of this thread: channel pair cp, token pair tp = lane bits 3-5 + 8 * k; the wave index selects 8 of the 32 channel pairs
    const int cp = (lane & 7) + 8 * wave, tb = lane >> 3;
    const int ca = min(m0 + 2 * cp, M - 2), cc = min(n0 + 2 * cp, N - 2);       // (clamped channels: rows of the result that are not stored)
    struct Stage { uint32_t a[4][2], c[4][2]; } st[2];
    // the stage at token k: tokens past the last are read as the last (and masked where they are used)
    auto load = [&](Stage &s, int64_t k) {
        k = min(k, tokens - 1);
        const char *const pa = (const char *)(a + k * M + ca), *const pc = (const char *)(c + k * N + cc);
        const uint32_t last = (uint32_t)min(tokens - 1 - k, (int64_t)KT);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint64_t tok = min((uint32_t)(2 * (tb + 8 * i) + h), last);
                s.a[i][h] = *(const uint32_t *)(pa + tok * (2u * (uint32_t)M));
                s.c[i][h] = *(const uint32_t *)(pc + tok * (2u * (uint32_t)N));
            }
    };
    f32x4 acc[2][2] = {};
    float bsum[2] = {};
    const bool sums = bias != nullptr && n0 == 0;
    auto step = [&](Stage &s, int64_t k) {
        __syncthreads();
        const int left = (int)max(min(k1 - k, (int64_t)KT), (int64_t)0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int tp = tb + 8 * i;
            const uint32_t keep = (2 * tp < left ? 0xffffu : 0u) | (2 * tp + 1 < left ? 0xffff0000u : 0u);
            // (low half of each word: the even channel) -> words of two tokens per channel
            const uint32_t e = ((s.a[i][0] & 0xffffu) | (s.a[i][1] << 16)) & keep, o = ((s.a[i][0] >> 16) | (s.a[i][1] & 0xffff0000u)) & keep;
            sA[(2 * cp) * PW + tp] = e;
            sA[(2 * cp + 1) * PW + tp] = o;
            sC[(2 * cp) * PW + tp] = ((s.c[i][0] & 0xffffu) | (s.c[i][1] << 16)) & keep;
            sC[(2 * cp + 1) * PW + tp] = ((s.c[i][0] >> 16) | (s.c[i][1] & 0xffff0000u)) & keep;
            if (sums) {
                bsum[0] += raw_to_f32((const T *)nullptr, e & 0xffffu) + raw_to_f32((const T *)nullptr, e >> 16);
                bsum[1] += raw_to_f32((const T *)nullptr, o & 0xffffu) + raw_to_f32((const T *)nullptr, o >> 16);
            }
        }
        __syncthreads();
        load(s, k + 2 * KT);
#pragma unroll
        for (int ks = 0; ks < KT; ks += 32) {
            Frag<T> fa[2], fc[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int w = (ks + (lane >> 4) * 8) / 2;
                __builtin_memcpy(fa[i].v, &sA[((wave >> 1) * 32 + 16 * i + (lane & 15)) * PW + w], 16);
                __builtin_memcpy(fc[i].v, &sC[((wave & 1) * 32 + 16 * i + (lane & 15)) * PW + w], 16);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = mma(fa[i], fc[j], acc[i][j]);
        }
    };
    load(st[0], k0);
    load(st[1], k0 + KT);
    for (int64_t k = k0; k < k1; k += 2 * KT) {
        step(st[0], k);
        if (k + KT < k1) step(st[1], k + KT);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + (wave >> 1) * 32 + 16 * i + (lane >> 4) * 4 + e, n = n0 + (wave & 1) * 32 + 16 * j + (lane & 15);
                if (m < M && n < N) glb_add(out + (int64_t)m * N + n, acc[i][j][e]);
            }
    if (sums) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float v = bsum[h];
            v += __shfl_xor(v, 8);
            v += __shfl_xor(v, 16);
            v += __shfl_xor(v, 32);
            if (lane < 8 && m0 + 2 * cp + h < M) glb_add(bias + m0 + 2 * cp + h, v);
        }
    }
}

// What the block's parameters are taken as: A = -exp(A_logs), the projection's weights in the activations' type and, for the
// backward, their transpose.  One launch instead of five.
template <typename T>
__global__ __launch_bounds__(256) void params_kernel(const float *A_logs, int nA, const float *wx, int rows, int cols, float *A, T *w, T *wt) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < nA) A[i] = -expf(A_logs[i]);
    if (i < rows * cols) {
        stg(w, i, wx[i]);
        if (wt) {                                   // (reads spaced by a row: a few ten thousand elements, all in the L2)
            const int c = i / rows, r = i - c * rows;
            stg(wt, i, wx[(int64_t)r * cols + c]);
        }
    }
}

bool shape_ok(const snd_block_shape *s) {
    return s && s->batch > 0 && s->nrows > 0 && s->ncols > 0 && s->inner > 0 && s->n_groups > 0 && s->dstate > 0 && s->rank > 0 &&
           s->rank <= SND_BLOCK_MAX_RANK && (int64_t)s->batch * s->n_groups < 65536 && (s->dtype == SND_F32 || s->dtype == SND_F16 || s->dtype == SND_BF16);
}
int launched() { return hipGetLastError() == hipSuccess ? SND_OK : SND_ERR_LAUNCH; }
// f(T *) with the element type of `dtype`
template <typename F> int by_type(int dtype, F f) {
    if (dtype == SND_F32) f((float *)nullptr);
    else if (dtype == SND_BF16) f((bf16_t *)nullptr);
    else if (dtype == SND_F16) f((f16_t *)nullptr);
    else return SND_ERR_DTYPE;
    return launched();
}
template <typename F> int by_types(int a, int b, F f) {
    int st = SND_ERR_DTYPE;
    by_type(a, [&](auto ea) { st = by_type(b, [&](auto eb) { f(ea, eb); }); });
    return st;
}
// f(lanes per token, channels per lane)
template <typename F> void by_channels(int C, F f) {
    std::integral_constant<int, 16> narrow;
    std::integral_constant<int, 64> wide;
    if (C <= 64) f(narrow, std::integral_constant<int, 4>());
    else if (C <= 128) f(narrow, std::integral_constant<int, 8>());
    else if (C <= 256) f(narrow, std::integral_constant<int, 16>());
    else if (C <= 512) f(wide, std::integral_constant<int, 8>());
    else f(wide, std::integral_constant<int, 16>());
}
template <typename F> void by_rank(int R, F f) {
    if (R <= 8) f(std::integral_constant<int, 8>());
    else if (R <= 16) f(std::integral_constant<int, 16>());
    else if (R <= 32) f(std::integral_constant<int, 32>());
    else f(std::integral_constant<int, 64>());
}
// Whether pixel maps of HW elements can be taken two pixels at a time (every row of every tensor starts on an even element).
bool px_pairs(int64_t HW, std::initializer_list<const void *> ptrs) {
    bool ok = HW % 2 == 0;
    for (const void *p : ptrs) ok = ok && ((uintptr_t)p & 3) == 0;
    return ok;
}
#define ELT(x) typename std::remove_pointer<decltype(x)>::type

}  // namespace
}  // namespace snd

using namespace snd;

int snd_block_norm_fwd(const void *x, int x_dtype, const float *gamma, const float *beta, float eps, int64_t tokens, int channels, void *y, int y_dtype,
                       float *stats, snd_stream_t stream) {
    if (!x || !y || !gamma || !beta) return SND_ERR_NULL;
    if (tokens <= 0 || channels <= 0 || channels > SND_BLOCK_MAX_NORM || (tokens + 3) / 4 >= ((int64_t)1 << 31)) return SND_ERR_SHAPE;
    return by_types(x_dtype, y_dtype, [&](auto ex, auto ey) {
        typedef ELT(ex) TX;
        typedef ELT(ey) TY;
        by_channels(channels, [&](auto gl, auto cpl) {
            constexpr int NG = 256 / decltype(gl)::value;
            hipLaunchKernelGGL((norm_fwd_kernel<TX, TY, decltype(gl)::value, decltype(cpl)::value>), dim3((unsigned)((tokens + NG - 1) / NG)), dim3(256), 0, (hipStream_t)stream,
                               (const TX *)x, gamma, beta, eps, tokens, channels, (TY *)y, stats);
        });
    });
}
int snd_block_norm_bwd(const void *dy, int dy_dtype, const void *x, int x_dtype, const float *gamma, const float *stats, int64_t tokens, int channels,
                       void *dx, float *dgamma, float *dbeta, snd_stream_t stream) {
    if (!dy || !x || !gamma || !stats || !dx || !dgamma || !dbeta) return SND_ERR_NULL;
    if (tokens <= 0 || channels <= 0 || channels > SND_BLOCK_MAX_NORM) return SND_ERR_SHAPE;
    return by_types(x_dtype, dy_dtype, [&](auto ex, auto ey) {
        typedef ELT(ex) TX;
        typedef ELT(ey) TY;
        by_channels(channels, [&](auto gl, auto cpl) {
            constexpr int GL = decltype(gl)::value, NT = norm_threads(GL), NG = NT / GL;
            const int grid = (int)std::min<int64_t>((tokens + NG - 1) / NG, 256 * 1024 / NT);
            hipLaunchKernelGGL((norm_bwd_kernel<TX, TY, GL, decltype(cpl)::value>), dim3(grid), dim3(NT), 0, (hipStream_t)stream, (const TY *)dy, (const TX *)x,
                               gamma, stats, tokens, channels, (TX *)dx, dgamma, dbeta);
        });
    });
}
int snd_block_params(const float *A_logs, int nA, const float *wx, int rows, int cols, int dtype, float *A, void *w, void *wt, snd_stream_t stream) {
    if (!A_logs || !wx || !A || !w) return SND_ERR_NULL;
    if (nA <= 0 || rows <= 0 || cols <= 0 || (int64_t)rows * cols >= (int64_t)1 << 31) return SND_ERR_SHAPE;
    return by_type(dtype, [&](auto e) {
        typedef ELT(e) T;
        hipLaunchKernelGGL((params_kernel<T>), dim3((unsigned)((std::max((int64_t)nA, (int64_t)rows * cols) + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                           A_logs, nA, wx, rows, cols, A, (T *)w, (T *)wt);
    });
}
static dim3 conv_grid(const snd_block_shape &s) {
    return dim3((unsigned)(((s.nrows + kCvR - 1) / kCvR) * ((s.ncols + kCvX - 1) / kCvX)), (unsigned)((s.inner + kCvC - 1) / kCvC), (unsigned)s.batch);
}
int snd_block_conv_fwd(const snd_block_shape *s, const void *xz, const float *w, const float *bias, void *pre, void *u, snd_stream_t stream) {
    if (!shape_ok(s)) return SND_ERR_SHAPE;
    if (!xz || !w || !u) return SND_ERR_NULL;
    return by_type(s->dtype, [&](auto e) {
        typedef ELT(e) T;
        hipLaunchKernelGGL((conv_fwd_kernel<T>), conv_grid(*s), dim3(256), 0, (hipStream_t)stream, *s, (const T *)xz, w, bias, (T *)pre, (T *)u);
    });
}
int snd_block_conv_bwd(const snd_block_shape *s, const void *du, const void *pre, const void *xz, const float *w, void *dxz, float *dw, float *dbias,
                       snd_stream_t stream) {
    if (!shape_ok(s)) return SND_ERR_SHAPE;
    if (!du || !pre || !xz || !w || !dxz || !dw) return SND_ERR_NULL;
    return by_type(s->dtype, [&](auto e) {
        typedef ELT(e) T;
        hipLaunchKernelGGL((conv_bwd_kernel<T>), conv_grid(*s), dim3(256), 0, (hipStream_t)stream, *s, (const T *)du, (const T *)pre, (const T *)xz, w,
                           (T *)dxz, dw, dbias);
    });
}
static dim3 gate_grid(const snd_block_shape &s) { return dim3((unsigned)(((int64_t)s.nrows * s.ncols + kGtP - 1) / kGtP), (unsigned)s.batch); }
int snd_block_gate_fwd(const snd_block_shape *s, const float *y, const void *xz, const float *gamma, const float *beta, float eps, void *out, float *stats,
                       snd_stream_t stream) {
    if (!shape_ok(s)) return SND_ERR_SHAPE;
    if (!y || !xz || !gamma || !beta || !out) return SND_ERR_NULL;
    return by_type(s->dtype, [&](auto e) {
        typedef ELT(e) T;
        hipLaunchKernelGGL((gate_fwd_kernel<T>), gate_grid(*s), dim3(kGtT), 0, (hipStream_t)stream, *s, y, (const T *)xz, gamma, beta, eps, (T *)out, stats);
    });
}
int snd_block_gate_bwd(const snd_block_shape *s, const void *dout, const float *y, const void *xz, const float *gamma, const float *beta, const float *stats,
                       float *dy, void *dxz, float *dgamma, float *dbeta, snd_stream_t stream) {
    if (!shape_ok(s)) return SND_ERR_SHAPE;
    if (!dout || !y || !xz || !gamma || !beta || !stats || !dy || !dxz || !dgamma || !dbeta) return SND_ERR_NULL;
    return by_type(s->dtype, [&](auto e) {
        typedef ELT(e) T;
        hipLaunchKernelGGL((gate_bwd_kernel<T>), gate_grid(*s), dim3(kGtT), 0, (hipStream_t)stream, *s, (const T *)dout, y, (const T *)xz, gamma, beta, stats,
                           dy, (T *)dxz, dgamma, dbeta);
    });
}
int snd_block_dt_fwd(const snd_block_shape *s, const void *proj, const float *w, void *delta, snd_stream_t stream) {
    if (!shape_ok(s)) return SND_ERR_SHAPE;
    if (!proj || !w || !delta) return SND_ERR_NULL;
    const int64_t HW = (int64_t)s->nrows * s->ncols;
    return by_type(s->dtype, [&](auto e) {
        typedef ELT(e) T;
        by_rank(s->rank, [&](auto rp) {
            auto go = [&](auto kernel, int V) {
                const int64_t bx = (HW + 256 * V - 1) / (256 * V), blocks = bx * s->batch * s->n_groups;
                const int share = (int)std::min<int64_t>(std::max<int64_t>(1, 2048 / blocks), std::max(1, s->inner / 16));
                hipLaunchKernelGGL(kernel, dim3((unsigned)bx, (unsigned)(s->batch * s->n_groups), (unsigned)share), dim3(256), 0, (hipStream_t)stream, *s,
                                   (const T *)proj, w, (T *)delta);
            };
            px_pairs(HW, {proj, delta}) ? go(dt_fwd_kernel<T, decltype(rp)::value, 2>, 2) : go(dt_fwd_kernel<T, decltype(rp)::value, 1>, 1);
        });
    });
}
int snd_block_dt_bwd(const snd_block_shape *s, const void *ddelta, const void *dB, const void *dC, const float *w, void *dproj, snd_stream_t stream) {
    if (!shape_ok(s)) return SND_ERR_SHAPE;
    if (!ddelta || !dB || !dC || !w || !dproj) return SND_ERR_NULL;
    const int64_t HW = (int64_t)s->nrows * s->ncols;
    return by_type(s->dtype, [&](auto e) {
        typedef ELT(e) T;
        by_rank(s->rank, [&](auto rp) {
            auto go = [&](auto kernel, int V) {
                hipLaunchKernelGGL(kernel, dim3((unsigned)((HW + 64 * V - 1) / (64 * V)), (unsigned)(s->batch * s->n_groups)), dim3(256), 0, (hipStream_t)stream,
                                   *s, (const T *)ddelta, (const T *)dB, (const T *)dC, w, (T *)dproj);
            };
            px_pairs(HW, {ddelta, dB, dC, dproj}) ? go(dt_bwd_kernel<T, decltype(rp)::value, 2>, 2) : go(dt_bwd_kernel<T, decltype(rp)::value, 1>, 1);
        });
    });
}
int snd_block_wgrad(const void *a, int64_t a_batch, int64_t a_group, const void *c, int64_t c_batch, int64_t c_group, int batch, int groups, int M, int N,
                    int64_t pixels, int dtype, float *out, snd_stream_t stream) {
    if (!a || !c || !out) return SND_ERR_NULL;
    if (batch <= 0 || groups <= 0 || groups > 65535 || M <= 0 || N <= 0 || pixels <= 0) return SND_ERR_SHAPE;
    return by_type(dtype, [&](auto e) {
        typedef ELT(e) T;
        constexpr int FK = Frag<T>::K;
        const bool vec = (((uintptr_t)a | (uintptr_t)c) & 15) == 0 && pixels % FK == 0 && a_batch % FK == 0 && a_group % FK == 0 && c_batch % FK == 0 &&
                         c_group % FK == 0;
        // a narrow side (the rank of the step-size projection) takes one column of tiles
        const bool narrow = N <= 16;
        const int tiles = ((M + 63) / 64) * (narrow ? 1 : (N + 63) / 64);
        // pixels are split until the grid has about four blocks per CU, in shares of 256 and more
        int splits = (int)std::min<int64_t>(std::max<int64_t>(1, 1024 / ((int64_t)tiles * batch * groups)), std::max<int64_t>(1, pixels / 256));
        while ((int64_t)splits * batch > 65535 && splits > 1) --splits;
        const dim3 grid((unsigned)tiles, (unsigned)(batch * splits), (unsigned)groups);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, (const T *)a, a_batch, a_group, (const T *)c, c_batch, c_group, M, N, pixels,
                               splits, out);
        };
        if (narrow) vec ? go(wgrad_kernel<T, 1, 1, 4, 1, true>) : go(wgrad_kernel<T, 1, 1, 4, 1, false>);
        else vec ? go(wgrad_kernel<T, 2, 2, 2, 2, true>) : go(wgrad_kernel<T, 2, 2, 2, 2, false>);
    });
}
int snd_block_linear_wgrad(const void *dy, const void *x, int64_t tokens, int M, int N, int dtype, float *dw, float *dbias, snd_stream_t stream) {
    if (!dy || !x || !dw) return SND_ERR_NULL;
    if (tokens <= 0 || M <= 0 || N <= 0 || M % 2 || N % 2 || (((uintptr_t)dy | (uintptr_t)x) & 3)) return SND_ERR_SHAPE;
    if (dtype != SND_BF16 && dtype != SND_F16) return SND_ERR_DTYPE;
    const int64_t tiles = (int64_t)((M + 63) / 64) * ((N + 63) / 64);
    if (tiles >= (int64_t)1 << 31) return SND_ERR_SHAPE;
    // Splits of 256 tokens, as many as give 768 blocks.  From 32 splits on they are whole rounds of the XCDs (9984 x 192 x 384, 39 splits,
    // 15.5 -> 14.9 us; 25088 x 96 x 192, 98, 15.5 -> 13.2), where the last of them only make the others longer; fewer would get
    // noticeably longer and larger in error (3837 x 64 x 64, 15 splits, 6.2 -> 8.6 us and 1.1e-7 -> 1.4e-7 as eight), and so would splits that are
    // few because of the tiles (32768 x 768 x 192, 21 splits, 34.8 -> 40.0 us and 2.5e-7 -> 2.8e-7 as 16).
    int splits = (int)std::min<int64_t>(std::max<int64_t>(1, 768 / tiles), (tokens + 255) / 256);
    if (splits >= 32 && splits == (tokens + 255) / 256) splits &= ~7;
    const dim3 grid((unsigned)(tiles * splits));
    if (dtype == SND_BF16)
        hipLaunchKernelGGL((wgrad_tokens_kernel<bf16_t>), grid, dim3(256), 0, (hipStream_t)stream, (const bf16_t *)dy, (const bf16_t *)x, tokens, M, N, splits, dw, dbias);
    else
        hipLaunchKernelGGL((wgrad_tokens_kernel<f16_t>), grid, dim3(256), 0, (hipStream_t)stream, (const f16_t *)dy, (const f16_t *)x, tokens, M, N, splits, dw, dbias);
    return launched();
}
