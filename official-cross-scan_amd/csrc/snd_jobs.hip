// The small passes around the scan kernels of a call - clearing what they accumulate into, and folding or casting what they
// leave - as jobs of one launch each side: a pass over a few KB costs its launch, not its bytes (a merged training call on
// 2 x 384 x 14x14 made 15 launches around its two kernels, 2 to 4 us each on the GPU and 3 to 5 on the host).
#include <type_traits>

#include "snd_device.h"

namespace snd {
namespace {

constexpr int kMaxJobs = 8, kThreads = 256;
constexpr int kClearBytes = kThreads * 16 * 4;      // per block: four 16-byte stores per thread in flight

struct Job {
    const void *in, *in2;
    void *out;
    int64_t units, per;                             // work items of the job, and items per (outer) row
    int64_t M, bytes;
    int32_t R, kind, in_dtype, out_dtype, vec, split, first;    // first: the job's first block
};
struct Jobs { Job j[kMaxJobs]; int n; };

// V neighbouring values as they are loaded
template <typename T, int V> struct Held;
template <typename T> struct Held<T, 1> {
    float v;
    __device__ __forceinline__ void load(const T *p) { v = ldg(p, 0); }
    __device__ __forceinline__ void add(float (&acc)[1]) const { acc[0] += v; }
};
template <typename T> struct Held<T, 4> {
    Raw4<T> q;
    __device__ __forceinline__ void load(const T *p) { ldraw4_b(q, p, 0); }
    __device__ __forceinline__ void add(float (&acc)[4]) const {
        float t[4];
        raw4_to_f32(q, t);
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[k] += t[k];
    }
};
template <typename T, int V> __device__ __forceinline__ void st_vec(T *p, const float (&v)[V]) {
    if constexpr (V == 1) {
        stg(p, 0, v[0]);
    } else {
#pragma unroll
        for (int k = 0; k < V; k += 4) {
            const float t[4] = {v[k], v[k + 1], v[k + 2], v[k + 3]};
            stg4_b(p, k * (uint32_t)sizeof(T), t);
        }
    }
}
// out[o*M + i] = sum over r < R of in[(o*R + r)*M + i], added up in fp32.  A thread requests its rows eight (fp32: four) at a
// time: one after the other they cost a load latency each.
template <int ROWS, typename TI, int V> __device__ __forceinline__ void add_batch(const TI *&src, int64_t M, float (&acc)[V]) {
    Held<TI, V> h[ROWS];                            // (kept as they are loaded: 16 registers, so that waves stay at eight per SIMD)
#pragma unroll
    for (int q = 0; q < ROWS; ++q) h[q].load(src + q * M);
#pragma unroll
    for (int q = 0; q < ROWS; ++q) h[q].add(acc);
    src += ROWS * M;
}
template <typename TI, int V> __device__ __forceinline__ void add_rows(const TI *src, int64_t M, int rows, float (&acc)[V]) {
    constexpr int ROWS = sizeof(TI) == 2 ? 8 : 4;
    for (; rows >= ROWS; rows -= ROWS) add_batch<ROWS, TI, V>(src, M, acc);
    if (ROWS > 4 && rows >= 4) {
        add_batch<4, TI, V>(src, M, acc);
        rows -= 4;
    }
    if (rows >= 2) {
        add_batch<2, TI, V>(src, M, acc);
        rows -= 2;
    }
    if (rows > 0) add_batch<1, TI, V>(src, M, acc);
}
// A thread takes a unit (V columns) with all its rows; split: a block takes kUnits units, with their rows dealt to kThreads /
// kUnits slices that are added up in LDS (runs of 128 bytes for 16-bit values).
constexpr int kUnits = 16, kSlices = kThreads / kUnits;
template <typename TI, typename TO, int V> __device__ __forceinline__ void sum_rows(const Job &j, uint32_t blk, float *part) {
    const int lane = threadIdx.x % kUnits, slice = threadIdx.x / kUnits;
    const int64_t unit = j.split ? (int64_t)blk * kUnits + lane : (int64_t)blk * kThreads + threadIdx.x, uc = min(unit, j.units - 1);
    const int64_t o = j.units >> 32 ? uc / j.per : (uint32_t)uc / (uint32_t)j.per, i = (uc - o * j.per) * V;
    const TI *src = (const TI *)j.in + (o * j.R * j.M + i);
    TO *dst = (TO *)j.out + (o * j.M + i);
    float acc[V] = {};
    if (!j.split) {
        if (unit >= j.units) return;
        add_rows<TI, V>(src, j.M, j.R, acc);
        st_vec<TO, V>(dst, acc);
        return;
    }
    const int n = (j.R + kSlices - 1) / kSlices;
    const int r0 = min(slice * n, j.R);
    add_rows<TI, V>(src + r0 * j.M, j.M, min(n, j.R - r0), acc);
#pragma unroll
    for (int k = 0; k < V; ++k) part[(slice * kUnits + lane) * V + k] = acc[k];
    __syncthreads();
    if (slice != 0 || unit >= j.units) return;
#pragma unroll 5
    for (int q = 1; q < kSlices; ++q)
#pragma unroll
        for (int k = 0; k < V; ++k) acc[k] += part[(q * kUnits + lane) * V + k];
    st_vec<TO, V>(dst, acc);
}
template <typename TI, typename TO> __device__ __forceinline__ void sum_rows_v(const Job &j, uint32_t blk, float *part) {
    if (j.vec) sum_rows<TI, TO, 4>(j, blk, part);
    else sum_rows<TI, TO, 1>(j, blk, part);
}
// Where the split pays: rows enough for the slices, and units for fewer than two blocks per CU, too few to hide the latency of a
// thread's walk.  A whole training call with one delta for all channels, one state, bf16, rows one at a time / eight at a
// time / split, us: 64 x 3072 x 7x7 (3072 rows of 784 units) 940 / 254 / 120, 8 x 768 x 28x28 276 / 94 / 58, 64 x 384 x 56x56
// (50176 units) 699 / 576 / 566; with a delta per group (96 rows of 200704 units) 583 / 570 / 577.
bool split_rows(int64_t units, int rows) { return rows >= 2 * kSlices && units < (int64_t)1 << 17; }
// Magnitude below which a merge weight enters the backward as this value (see snd_job)
__device__ __forceinline__ float floor_weight(float w) { return fabsf(w) < SND_MERGE_WEIGHT_FLOOR ? SND_MERGE_WEIGHT_FLOOR : w; }

__global__ __launch_bounds__(kThreads) void jobs_kernel(const Jobs a) {
    int k = 0;
    while (k + 1 < a.n && (int)blockIdx.x >= a.j[k + 1].first) ++k;
    const Job &j = a.j[k];
    const uint32_t blk = blockIdx.x - j.first;
    if (j.kind == SND_JOB_CLEAR) {
        const int64_t base = (int64_t)blk * kClearBytes + threadIdx.x * 16;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t o = base + q * kThreads * 16;
            char *dst = (char *)j.out + o;
            if (o + 16 <= j.bytes) *(uint4 *)dst = make_uint4(0, 0, 0, 0);
            else for (int e = 0; o + 4 * e < j.bytes && e < 4; ++e) ((uint32_t *)dst)[e] = 0;
        }
        return;
    }
    if (j.kind == SND_JOB_WEIGHT_GROUP) {           // one block per group: sum over its M channels
        __shared__ float part[kThreads / 64];
        float v = 0.f;
        for (int64_t i = threadIdx.x; i < j.M; i += kThreads) v += ((const float *)j.in)[blk * j.M + i] / floor_weight(((const float *)j.in2)[blk * j.M + i]);
        v = wave_sum_to_last(v);
        if ((threadIdx.x & 63) == 63) part[threadIdx.x >> 6] = v;
        __syncthreads();
        if (threadIdx.x == 0) ((float *)j.out)[blk] = (part[0] + part[1]) + (part[2] + part[3]);
        return;
    }
    if (j.kind == SND_JOB_SUM) {
        __shared__ float part[kThreads * 4];
        if (j.in_dtype == SND_F32) {
            if (j.out_dtype == SND_F32) sum_rows_v<float, float>(j, blk, part);
            else if (j.out_dtype == SND_BF16) sum_rows_v<float, bf16_t>(j, blk, part);
            else sum_rows_v<float, f16_t>(j, blk, part);
        } else if (j.in_dtype == SND_BF16) {
            sum_rows_v<bf16_t, bf16_t>(j, blk, part);
        } else {
            sum_rows_v<f16_t, f16_t>(j, blk, part);
        }
        return;
    }
    const int64_t unit = (int64_t)blk * kThreads + threadIdx.x;
    if (unit >= j.units) return;
    if (j.kind == SND_JOB_WEIGHT) ((float *)j.out)[unit] = ((const float *)j.in)[unit] / floor_weight(((const float *)j.in2)[unit]);
    else ((float *)j.out)[unit] = floor_weight(((const float *)j.in)[unit]);
}

}  // namespace
}  // namespace snd

extern "C" int snd_run_jobs(const snd_job *jobs, int n, snd_stream_t stream) {
    if (!jobs || n < 0 || n > snd::kMaxJobs) return SND_ERR_NULL;
    snd::Jobs a;
    a.n = 0;
    int64_t blocks = 0;
    for (int k = 0; k < n; ++k) {
        const snd_job &q = jobs[k];
        snd::Job j{};
        j.in = q.in; j.in2 = q.in2; j.out = q.out;
        j.kind = q.kind; j.in_dtype = q.in_dtype; j.out_dtype = q.out_dtype;
        j.first = (int32_t)blocks;
        int64_t nb = 0;
        if (q.kind == SND_JOB_CLEAR) {
            if (q.outer <= 0) continue;
            if (!q.out || ((uintptr_t)q.out & 15) || q.outer % 4) return SND_ERR_ALIGN;
            j.bytes = q.outer;
            nb = (q.outer + snd::kClearBytes - 1) / snd::kClearBytes;
        } else {
            const int64_t total = q.outer * q.cols;
            if (total <= 0) continue;
            if (!q.in || !q.out || q.rows < 1) return SND_ERR_NULL;
            j.M = q.cols; j.R = q.rows;
            if (q.kind == SND_JOB_WEIGHT_GROUP) {
                if (!q.in2) return SND_ERR_NULL;
                nb = q.outer;
            } else {
                if (q.kind == SND_JOB_WEIGHT && !q.in2) return SND_ERR_NULL;
                if (q.kind < SND_JOB_CLEAR || q.kind > SND_JOB_WEIGHT_FLOOR) return SND_ERR_SHAPE;
                if (q.kind == SND_JOB_SUM && q.in_dtype != SND_F32 && q.out_dtype != q.in_dtype) return SND_ERR_DTYPE;
                const int ei = q.in_dtype == SND_F32 ? 4 : 2, eo = q.out_dtype == SND_F32 ? 4 : 2;
                j.vec = q.kind == SND_JOB_SUM && q.cols % 4 == 0 && (uintptr_t)q.in % (4 * ei) == 0 && (uintptr_t)q.out % (4 * eo) == 0;
                const int64_t units = total / (j.vec ? 4 : 1);
                j.units = units;
                j.per = q.cols / (j.vec ? 4 : 1);
                j.split = q.kind == SND_JOB_SUM && snd::split_rows(units, q.rows);
                const int per_block = j.split ? snd::kUnits : snd::kThreads;
                nb = (units + per_block - 1) / per_block;
            }
        }
        blocks += nb;
        if (blocks >= (int64_t)1 << 31) return SND_ERR_SHAPE;
        a.j[a.n++] = j;
    }
    if (a.n == 0) return SND_OK;
    hipLaunchKernelGGL(snd::jobs_kernel, dim3((unsigned)blocks), dim3(snd::kThreads), 0, (hipStream_t)stream, a);
    return hipGetLastError() == hipSuccess ? SND_OK : SND_ERR_LAUNCH;
}
