// Conversion of a BF16 weight: the passes around the encoders, each one read and one write.
//
// Stands in for the tensor operations of the reference's compress_split_n
// (bf16_huffman_infer/functional.py:195-238).  As operations of a tensor library the planes, the task
// order, the pair histogram and the placing of the streams were over a hundred kernels that passed a
// 12288x4096 weight through memory as 32- and 64-bit integers, 2.9 ms in all.  Here: split_planes 34 us
// (bound by memory: 100 MB in, 100 MB out, 5.9 TB/s), pair_histogram 23 us (bound by LDS atomics),
// place_streams 4 us per chunk.
#include "bhi_task.h"

namespace bhi {

// BF16 [M, K] -> the rem plane as it is stored ([split][group][step][lane][column], bhi_common.h) and the
// exponents in task order: chunk by chunk, tasks (split, group) of a chunk one after the other, the same
// step order inside.  A thread owns one lane of one step: sixteen bytes in, eight out twice; a wavefront
// reads 256 contiguous bytes of four rows and writes 512 contiguous bytes.
__global__ __launch_bounds__(kBlockThreads)
void split_planes_kernel(const uint16_t* __restrict__ W, uint2* __restrict__ rem, uint2* __restrict__ exp, Shape s) {
    const int G = s.M / kGroupRows, K = s.Ks * s.split_k;
    const int lane = threadIdx.x & (kLanes - 1);
    const long long step = (long long)blockIdx.x * kWavesPerBlock + threadIdx.x / kLanes;      // (split, group, step)
    if (step >= (long long)s.split_k * G * s.steps) return;
    const int t = (int)(step % s.steps);
    const long long kg = step / s.steps;
    const int k = (int)(kg / G), g = (int)(kg % G);
    // (two-byte loads where the weight is not aligned to sixteen)
    const uint16_t* p = W + (size_t)(kGroupRows * g + (lane & 3)) * K + (size_t)k * s.Ks + (size_t)t * kStepCols + (lane >> 2) * kLaneCols;
    uint16_t v[kLaneCols];
    if (((uintptr_t)W & 15) == 0) {
        const uint4 q = *(const uint4*)p;
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int j = 0; j < kLaneCols; ++j) v[j] = (uint16_t)(w[j / 2] >> (16 * (j & 1)));
    } else {
#pragma unroll
        for (int j = 0; j < kLaneCols; ++j) v[j] = p[j];
    }
    uint32_t r[2] = {0, 0}, e[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < kLaneCols; ++j) {
        r[j / 4] |= (uint32_t)((v[j] >> 8 & 0x80) | (v[j] & 0x7F)) << (8 * (j & 3));
        e[j / 4] |= (uint32_t)(v[j] >> 7 & 0xFF) << (8 * (j & 3));
    }
    rem[step * kLanes + lane] = make_uint2(r[0], r[1]);
    int c = 0;
    while (t >= (s.steps * (c + 1)) >> s.nc_log2) ++c;                     // the chunk of step t (task_of)
    const int t0 = (s.steps * c) >> s.nc_log2, t1 = (s.steps * (c + 1)) >> s.nc_log2;
    const long long at = (long long)s.split_k * G * t0 + kg * (t1 - t0) + (t - t0);
    exp[at * kLanes + lane] = make_uint2(e[0], e[1]);
}

// Occurrences of every exponent pair a | b << 8 (a = even column) among 8-byte groups of one row's
// exponents.  Weights use a few dozen exponents: pairs below 200 x 200 are counted in LDS (160 000
// bytes, one block per compute unit) and added to the result once per block, others there directly.
constexpr int kHistSide = 200, kHistThreads = 1024;
__global__ __launch_bounds__(kHistThreads)
void pair_histogram_kernel(const uint2* __restrict__ exp, long long n, unsigned long long* __restrict__ counts) {
    __shared__ uint32_t bins[kHistSide * kHistSide];
    for (int i = threadIdx.x; i < kHistSide * kHistSide; i += kHistThreads) bins[i] = 0;
    __syncthreads();
    for (long long i = (long long)blockIdx.x * kHistThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kHistThreads) {
        const uint2 d = exp[i];
        const uint32_t pair[4] = {d.x & 0xFFFFu, d.x >> 16, d.y & 0xFFFFu, d.y >> 16};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t a = pair[j] & 0xFFu, b = pair[j] >> 8;
            if (a < kHistSide && b < kHistSide) atomicAdd(&bins[b * kHistSide + a], 1u);
            else atomicAdd(&counts[pair[j]], 1ull);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kHistSide * kHistSide; i += kHistThreads)
        if (bins[i]) atomicAdd(&counts[(i % kHistSide) | (i / kHistSide) << 8], (unsigned long long)bins[i]);
}

// Streams of the encoders (row `task` of [n_tasks, stride], lengths[task] words of it) to their places
// in the exponent stream.  Lengths, places and strides are multiples of four words.
__global__ __launch_bounds__(kBlockThreads)
void place_streams_kernel(const uint4* __restrict__ streams, long long stride, const uint32_t* __restrict__ lengths,
                          const long long* __restrict__ starts, long long starts_stride, uint4* __restrict__ words, long long n_words) {
    const long long task = blockIdx.x, start = starts[task * starts_stride] / 4;
    const uint32_t n = lengths[task] / 4;
    if (start < 0 || start + n > n_words / 4 || n > stride / 4) return;
    const uint4* src = streams + task * (stride / 4);
    for (uint32_t i = threadIdx.x; i < n; i += kBlockThreads) words[start + i] = src[i];
}

}  // namespace bhi

using namespace bhi;

extern "C" int bhi_split_planes(const void* W, void* rem, void* exp, int split_k, int M, int Ks, void* stream) {
    if (!W || !rem || !exp) return bhi_fail(BHI_EINVAL, "null pointer");
    Shape s;
    if (int rc = check_shape(split_k, M, Ks, kTailPadWords, &s)) return rc;
    const long long steps = (long long)split_k * (M / kGroupRows) * s.steps;
    const long long blocks = (steps + kWavesPerBlock - 1) / kWavesPerBlock;
    if (blocks > 0x7FFFFFFFll) return bhi_fail(BHI_EINVAL, "weight too large for one launch");
    hipLaunchKernelGGL(split_planes_kernel, dim3((unsigned)blocks), dim3(kBlockThreads), 0, (hipStream_t)stream,
                       (const uint16_t*)W, (uint2*)rem, (uint2*)exp, s);
    return bhi_launch_status("split_planes");
}

extern "C" int bhi_pair_histogram(const void* exp, int64_t bytes, void* counts, void* stream) {
    if (!exp || !counts) return bhi_fail(BHI_EINVAL, "null pointer");
    if (bytes < kLaneCols || bytes % kLaneCols != 0) return bhi_fail(BHI_EINVAL, "exponents come in groups of eight");
    if (bytes / 2 / 256 >= (int64_t)1 << 32) return bhi_fail(BHI_EINVAL, "more exponents than 32-bit counts per block hold");
    const long long n = bytes / kLaneCols, blocks = (n + kHistThreads - 1) / kHistThreads;
    hipLaunchKernelGGL(pair_histogram_kernel, dim3((unsigned)(blocks < 256 ? blocks : 256)), dim3(kHistThreads), 0, (hipStream_t)stream,
                       (const uint2*)exp, n, (unsigned long long*)counts);
    return bhi_launch_status("pair_histogram");
}

extern "C" int bhi_place_streams(const void* streams, int64_t stride, const void* lengths, const void* starts, int64_t starts_stride,
                                 int n_tasks, void* words, int64_t n_words, void* stream) {
    if (!streams || !lengths || !starts || !words) return bhi_fail(BHI_EINVAL, "null pointer");
    if (n_tasks < 1 || stride % kAlignWords != 0) return bhi_fail(BHI_EINVAL, "need n_tasks >= 1 and a stride of whole 16-byte pieces");
    hipLaunchKernelGGL(place_streams_kernel, dim3((unsigned)n_tasks), dim3(kBlockThreads), 0, (hipStream_t)stream,
                       (const uint4*)streams, (long long)stride, (const uint32_t*)lengths, (const long long*)starts,
                       (long long)starts_stride, (uint4*)words, (long long)n_words);
    return bhi_launch_status("place_streams");
}
