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

// The pair code of a matrix (huffman.py, LUTHuffmanEncoder.build_lut): optimal code lengths of at most eleven bits for the
// most frequent pairs and ESC (package-merge), for four cut-offs; the cheapest, or an escape-free one that costs at
// most 1/32 more; canonical codes; the encoder's and the decoder's table.
//
// One block: 65536 counts, up to 1537 symbols, ten merges each of which needs the one before.  As Python lists
// this was 6.2 of the 17.7 ms that converting a 12288x4096 weight took (18.3 -> 12.4 ms in turn with it).  A merge is parallel: an element's
// place is its own index plus the number of elements of the other list in front of it (a binary search), and since the
// first k elements of a merged list are its first a leaves and its first k - a packages, all that has to be kept
// of a merge is where its leaves went.
constexpr int kCodeThreads = 1024, kMaxCoded = 1536, kCodeSymbols = kMaxCoded + 1;
constexpr uint32_t kEscIndex = 65536;
constexpr int kEscSideBits = 32, kEscFreeShift = 5;

// Elements of the ascending a[0..n) that are smaller than v (OR_EQUAL: or equal to it).
template <bool OR_EQUAL>
__device__ __forceinline__ int count_below(const unsigned long long* a, int n, unsigned long long v) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (OR_EQUAL ? a[mid] <= v : a[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// counts: descending, with ids[i] the pair of counts[i]; pairs of one count in ascending order.
// info: expected bits, code length of ESC, whether pairs escape; -1, 0, 0 and no tables for counts that are negative or
// not descending: the places of the leaves below come from searches that rely on the order.
__global__ __launch_bounds__(kCodeThreads)
void pair_code_kernel(const unsigned long long* __restrict__ counts, const long long* __restrict__ ids, uint32_t* __restrict__ enc,
                      uint32_t* __restrict__ dec, long long* __restrict__ info) {
    __shared__ unsigned long long leaves[kCodeSymbols], list[2][2 * kCodeSymbols], packs[kCodeSymbols];
    __shared__ uint16_t place[kTableBits][kCodeSymbols];                  // of every leaf in the list of a merge
    __shared__ uint16_t rank_of[kCodeSymbols];                            // of symbol i among the leaves
    __shared__ uint8_t lengths[2][kCodeSymbols];                          // of the cut-off at hand and of the best one
    __shared__ uint16_t id_of[kMaxCoded];
    __shared__ unsigned long long sums[2];
    __shared__ uint32_t unfit, seen[4], chosen[kTableBits], per_length[kTableBits + 2], first_code[kTableBits + 2];
    const int tid = threadIdx.x;
    if (tid < 2) sums[tid] = 0;
    if (tid < 4) seen[tid] = 0;
    if (tid == 0) unfit = 0;
    __syncthreads();
    {
        const unsigned long long least[4] = {1, 2, 4, 16};
        unsigned long long sum = 0;
        uint32_t n[4] = {0, 0, 0, 0};
        bool fits = true;
        for (int i = tid; i < 65536; i += kCodeThreads) {
            const unsigned long long c = counts[i];
            fits = fits && (long long)c >= 0 && (i == 0 || counts[i - 1] >= c);
            sum += c;
#pragma unroll
            for (int k = 0; k < 4; ++k) n[k] += c >= least[k] ? 1 : 0;
        }
        atomicAdd(&sums[0], sum);
#pragma unroll
        for (int k = 0; k < 4; ++k) atomicAdd(&seen[k], n[k]);
        if (!fits) atomicOr(&unfit, 1u);
    }
    __syncthreads();
    if (unfit) {
        if (tid < 3) info[tid] = tid == 0 ? -1 : 0;
        return;
    }
    for (int i = tid; i < kMaxCoded; i += kCodeThreads) id_of[i] = (uint16_t)ids[i];
    for (int i = tid; i <= (int)kEscIndex; i += kCodeThreads) enc[i] = 0;
    __syncthreads();
    const unsigned long long total = sums[0];
    const int present = (int)seen[0];

    unsigned long long best_bits = 0, free_bits = 0;
    int best = 0, last = 0, all_coded = 0;                                // symbols without ESC; 0: none yet
    unsigned long long best_escapes = 0;
    for (int cut = 0; cut < 4; ++cut) {
        int m = min((int)seen[cut], kMaxCoded);
        if (m == 0) m = 1;
        if (m == last) continue;
        last = m;
        const int n = m + 1;
        __syncthreads();
        if (tid == 0) sums[1] = 0;
        __syncthreads();
        unsigned long long part = 0;
        for (int i = tid; i < m; i += kCodeThreads) part += counts[i];
        atomicAdd(&sums[1], part);
        __syncthreads();
        const unsigned long long escapes = total - sums[1], esc = escapes > 1 ? escapes : 1;
        __syncthreads();
        // leaves in ascending order, of one weight in the order of the symbols: ESC is the last symbol
        for (int i = tid; i < m; i += kCodeThreads) packs[m - 1 - i] = counts[i];              // ascending
        __syncthreads();
        for (int i = tid; i < n; i += kCodeThreads) {
            int r;
            unsigned long long w;
            if (i < m) {
                w = packs[m - 1 - i];
                const int below = count_below<false>(packs, m, w), up_to = count_below<true>(packs, m, w);
                r = below + (i - (m - up_to)) + (esc < w ? 1 : 0);
            } else {
                w = esc;
                r = count_below<true>(packs, m, esc);
            }
            rank_of[i] = (uint16_t)r;
            leaves[r] = w;
        }
        __syncthreads();
        for (int i = tid; i < n; i += kCodeThreads) list[0][i] = leaves[i];
        int len = n, from = 0;
        for (int merge = 1; merge < kTableBits; ++merge) {
            __syncthreads();
            const int half = len / 2;
            for (int j = tid; j < half; j += kCodeThreads) packs[j] = list[from][2 * j] + list[from][2 * j + 1];
            __syncthreads();
            for (int i = tid; i < n; i += kCodeThreads) {                 // a leaf in front of packages of its weight
                const int at = i + count_below<false>(packs, half, leaves[i]);
                place[merge][i] = (uint16_t)at;
                list[from ^ 1][at] = leaves[i];
            }
            for (int j = tid; j < half; j += kCodeThreads) list[from ^ 1][j + count_below<true>(leaves, n, packs[j])] = packs[j];
            from ^= 1;
            len = n + half;
        }
        __syncthreads();
        if (tid == 0) {                                                   // leaves among the elements taken from every list
            int k = 2 * n - 2;
            for (int merge = kTableBits - 1; merge > 0; --merge) {
                int lo = 0, hi = n;
                while (lo < hi) {
                    const int mid = (lo + hi) / 2;
                    if (place[merge][mid] < k) lo = mid + 1;
                    else hi = mid;
                }
                chosen[merge] = (uint32_t)lo;
                k = 2 * (k - lo);
            }
            chosen[0] = (uint32_t)k;
            sums[1] = 0;
        }
        __syncthreads();
        part = 0;
        for (int i = tid; i < n; i += kCodeThreads) {
            uint32_t bits = 0;
#pragma unroll
            for (int merge = 0; merge < kTableBits; ++merge) bits += rank_of[i] < chosen[merge] ? 1 : 0;
            lengths[0][i] = (uint8_t)bits;
            part += i < m ? counts[i] * bits : escapes * (bits + kEscSideBits);
        }
        atomicAdd(&sums[1], part);
        __syncthreads();
        const unsigned long long bits = sums[1];
        if (m == present) {                                               // the first cut-off, if any
            all_coded = m;
            free_bits = bits;
        }
        // an escape-free code stays unless a later one is cheaper by more than 1/32
        const bool taken = best == 0 || bits < best_bits;
        if (taken) best_bits = bits;
        if (best == 0 || (taken && !(all_coded && free_bits <= best_bits + (best_bits >> kEscFreeShift)))) {
            best = m;
            best_escapes = escapes;
            for (int i = tid; i < n; i += kCodeThreads) lengths[1][i] = lengths[0][i];
        }
    }
    // canonical codes: shorter first, of one length in the order of the ids, ESC last
    __syncthreads();
    const int n = best + 1;
    if (tid < kTableBits + 2) per_length[tid] = 0;
    __syncthreads();
    for (int i = tid; i < n; i += kCodeThreads) atomicAdd(&per_length[lengths[1][i]], 1u);
    __syncthreads();
    if (tid == 0) {
        uint32_t code = 0;
        for (int l = 1; l <= kTableBits; ++l) {
            code = (code + per_length[l - 1]) << 1;
            first_code[l] = code;
        }
    }
    __syncthreads();
    for (int i = tid; i < n; i += kCodeThreads) {
        const uint32_t l = lengths[1][i], id = i < best ? id_of[i] : kEscIndex;
        uint32_t before = 0;
        for (int j = 0; j < best; ++j) before += lengths[1][j] == l && id_of[j] < id ? 1 : 0;
        const uint32_t reversed = __brev(first_code[l] + before) >> (32 - l);
        enc[id] = reversed | l << 16;
        const uint32_t entry = l | (id == kEscIndex ? kEscFlag : (id & 0xFFu) << 7 | (id >> 8) << 23);
        for (uint32_t at = reversed; at < (uint32_t)kTableEntries; at += 1u << l) dec[at] = entry;
    }
    if (tid == 0) {
        info[0] = (long long)(all_coded && best == all_coded ? free_bits : best_bits);
        info[1] = lengths[1][best];
        info[2] = best_escapes > 0 ? 1 : 0;
    }
}

}  // namespace bhi

using namespace bhi;

extern "C" int bhi_pair_code(const void* counts, const void* ids, void* enc, void* dec, void* info, void* stream) {
    if (!counts || !ids || !enc || !dec || !info) return bhi_fail(BHI_EINVAL, "null pointer");
    hipLaunchKernelGGL(pair_code_kernel, dim3(1), dim3(kCodeThreads), 0, (hipStream_t)stream, (const unsigned long long*)counts,
                       (const long long*)ids, (uint32_t*)enc, (uint32_t*)dec, (long long*)info);
    return bhi_launch_status("pair_code");
}

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
