// One token's attention step of a decoder layer in one launch: per-head RMSNorm and rotary
// embedding of the projected q and k heads, the write of k and v into the cache at the token's
// position, and the attention of the one query per head over the cache slots up to that
// position (grouped-query: several q heads share a k/v head).
//
// No counterpart in the reference, which leaves the attention to the model code it is given
// (transformers' attention over torch kernels).  It is here because the recorded decode step
// spends its time between the linear layers otherwise: written with torch operations this
// part is 14 kernels per layer, about 5 us each inside a graph, beside 4 launches of this
// library.  The position is read from device memory, so a recorded graph follows it.
//
// Bound by latency at short contexts (a chain of launch, position, rows, hand-over) and by the
// cache rows (512 bytes per k/v head and slot) at long ones.  What follows from that:
//
//  * The slots are cut into splits of at least 64, one block of 256 threads per (split, k/v head,
//    up to 4 of its q heads): q heads of a group share the k and v rows a block reads, and the
//    splits cover the GPU (about 256 blocks at the longest context).  More q heads per block read
//    the rows fewer times but take longer over them and have more to hand over: with up to 16, 24
//    heads over 2 took 10.2 / 14.0 us at 33 / 301 slots (4: 6.6 / 9.2), 28 over 4 took 17.6 us at 6001
//    slots (4: 17.3); with 2, 1 us less up to 301 slots and 1-2 us more from 1000 on.  The cut follows the
//    position, which only the device knows: the grid is sized for the cache, and blocks beyond
//    the splits that the position needs leave at once.
//  * A wavefront owns a quarter of its block's slots and treats them without meeting the others:
//    scores by v_mfma_f32_16x16x32_bf16 (A: 16 k rows as they lie in memory, 16 bytes per lane;
//    B: the q heads from LDS), its own running maximum, weights through its own corner of LDS,
//    and the weighted sum of the v rows in registers (8 bytes of two rows per lane and load).
//    All rows of up to 64 slots are requested before any is used.
//  * The four wavefronts' sums meet in LDS; where there is more than one split, the blocks leave
//    their (maximum, sum, weighted sum) in a workspace and the last one to arrive at the counter
//    of its (k/v head, q heads) adds them and leaves the counter at zero.  The stores and loads
//    are agent-scope, the arrival is relaxed, and the last block executes one acquire: the scheme
//    of the K-sliced matrix product (bhi_mma.h), for the reasons and with the costs given there.
//
// Measured in a recorded graph, cache rows not in any cache, us (one block per q head walking all
// slots with dot products before -> now): 28 / 4 heads at 6001 slots 149 -> 15.9, 32 / 8 heads at 301
// slots 14.3 -> 7.5, at 1001 slots 8.8 now; 4.8 at one slot is what launch, position, rows and
// output take in a row, and a hand-over costs 2.5 more.  Splits of 32 or 128 slots at least, and at
// most 16 or 32 splits, were within 1 us of this or slower.  Without a workspace (one block per q
// head, the looping kernel): 154 -> 81 at 6001 slots of 28 / 4 heads, 30.2 -> 22.5 and 14.3 -> 12.5 at
// 1001 and 301 of 32 / 8, 5.5 -> 4.3 at one.
#include <type_traits>
#include "bhi_common.h"
#include "bhi_host.h"

namespace bhi {

constexpr int kAttnDim = 128;          // head dimension the kernel is written for
constexpr int kAttnThreads = 256;
constexpr int kAttnWaves = kAttnThreads / kLanes;
constexpr int kAttnMaxLen = 8192;
constexpr int kAttnTile = 16;          // slots of one matrix instruction
constexpr int kAttnBatch = 64;         // slots a wavefront has in flight at most
constexpr int kAttnMinSplit = 64;      // slots of the shortest split
constexpr int kAttnBlocks = 256;       // blocks wanted at the longest context
constexpr int kAttnMaxSplits = 64;     // what the last block has to add up (unless shares would get too long)
constexpr int kAttnAhead = 16;         // splits a thread of the last block has in flight
constexpr int kAttnHeads = 4;          // q heads of a block at most
constexpr int kAttnCounters = 1024;    // (k/v head, q heads) pairs a workspace has counters for

struct AttnArgs {
    const uint16_t* qk;        // bf16 [q_heads + kv_heads, 128]: the projections of the token
    const uint16_t* v;         // bf16 [kv_heads, 128]
    const uint16_t* norm_w;    // bf16 [q_heads + kv_heads, 128] RMSNorm weights per head, or null
    const float* cos;          // fp32 [max_len, 128]: cos(angle) for both halves
    const float* sin;          // fp32 [max_len, 128]: -sin for the first half, +sin for the second
    const long long* pos;      // the token's position (device memory)
    uint16_t* k_cache;         // bf16 [kv_heads, max_len, 128]
    uint16_t* v_cache;
    uint16_t* out;             // bf16 [q_heads, 128]
    int q_heads, kv_heads, max_len;
    float eps, scale;
    int heads;                 // q heads per block
    int tiles;                 // blocks per k/v head and split: ceil(q heads of the group / heads)
    int splits;                // splits the grid is sized for
    uint32_t* counters;        // [kv_heads * tiles], zero between launches (splits > 1)
    float* partial;            // [kv_heads * tiles][splits][GT][kAttnPartial]
};
constexpr int kAttnPartial = kAttnDim + 2;   // weighted sum, maximum, sum of weights

__device__ __forceinline__ float bf16_lo(uint32_t pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t pair) { return __uint_as_float(pair & 0xFFFF0000u); }

// Reductions without a trip through the LDS crossbar (six dependent __shfl_xor in a row are longer
// than the rest of a head's normalisation): the two row-swap instructions of gfx950.
typedef uint32_t swapped_t __attribute__((ext_vector_type(2)));
template <class Op>
__device__ __forceinline__ float across_halves(float v, Op op) {            // lanes l and l ^ 32
    const swapped_t p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(p.x), __uint_as_float(p.y));
}
template <class Op>
__device__ __forceinline__ float across_rows(float v, Op op) {              // the four rows of 16 lanes
    const swapped_t p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return across_halves(op(__uint_as_float(p.x), __uint_as_float(p.y)), op);
}
struct Add { __device__ __forceinline__ float operator()(float x, float y) const { return x + y; } };
struct Max { __device__ __forceinline__ float operator()(float x, float y) const { return fmaxf(x, y); } };

// One head by one wavefront: RMSNorm (fp32, weight applied after the normalisation) and
// rotation; lane l holds elements l and l + 64, the two halves the rotation pairs up.  Loads and
// arithmetic apart, so that several heads' loads are in flight together.
struct HeadRow {
    float a, b, wa, wb;
    __device__ __forceinline__ void load(const AttnArgs& g, int row, int lane) {
        const uint16_t* head = g.qk + (size_t)row * kAttnDim;
        a = __uint_as_float((uint32_t)head[lane] << 16);
        b = __uint_as_float((uint32_t)head[lane + 64] << 16);
        wa = wb = 1.0f;
        if (g.norm_w) {
            const uint16_t* w = g.norm_w + (size_t)row * kAttnDim;
            wa = __uint_as_float((uint32_t)w[lane] << 16);
            wb = __uint_as_float((uint32_t)w[lane + 64] << 16);
        }
    }
    // out = x * cos + swap_halves(x) * sin, sin carrying the sign; times `scale`, as BF16
    __device__ __forceinline__ void store(uint16_t* dst, float r, float c0, float c1, float s0, float s1, float scale, int lane) const {
        const float x = a * r * wa, y = b * r * wb;
        dst[lane] = f32_to_bf16_rne((x * c0 + y * s0) * scale);
        dst[lane + 64] = f32_to_bf16_rne((y * c1 + x * s1) * scale);
    }
};

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4a_t __attribute__((ext_vector_type(4)));
typedef unsigned long long u64_t;
// rows of v, of the new token and of the output: aligned as their element type, no more
typedef uint32_t row8_t __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t row16_t __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ uint2 load_row8(const uint16_t* p) {
    const row8_t v = *(const row8_t*)p;
    return make_uint2(v.x, v.y);
}
// four values, normalised and rounded
__device__ __forceinline__ void store_row8(uint16_t* p, const f32x4a_t& o, float inv) {
    *(row8_t*)p = row8_t{f32_to_bf16_rne(o[0] * inv) | (uint32_t)f32_to_bf16_rne(o[1] * inv) << 16,
                         f32_to_bf16_rne(o[2] * inv) | (uint32_t)f32_to_bf16_rne(o[3] * inv) << 16};
}

__device__ __forceinline__ void agent_store(float* p, float x, float y) {
    __hip_atomic_store((u64_t*)p, ((u64_t)__float_as_uint(y) << 32) | __float_as_uint(x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// partial sums: rows of 130 floats, 8-byte aligned
typedef float f32x4p_t __attribute__((ext_vector_type(4), aligned(8)));
typedef float f32x2p_t __attribute__((ext_vector_type(2), aligned(8)));
// exp(m - top) where both may be -inf (a wavefront or split without slots): then 0
__device__ __forceinline__ float rescale(float m, float top) { return m == -INFINITY ? 0.f : __expf(m - top); }

// GT: q heads a block is built for (1, 2 or 4): sums and weights are kept for that many.
// LOOP: a wavefront's share may be more slots than it has in flight at once.  Built for one q head
// only, for launches without a workspace: the loop keeps both ends of its registers alive (254 where
// 218 do; above 256 a compute unit would hold one block, not two), and with splits no share is that long.
template <int GT, bool LOOP>
__global__ __launch_bounds__(kAttnThreads, 2) void decode_attention_kernel(const AttnArgs a) {
    constexpr int kRow = kAttnDim + 8;                           // q rows 16 bytes apart in bank order
    __shared__ __align__(16) uint16_t q[kAttnTile][kRow];
    __shared__ __align__(16) uint16_t k_new[kAttnDim];
    __shared__ __align__(16) float weights[kAttnWaves][kAttnBatch][GT];
    __shared__ __align__(16) float factor[kAttnWaves][GT];    // rescaling of earlier slots
    __shared__ __align__(16) float own_weight[GT];
    __shared__ __align__(16) float part[kAttnWaves][GT][kAttnDim];
    __shared__ float tops[kAttnWaves][GT], sums[kAttnWaves][GT];
    __shared__ uint32_t is_last;

    const int tid = threadIdx.x, lane = tid & (kLanes - 1), wave = (int)uniform(tid >> 6);
    const int split = blockIdx.x, kh = (int)blockIdx.y / a.tiles, tile = (int)blockIdx.y % a.tiles;
    const int group = a.q_heads / a.kv_heads;
    const int h0 = kh * group + tile * a.heads;                  // first q head of this block
    const int nh = min(a.heads, group - tile * a.heads);         // and how many it has
    // what does not depend on the position travels with it
    constexpr int kHeadsPerWave = (GT + kAttnWaves - 1) / kAttnWaves;
    HeadRow qh[kHeadsPerWave];
#pragma unroll
    for (int i = 0; i < kHeadsPerWave; ++i) {
        const int h = wave + i * kAttnWaves;
        if (h < nh) qh[i].load(a, h0 + h, lane);
    }
    HeadRow kn;
    if (wave == kAttnWaves - 1) kn.load(a, a.q_heads + kh, lane);

    long long p = *a.pos;
    p = p < 0 ? 0 : (p >= a.max_len ? a.max_len - 1 : p);
    const int n = (int)p + 1;                                    // visible slots: 0 .. pos
    // splits in use: as many as there are, each a multiple of 64 slots
    const int per_split = ((n + a.splits - 1) / a.splits + kAttnMinSplit - 1) / kAttnMinSplit * kAttnMinSplit;
    const int used = (n + per_split - 1) / per_split;
    if (split >= used) return;
    const int first = split * per_split;
    const bool newest = split == used - 1;                       // this block's slots include the token's own
    const int slots = newest ? n - first : per_split;
    // a wavefront's slots: a quarter of the block's, in whole matrix tiles
    const int share = ((slots + kAttnWaves - 1) / kAttnWaves + kAttnTile - 1) / kAttnTile * kAttnTile;
    const int w0 = first + wave * share, w1 = min(w0 + share, first + slots);
    const bool has_own = newest && w0 < w1 && w1 == n;           // the token's own slot is this wavefront's

    const uint16_t* v_own = a.v + (size_t)kh * kAttnDim;
    // With nothing cached yet (n == 1) the token's own v row stands in for both: the only slot of
    // the cache is then one that was never written and that another block may be writing.
    const uint16_t* kc = n > 1 ? a.k_cache + (size_t)kh * a.max_len * kAttnDim : v_own;
    const uint16_t* vc = n > 1 ? a.v_cache + (size_t)kh * a.max_len * kAttnDim : v_own;
    const int cached = min(w1, n - 1);                           // end of this wavefront's slots whose rows are in the cache
    const int col = lane & 15, quarter = lane >> 4, half = lane >> 5;

    // this position's cosines and sines ahead of the rows: vector loads return in issue order
    const float *cs = a.cos + (size_t)p * kAttnDim, *sn = a.sin + (size_t)p * kAttnDim;
    const float c0 = cs[lane], c1 = cs[lane + 64], s0 = sn[lane], s1 = sn[lane + 64];

    float top = -INFINITY, sum = 0.f;                            // of q head `col`; `sum` over this lane's slots only
    f32x4a_t acc[GT];                                            // elements 4 * (lane & 31) .. + 3 over this half's slots
#pragma unroll
    for (int h = 0; h < GT; ++h) acc[h] = f32x4a_t{0.f, 0.f, 0.f, 0.f};

    constexpr int kMaxTiles = kAttnBatch / kAttnTile;
    // The walk over a wavefront's slots, NT tiles of 16 at a time.  NT is what a block's shares need
    // (at most four; three as four read a third more rows: at 6001 slots of 28 / 4 heads the layer's step took
    // 104.1 us, 102.7 so), as a constant: every load is then unconditional, and the wait for the q/k work
    // does not become a wait for the rows behind it.
    auto walk = [&](auto tiles_c) __attribute__((always_inline)) {
        constexpr int NT = decltype(tiles_c)::value;
        uint4 kr[NT][4];                                         // [tile][32 of the 128 elements]
        uint2 vr[NT][8];                                         // [tile][two slots]: 4 elements of one of them
        const int last = n > 1 ? n - 2 : 0;
        auto load = [&](int b0) __attribute__((always_inline)) {
            // slots past the visible ones read a valid row, whose score and values are dropped below
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                int j = b0 + t * kAttnTile + col;
                j = j < last ? j : last;
                // 32-bit offsets from a uniform base: a head of the cache is at most 2 MiB
                const char* row = (const char*)kc + (uint32_t)(j * (2 * kAttnDim) + quarter * 16);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const row16_t r = *(const row16_t*)(row + 64 * c);
                    kr[t][c] = make_uint4(r.x, r.y, r.z, r.w);
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    int j = b0 + t * kAttnTile + 2 * i + half;
                    j = j < last ? j : last;
                    vr[t][i] = load_row8((const uint16_t*)((const char*)vc + (uint32_t)(j * (2 * kAttnDim) + 8 * (lane & 31))));
                }
            }
        };
        const uint2 vo = load_row8(v_own + 4 * (lane & 31));
        load(w0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kHeadsPerWave; ++i) {
            const int h = wave + i * kAttnWaves;
            if (h < nh) {
                const float r = rsqrtf(wave_sum(qh[i].a * qh[i].a + qh[i].b * qh[i].b) * (1.0f / kAttnDim) + a.eps);
                qh[i].store(q[h], r, c0, c1, s0, s1, a.scale, lane);
            }
        }
        for (int h = nh + wave; h < kAttnTile; h += kAttnWaves) q[h][lane] = q[h][lane + 64] = 0;
        if (newest && wave == kAttnWaves - 1) {
            const float r = rsqrtf(wave_sum(kn.a * kn.a + kn.b * kn.b) * (1.0f / kAttnDim) + a.eps);
            kn.store(k_new, r, c0, c1, s0, s1, 1.0f, lane);
        }
        lds_barrier();
        bf16x8_t qf[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) qf[c] = *(const bf16x8_t*)&q[col][32 * c + 8 * quarter];

        int b0 = w0;
        for (;;) {
            f32x4a_t s[NT];
            float best = -INFINITY;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                f32x4a_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    uint4 k = kr[t][c];
                    if (newest && b0 + t * kAttnTile + col == n - 1) k = *(const uint4*)&k_new[32 * c + 8 * quarter];
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, k), qf[c], d, 0, 0, 0);
                }
                // lane: q head `col`, slots 4 * quarter .. + 3 of the tile
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[t][i] = b0 + t * kAttnTile + 4 * quarter + i < w1 ? d[i] : -INFINITY;
                    best = fmaxf(best, s[t][i]);
                }
            }
            best = across_rows(best, Max{});
            const float new_top = fmaxf(top, best);
            const float scale_old = rescale(top, new_top);
            top = new_top;
            sum *= scale_old;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float w = rescale(s[t][i], new_top);
                    sum += w;
                    // the token's own v is not in the cache yet: its weight goes aside
                    const int j = t * kAttnTile + 4 * quarter + i;
                    const bool own = has_own && b0 + j == n - 1;
                    if (col < GT) {
                        weights[wave][j][col] = own ? 0.f : w;
                        if (own) own_weight[col] = w;
                    }
                }
            }
            // Rows that are not this wavefront's are dropped by value: a weight of 0 would make NaN of an Inf
            // or NaN in them.  In the loop once, at the end of the walk (at 6001 slots 85.5 us with the
            // selects in every batch, 80.6 so); without a loop where they are used (0.2 us of 15.9; a branch
            // around them 0.1 more).
            if (LOOP && b0 + NT * kAttnTile > cached) {
#pragma unroll
                for (int t = 0; t < NT; ++t) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        if (b0 + t * kAttnTile + 2 * i + half >= cached) vr[t][i] = make_uint2(0, 0);
                    }
                }
            }
            if (LOOP && b0 != w0) {                              // earlier slots were weighted against an older maximum
                if (lane < GT) factor[wave][lane] = scale_old;
#pragma unroll
                for (int h = 0; h < GT; ++h) acc[h] *= factor[wave][h];
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float* w = weights[wave][t * kAttnTile + 2 * i + half];
                    const bool in = LOOP || b0 + t * kAttnTile + 2 * i + half < cached;
                    const uint32_t lo = in ? vr[t][i].x : 0u, hi = in ? vr[t][i].y : 0u;
                    const f32x4a_t v = {bf16_lo(lo), bf16_hi(lo), bf16_lo(hi), bf16_hi(hi)};
#pragma unroll
                    for (int h = 0; h < GT; ++h) acc[h] += w[h] * v;
                }
                __builtin_amdgcn_sched_barrier(0);               // one tile's weights in registers at a time
            }
            b0 += NT * kAttnTile;
            if (!LOOP || NT < kMaxTiles || b0 >= w1) {
                if (has_own && half == 0) {
                    const f32x4a_t v = {bf16_lo(vo.x), bf16_hi(vo.x), bf16_lo(vo.y), bf16_hi(vo.y)};
#pragma unroll
                    for (int h = 0; h < GT; ++h) acc[h] += own_weight[h] * v;
                }
                break;
            }
            load(b0);
        }
    };
    if (share == kAttnTile) walk(std::integral_constant<int, 1>{});
    else if (share == 2 * kAttnTile) walk(std::integral_constant<int, 2>{});
    else if (!LOOP && share == 3 * kAttnTile) walk(std::integral_constant<int, 3>{});
    else walk(std::integral_constant<int, kMaxTiles>{});
    if (newest && tile == 0 && tid < 32) {                       // the token's k and v enter the cache
        const uint16_t* src = (tid < 16 ? k_new : v_own) + 8 * (tid & 15);
        uint16_t* dst = (tid < 16 ? a.k_cache : a.v_cache) + ((size_t)kh * a.max_len + p) * kAttnDim + 8 * (tid & 15);
        *(row16_t*)dst = *(const row16_t*)src;
    }
    sum = across_rows(sum, Add{});
#pragma unroll
    for (int h = 0; h < GT; ++h) {
        f32x4a_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = across_halves(acc[h][e], Add{});
        if (lane < 32) *(f32x4a_t*)&part[wave][h][4 * lane] = o;
    }
    if (lane < GT) {
        tops[wave][lane] = top;
        sums[wave][lane] = sum;
    }
    __syncthreads();

    // the block's sums: thread (head, 4 elements)
    float* mine = a.partial + ((size_t)blockIdx.y * a.splits + split) * GT * kAttnPartial;
    for (int e = tid; e < nh * 32; e += kAttnThreads) {
        const int h = e >> 5, d = 4 * (e & 31);
        const float m = fmaxf(fmaxf(tops[0][h], tops[1][h]), fmaxf(tops[2][h], tops[3][h]));
        float l = 0.f;
        f32x4a_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kAttnWaves; ++w) {
            const float f = rescale(tops[w][h], m);
            l += f * sums[w][h];
            o += f * *(const f32x4a_t*)&part[w][h][d];
        }
        if (used == 1) {
            store_row8(a.out + (size_t)(h0 + h) * kAttnDim + d, o, 1.0f / l);
        } else {
            float* dst = mine + h * kAttnPartial;
            agent_store(dst + d, o[0], o[1]);
            agent_store(dst + d + 2, o[2], o[3]);
            if (d == 0) agent_store(dst + kAttnDim, m, l);
        }
    }
    if (used == 1) return;

    __builtin_amdgcn_s_waitcnt(0x0F70);                          // vmcnt(0): the stores above have completed
    __syncthreads();
    if (tid == 0) {
        const uint32_t old = __hip_atomic_fetch_add(a.counters + blockIdx.y, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        is_last = old == (uint32_t)used - 1;
        if (is_last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    if (!is_last) return;
    // Ordinary loads: the acquire above has dropped whatever older lines of the workspace this die
    // held.  One round trip where the splits fit, and short code: it runs once, on a unit that has
    // not run it lately, and its instructions have to be fetched too (with the splits' factors
    // worked out first, through LDS, and 24 splits unrolled behind guards, 5 splits of 4 heads took
    // 1.1 us longer to meet).
    const float* all = a.partial + (size_t)blockIdx.y * a.splits * GT * kAttnPartial;
#pragma unroll 1
    for (int e = tid; e < nh * 32; e += kAttnThreads) {
        const int h = e >> 5, d = 4 * (e & 31);
        const float* src = all + (size_t)h * kAttnPartial;
        float m = -INFINITY, l = 0.f;
        f32x4a_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int s0 = 0; s0 < used; s0 += kAttnAhead) {
            f32x4a_t x[kAttnAhead];
            f32x2p_t ml[kAttnAhead];
            float best = m;
#pragma unroll
            for (int i = 0; i < kAttnAhead; ++i) {
                const float* q_ = src + (size_t)min(s0 + i, used - 1) * GT * kAttnPartial;
                ml[i] = *(const f32x2p_t*)(q_ + kAttnDim);
                x[i] = *(const f32x4p_t*)(q_ + d);
            }
#pragma unroll
            for (int i = 0; i < kAttnAhead; ++i) best = fmaxf(best, ml[i].x);
            const float f = rescale(m, best);
            m = best;
            l *= f;
            o *= f;
#pragma unroll
            for (int i = 0; i < kAttnAhead; ++i) {
                if (s0 + i < used) {                             // else the last split once more
                    const float w = rescale(ml[i].x, m);
                    l += w * ml[i].y;
                    o += w * x[i];
                }
            }
        }
        store_row8(a.out + (size_t)(h0 + h) * kAttnDim + d, o, 1.0f / l);
    }
    if (tid == 0) __hip_atomic_store(a.counters + blockIdx.y, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// How a step is cut.  `heads` q heads per block: the whole group where 4 hold it, else equal
// tiles.  Splits: as many as bring the grid to about a block per compute unit at the longest
// context, none shorter than 64 slots, and as many as it takes for a wavefront to hold its share
// in registers.  Without a workspace there is one split, and one q head per block keeps as many
// blocks as possible.
struct AttnPlan { int heads, tiles, splits, built; };      // built: the kernel's GT, 0 for the looping one

inline AttnPlan attn_plan(int q_heads, int kv_heads, int max_len, bool workspace) {
    const int group = q_heads / kv_heads;
    AttnPlan p = {1, group, 1, 0};
    const int tiles = (group + kAttnHeads - 1) / kAttnHeads;
    if (workspace && kv_heads * tiles <= kAttnCounters) {
        p.heads = (group + tiles - 1) / tiles;
        p.tiles = (group + p.heads - 1) / p.heads;
        p.built = 1;
        while (p.built < p.heads) p.built *= 2;
        const int per_block = kAttnWaves * kAttnBatch;
        const int least = (max_len + per_block - 1) / per_block, longest = (max_len + kAttnMinSplit - 1) / kAttnMinSplit;
        p.splits = kAttnBlocks / (kv_heads * p.tiles);
        p.splits = p.splits < kAttnMaxSplits ? p.splits : kAttnMaxSplits;
        p.splits = p.splits < longest ? p.splits : longest;
        p.splits = p.splits > least ? p.splits : least;
    }
    return p;
}

inline int64_t attn_workspace(const AttnPlan& p, int kv_heads) {
    return p.splits > 1 ? (int64_t)kAttnCounters * 4 + (int64_t)kv_heads * p.tiles * p.splits * p.built * kAttnPartial * 4 : 0;
}

}  // namespace bhi

static int check_attention(int q_heads, int kv_heads, int head_dim, int max_len) {
    using namespace bhi;
    if (head_dim != kAttnDim) return bhi_fail(BHI_EINVAL, "decode_attention is written for a head dimension of 128");
    if (q_heads < 1 || kv_heads < 1 || q_heads % kv_heads != 0) return bhi_fail(BHI_EINVAL, "q_heads must be a multiple of kv_heads");
    if (max_len < 1 || max_len > kAttnMaxLen) return bhi_fail(BHI_EINVAL, "decode_attention takes a cache of 1 to 8192 slots");
    return 0;
}

extern "C" int64_t bhi_decode_attention_workspace_bytes(int q_heads, int kv_heads, int head_dim, int max_len) {
    using namespace bhi;
    if (int rc = check_attention(q_heads, kv_heads, head_dim, max_len)) return rc;
    return attn_workspace(attn_plan(q_heads, kv_heads, max_len, true), kv_heads);
}

extern "C" int bhi_decode_attention_split(const void* qk, const void* v, const void* norm_weight, const void* cos, const void* sin,
                                          const void* pos, void* k_cache, void* v_cache, void* out, int q_heads, int kv_heads,
                                          int head_dim, int max_len, float eps, float scale, void* workspace,
                                          int64_t workspace_bytes, void* stream) {
    using namespace bhi;
    if (!qk || !v || !cos || !sin || !pos || !k_cache || !v_cache || !out) return bhi_fail(BHI_EINVAL, "null pointer");
    if (int rc = check_attention(q_heads, kv_heads, head_dim, max_len)) return rc;
    const AttnPlan plan = attn_plan(q_heads, kv_heads, max_len, workspace != nullptr);
    if (workspace && (workspace_bytes < attn_workspace(plan, kv_heads) || ((uintptr_t)workspace & 15)))
        return bhi_fail(BHI_EINVAL, "workspace too small: see bhi_decode_attention_workspace_bytes");
    AttnArgs a;
    a.qk = (const uint16_t*)qk; a.v = (const uint16_t*)v; a.norm_w = (const uint16_t*)norm_weight;
    a.cos = (const float*)cos; a.sin = (const float*)sin; a.pos = (const long long*)pos;
    a.k_cache = (uint16_t*)k_cache; a.v_cache = (uint16_t*)v_cache; a.out = (uint16_t*)out;
    a.q_heads = q_heads; a.kv_heads = kv_heads; a.max_len = max_len; a.eps = eps; a.scale = scale;
    a.heads = plan.heads; a.tiles = plan.tiles; a.splits = plan.splits;
    a.counters = (uint32_t*)workspace;
    a.partial = workspace ? (float*)((char*)workspace + kAttnCounters * 4) : nullptr;
    const dim3 grid((unsigned)plan.splits, (unsigned)(kv_heads * plan.tiles)), block(kAttnThreads);
    const hipStream_t st = (hipStream_t)stream;
    switch (plan.built) {
        case 1: hipLaunchKernelGGL((decode_attention_kernel<1, false>), grid, block, 0, st, a); break;
        case 2: hipLaunchKernelGGL((decode_attention_kernel<2, false>), grid, block, 0, st, a); break;
        case 4: hipLaunchKernelGGL((decode_attention_kernel<4, false>), grid, block, 0, st, a); break;
        default: hipLaunchKernelGGL((decode_attention_kernel<1, true>), grid, block, 0, st, a); break;
    }
    return bhi_launch_status("decode_attention");
}

extern "C" int bhi_decode_attention(const void* qk, const void* v, const void* norm_weight, const void* cos, const void* sin,
                                    const void* pos, void* k_cache, void* v_cache, void* out, int q_heads, int kv_heads,
                                    int head_dim, int max_len, float eps, float scale, void* stream) {
    return bhi_decode_attention_split(qk, v, norm_weight, cos, sin, pos, k_cache, v_cache, out, q_heads, kv_heads, head_dim,
                                      max_len, eps, scale, nullptr, 0, stream);
}
