// Fused decode + matrix product for 17 to 640 rows of X: the weights of a step meet in LDS as matrix operands,
// every wavefront multiplies all of them with its own part of X.
//
// What bounds the range.  tile_kernel keeps a wavefront's decoded weights in its registers, so every wavefront
// reads all of X from LDS for sixteen weight rows; from 65 rows those reads and the table lookups take most of a
// step (77 rows of 4096x12288: 2800 of 3900 clocks, counted from the instructions), and its windows of X end at 128 rows.  Decoding to
// BF16 and a library GEMM moves the weight through memory twice (12288x4096: 32 us to write it, 37-47 us to
// read and multiply it at 144 to 512 rows).
//
// Split.  A block owns 64 weight rows.  Eight wavefronts decode two row groups each and store their 128 columns
// as matrix operands (16 KB a step, double buffered, one barrier a step that orders LDS only).  Each wavefront
// holds the tiles of X that only it multiplies (SPLIT 1: with all 64 rows; SPLIT 2: with 32 of them, which halves the
// LDS reads of weights and doubles the loads of X: up to 9 tiles, rANS 12) in registers, a whole step ahead.  X is
// put into operand order by a launch of its own, because sixteen neighbouring lanes of an operand are sixteen
// rows of X: read in place a load took 64 clocks instead of 16 (300 rows of 11008x4096 100 us instead of 76).
// Step t - 1 is multiplied while step t is decoded: the products of a chunk stand behind the lookups of a
// round, between scheduling fences, since the compiler otherwise runs the streams one after the other (rANS
// 91 us instead of 70 with four wavefronts).  Two wavefronts per SIMD with two streams each, rather than one with
// four: 58.4 -> 51.6 us at 300 rows of 11008x4096.
//
// Measured on MI355X in recorded graphs (four to twelve copies of a weight in turn, us, before / now; before:
// tile_kernel up to 128 rows where its rule takes it, decoding and library GEMM else):
//
//   M x K               33 rows      64 rows      96 rows      128 rows     192 rows     300 rows     512 rows
//   4096x4096   Huff    18.6 / 18.1  20.4 / 18.3  24.9 / 21.6  28.9 / 22.7  40.1 / 28.1  35.8 / 33.4  41.7 / 45.0
//   12288x4096  Huff    32.1 / 33.9  35.8 / 35.5  42.9 / 36.9  47.9 / 39.7  70.9 / 45.8  77.6 / 51.7  86.0 / 70.7
//   12288x4096  rANS    41.0 / 42.7  43.6 / 43.7  54.7 / 44.3  56.9 / 45.4  72.5 / 50.2  80.8 / 58.5  90.5 / 76.7
//   4096x12288  Huff    36.3 / 33.4  40.9 / 35.1  49.5 / 38.2  58.0 / 41.5   103 / 51.7  92.4 / 61.1   111 / 84.5
//   18944x3584  Huff    41.9 / 52.4  45.6 / 54.9  61.6 / 56.6  66.3 / 63.1  79.4 / 73.5  95.4 / 87.0   110 / 118
//   3584x18944  Huff    54.3 / 40.7  60.9 / 43.4  65.6 / 47.9  69.1 / 51.6   130 / 61.7   138 / 77.9   213 / 101
//   8192x8192   rANS    65.7 / 44.6  69.4 / 46.5  71.0 / 49.8  73.2 / 51.5  96.5 / 58.6   103 / 74.8   117 / 100
//
// (functional.prefers_wide picks the sides.)  What bounds it now, by counters (share of the time that a compute unit
// with a block has the LDS pipe / matrix cores / VALU / address unit of its vector memory busy): 77 rows of 4096x12288
// 44 / 12 / 22 / 54 %, and wavefronts wait half of their time for memory or LDS: nothing is full, a step is as long
// as its chain of lookups between two barriers at two wavefronts per SIMD; 300 rows of 11008x4096 rANS
// 58 / 35 / 43 / 61 %; 640 rows of 12288x4096 36 / 53 / 25 / 81 %: the loads of X, which every block reads whole
// (0.041 us per tile and step, 41 bytes a clock and unit; 0.057 us while a tile of X was one piece of memory, whose
// chunks all fell on the same channels of the cache: 92 us instead of 84).  Beside that the units without a block:
// 11008 rows are 172 blocks for 256 units, 18944 are 296.
#pragma once
// (included by bhi_task.h users after bhi_tile.h, whose argument block and workspace rules it shares)

namespace bhi {

constexpr int kWideWaves = 8;
constexpr int kWideGroups = 2;                               // row groups a wavefront decodes side by side
constexpr int kWideQuads = kWideWaves * kWideGroups * kGroupRows / 16;      // sixteen weight rows each
constexpr int kWideRows = kWideQuads * 16;                   // weight rows of a block
constexpr int kWideChunks = 4;                               // 32 columns of a step: what one matrix instruction takes
constexpr int kWideMaxTiles = 5;                             // tiles of X per wavefront
constexpr int kWideThreads = kWideWaves * kLanes;
constexpr int kWideUnits = 256;                              // compute units
constexpr int kWideMaxSlices = 8;
constexpr int kWideCounterBytes = 1024;                      // sliced launches have at most 256 blocks
constexpr int kWideMinBatch = 17, kWideMaxBatch = kWideMaxTiles * kWideWaves * kTileBatch;

// The streams of two row groups decoded side by side: every round looks up one table entry (Huffman: a pair, rANS: a
// symbol) of each, and `between(round, rounds)` runs while the lookups of a round are in flight.
template <bool HAS_ESC, class Between>
__device__ __forceinline__ void decode_wide(HuffCursor (&cur)[kWideGroups], const uint32_t* __restrict__ table,
                                            const uint32_t (&lo)[kWideGroups], const uint32_t (&hi)[kWideGroups],
                                            const uint32_t (&nx)[kWideGroups], uint32_t (&e)[kWideGroups][4], Between between) {
    constexpr int N = kWideGroups;
    typedef std::integral_constant<int, 4> rounds;
    const char* tb = (const char*)table;
    uint32_t w[N], t01[N];
#pragma unroll
    for (int g = 0; g < N; ++g) {
        w[g] = __builtin_amdgcn_alignbit(hi[g], lo[g], cur[g].pos & 31u);
        e[g][0] = table_entry(tb, w[g]);
    }
    between(std::integral_constant<int, 0>{}, rounds{});
#pragma unroll
    for (int g = 0; g < N; ++g) e[g][1] = table_entry(tb, w[g] >> (e[g][0] & 31u));
    between(std::integral_constant<int, 1>{}, rounds{});
#pragma unroll
    for (int g = 0; g < N; ++g) {
        const uint32_t whi = __builtin_amdgcn_alignbit(nx[g], hi[g], cur[g].pos & 31u);
        t01[g] = e[g][0] + e[g][1];
        w[g] = __builtin_amdgcn_alignbit(whi, w[g], t01[g]);
        e[g][2] = table_entry(tb, w[g]);
    }
    between(std::integral_constant<int, 2>{}, rounds{});
#pragma unroll
    for (int g = 0; g < N; ++g) e[g][3] = table_entry(tb, w[g] >> (e[g][2] & 31u));
    between(std::integral_constant<int, 3>{}, rounds{});
    uint32_t any = 0;
#pragma unroll
    for (int g = 0; g < N; ++g) {
        cur[g].pos += (t01[g] + e[g][2] + e[g][3]) & 0x3Fu;
        if (HAS_ESC) any |= e[g][0] | e[g][1] | e[g][2] | e[g][3];
    }
    if (HAS_ESC && __builtin_expect(ballot((int32_t)any < 0) != 0, 0)) {
#pragma unroll
        for (int g = 0; g < N; ++g) cur[g].escapes(e[g]);
    }
}

template <bool UNUSED, class Between>
__device__ __forceinline__ void decode_wide(AnsCursor (&cur)[kWideGroups], const uint32_t* __restrict__ table,
                                            const uint32_t (&lo)[kWideGroups], const uint32_t (&hi)[kWideGroups],
                                            const uint32_t (&)[kWideGroups], uint32_t (&e)[kWideGroups][4], Between between) {
    constexpr int N = kWideGroups;
    typedef std::integral_constant<int, 8> rounds;
    uint2 a[N], b[N];
    bool first[N];
    auto pair = [&](auto pair_c) __attribute__((always_inline)) {
        constexpr int d = decltype(pair_c)::value;
#pragma unroll
        for (int g = 0; g < N; ++g) a[g] = AnsCursor::look(table, cur[g].xl);
        between(std::integral_constant<int, 2 * d>{}, rounds{});
#pragma unroll
        for (int g = 0; g < N; ++g) {
            AnsCursor::advance(a[g], cur[g].xl, cur[g].xh);
            b[g] = AnsCursor::look(table, cur[g].xl);
        }
        between(std::integral_constant<int, 2 * d + 1>{}, rounds{});
#pragma unroll
        for (int g = 0; g < N; ++g) {
            AnsCursor::advance(b[g], cur[g].xl, cur[g].xh);
            e[g][d] = __builtin_amdgcn_perm(b[g].y, a[g].y, 0x07060302u);
            if (d == 1) {
                first[g] = cur[g].xh == 0u;
                cur[g].refill(lo[g]);
            }
            if (d == 3) cur[g].refill(first[g] ? hi[g] : lo[g]);
        }
    };
    pair(std::integral_constant<int, 0>{});
    pair(std::integral_constant<int, 1>{});
    pair(std::integral_constant<int, 2>{});
    pair(std::integral_constant<int, 3>{});
}

// X in the order the matrix instructions take it: 1 KB per tile of sixteen rows and chunk of 32 columns, the tiles of
// a chunk side by side.  Under a trace, which adds 1 to 2 us, 2.3 us for 40 rows of 4096 columns, 3.2 for 77 of 12288,
// 5.4 for 300 of 4096 and 6.3 for 640: its launch and one round trip, and a tenth of the call.  Rows past the batch repeat its last row.
static __global__ __launch_bounds__(256) void pack_x_kernel(const uint16_t* __restrict__ X, u32x4v_t* __restrict__ out, int rows, int K, int tiles) {
    const int piece = (int)(blockIdx.x * 4 + threadIdx.x / kLanes), lane = threadIdx.x & (kLanes - 1);
    const int tile = piece % tiles, chunk = piece / tiles;
    if (chunk >= K / 32) return;
    const int r = tile * kTileBatch + (lane & 15);
    out[(size_t)piece * kLanes + lane] = *(const u32x4v_t*)(X + (size_t)(r < rows ? r : rows - 1) * K + chunk * 32 + 8 * (lane >> 4));
}

struct WideArgs {
    MmaArgs a;
    int tiles;               // of sixteen rows of X
};

template <class Codec, int NT, int SPLIT>
__global__ __launch_bounds__(kWideThreads, 2)
void wide_kernel(const uint16_t* __restrict__ X, const WideArgs wa) {
    const MmaArgs& a = wa.a;
    constexpr int kParts = kWideWaves / SPLIT, kQuads = kWideQuads / SPLIT;      // of X, and the quads of a wavefront
    constexpr int kBuffer = kWideQuads * kWideChunks * kLanes;                  // 16-byte pieces of a step's weights
    __shared__ uint32_t rings[kWideWaves * kWideGroups][kRingWords];
    __shared__ uint32_t lut[Codec::Table::kLdsWords];
    __shared__ u32x4v_t wt[2][kBuffer];

    const Shape s = a.s;
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = (int)uniform(threadIdx.x / kLanes);
    const int rb = (int)blockIdx.x / a.slices, ks = (int)blockIdx.x % a.slices;
    const int g0 = (rb * kWideWaves + wave) * kWideGroups;
    const int tpk = s.split_k * s.nc / a.slices;
    const int kc0 = ks * tpk, kc1 = kc0 + tpk;
    const int K = s.Ks * s.split_k;
    const bool variant = Codec::variant(a.header);
    const int B = a.batch;
    // this wavefront's quads quad0, ... and tiles of X tile0, tile0 + kParts, ...
    const int quad0 = wave / kParts * kQuads, tile0 = wave % kParts;
    const bool all_tiles = tile0 + (NT - 1) * kParts < wa.tiles;

    f32x4_t acc[kQuads][NT];
#pragma unroll
    for (int w = 0; w < kQuads; ++w) {
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[w][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    // buffer loads: place of tile and chunk as a scalar offset
    const uint32_t chunk_bytes = (uint32_t)wa.tiles * 1024u;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)X, 0, (int)(chunk_bytes * (uint32_t)(K / 32)), 0x00020000);
    uint32_t x_tile[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) x_tile[n] = (uint32_t)min(tile0 + n * kParts, wa.tiles - 1) * 1024u;

    // lane 4 b + i of a group's stream holds row i and columns 8 b .. 8 b + 7; the operand of a chunk of 32 columns wants
    // row r of sixteen and columns 8 q .. in lane 16 q + r.  Rows of odd q are stored four places on, so that eight
    // neighbouring lanes write to different banks.
    const int b = lane >> 2, q_of = b & 3;
    u32x4v_t* put[kWideGroups];
#pragma unroll
    for (int g = 0; g < kWideGroups; ++g) {
        const int row = (wave * kWideGroups + g) * kGroupRows + (lane & 3);
        put[g] = &wt[0][((row >> 4) * kWideChunks + (b >> 2)) * kLanes + 16 * q_of + ((row & 15) ^ (4 * (q_of & 1)))];
    }
    const u32x4v_t* const get = &wt[0][quad0 * kWideChunks * kLanes + (lane & 48) + ((lane & 15) ^ (4 * ((lane >> 4) & 1)))];

    typename Codec::Cursor cur[kWideGroups];
    auto run = [&](auto has_esc, auto tiles_c) __attribute__((always_inline)) {
        constexpr bool HAS_ESC = decltype(has_esc)::value;
        constexpr int N = decltype(tiles_c)::value;
        u32x4v_t xf[kWideChunks][N > 0 ? N : 1];
#pragma unroll
        for (int c = 0; c < kWideChunks; ++c) {
#pragma unroll
            for (int n = 0; n < N; ++n) xf[c][n] = u32x4v_t{0, 0, 0, 0};
        }
        auto x_load = [&](uint32_t x0, int c) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < N; ++n)
                xf[c][n] = __builtin_amdgcn_raw_buffer_load_b128(xr, lane * 16, (int)(x_tile[n] + x0 + (uint32_t)c * chunk_bytes), 0);
        };
        auto fetch = [&](u32x4v_t (&f)[kQuads], int from, int c) __attribute__((always_inline)) {
#pragma unroll
            for (int w = 0; w < kQuads; ++w) f[w] = get[from * kBuffer + (w * kWideChunks + c) * kLanes];
        };
        // the products of one step's chunk c with quads w0 .. w1
        auto multiply = [&](const u32x4v_t (&f)[kQuads], int c, int w0, int w1) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < N; ++n) {
#pragma unroll
                for (int w = w0; w < w1; ++w)
                    acc[w][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, f[w]),
                                                                       __builtin_bit_cast(bf16x8_t, xf[c][n]), acc[w][n], 0, 0, 0);
            }
        };
        int par = 0;
        for (int kc = kc0; kc < kc1; ++kc) {
            const TaskId id = task_of(s, kc);
            const int ns = id.t1 - id.t0;
            const uint2* rem0[kWideGroups];
#pragma unroll
            for (int g = 0; g < kWideGroups; ++g) {
                const TaskSpan span = task_span(a.offsets, s.M, s.split_k, s.nc, id.k, g0 + g, id.c, s.total_words);
                cur[g].open(a.exp, span, lane, rings[wave * kWideGroups + g]);
                rem0[g] = (const uint2*)(a.rem + ((size_t)id.k * s.M + (size_t)kGroupRows * (g0 + g)) * s.Ks + (size_t)id.t0 * kLanes * 8) + lane;
            }
            uint2 rem[kTileSteps][kWideGroups];
            auto rem_load = [&](uint2 (&dst)[kWideGroups], int t) __attribute__((always_inline)) {
                t = t < ns ? t : ns - 1;
#pragma unroll
                for (int g = 0; g < kWideGroups; ++g) dst[g] = stream_load(rem0[g] + (size_t)t * kLanes);
            };
            uint32_t first[kWideGroups][kPrimeRows];
#pragma unroll
            for (int g = 0; g < kWideGroups; ++g) cur[g].prime_issue(first[g]);
#pragma unroll
            for (int i = 0; i < kTileSteps; ++i) rem_load(rem[i], i);
            if (kc == kc0) {
                Codec::Table::fill(lut, a.table);
                // the first step is decoded while a step of zeros is multiplied
#pragma unroll
                for (int j = 0; j < kBuffer; j += kWideThreads) wt[1][j + (int)threadIdx.x] = u32x4v_t{0, 0, 0, 0};
                lds_barrier();
            }
#pragma unroll
            for (int g = 0; g < kWideGroups; ++g) {
                cur[g].prime_commit(first[g]);
                cur[g].start(lut);
            }
            uint32_t rows[kWideGroups][kTileSteps];
            bool pending[kWideGroups];
#pragma unroll
            for (int g = 0; g < kWideGroups; ++g) pending[g] = false;
            // step t is decoded while step t - 1 is multiplied
            auto one = [&](int i, int t) __attribute__((always_inline)) {
                const uint32_t x_now = (uint32_t)(id.k * s.steps + id.t0 + t) * kWideChunks * chunk_bytes;
                u32x4v_t f[2][kQuads];
                fetch(f[0], par ^ 1, 0);
                uint32_t lo[kWideGroups], hi[kWideGroups], nx[kWideGroups];
                bool behind = false;
#pragma unroll
                for (int g = 0; g < kWideGroups; ++g) {
                    const lds_u32* w = cur[g].slot_of(cur[g].pos);
                    lo[g] = w[0];
                    hi[g] = w[kLanes];
                    nx[g] = w[2 * kLanes];
                    behind = behind || cur[g].pos >= cur[g].lim;
                }
                if (__builtin_expect(ballot(behind) != 0, 0)) {
#pragma unroll
                    for (int g = 0; g < kWideGroups; ++g) cur[g].fetch_behind(lo[g], hi[g], nx[g]);
                }
                uint32_t e[kWideGroups][4];
                decode_wide<HAS_ESC>(cur, lut, lo, hi, nx, e, [&](auto round_c, auto rounds_c) __attribute__((always_inline)) {
                    constexpr int kPer = decltype(rounds_c)::value / kWideChunks, c = decltype(round_c)::value / kPer;
                    constexpr int part = decltype(round_c)::value % kPer;
                    __builtin_amdgcn_sched_barrier(0);
                    if (part == 0 && c + 1 < kWideChunks) fetch(f[(c + 1) & 1], par ^ 1, c + 1);
                    multiply(f[c & 1], c, part * kQuads / kPer, (part + 1) * kQuads / kPer);
                    if (part == kPer - 1) x_load(x_now, c);
                    __builtin_amdgcn_sched_barrier(0);
                });
#pragma unroll
                for (int g = 0; g < kWideGroups; ++g) {
                    const uint2 r = rem[i][g];
                    put[g][par * kBuffer] = u32x4v_t{rebuild_pair(e[g][0], rem_lo_pair(r.x)), rebuild_pair(e[g][1], rem_hi_pair(r.x)),
                                                     rebuild_pair(e[g][2], rem_lo_pair(r.y)), rebuild_pair(e[g][3], rem_hi_pair(r.y))};
                }
                rem_load(rem[i], t + kTileSteps);
                lds_barrier();
                par ^= 1;
            };
            for (int t0 = 0; t0 < ns; t0 += kTileSteps) {
#pragma unroll
                for (int g = 0; g < kWideGroups; ++g) {
                    if (pending[g]) cur[g].commit(rows[g]);
                    pending[g] = cur[g].template room<kTileSteps>();
                    if (pending[g]) cur[g].prefetch(rows[g]);
                }
                one(0, t0);
                if (t0 + 1 < ns) one(1, t0 + 1);
            }
        }
#pragma unroll
        for (int c = 0; c < kWideChunks; ++c) {
            u32x4v_t f[kQuads];
            fetch(f, par ^ 1, c);
            multiply(f, c, 0, kQuads);
        }
    };
    if (all_tiles) {
        if (variant) run(std::true_type{}, std::integral_constant<int, NT>{});
        else run(std::false_type{}, std::integral_constant<int, NT>{});
    } else {
        if (variant) run(std::true_type{}, std::integral_constant<int, NT - 1>{});
        else run(std::false_type{}, std::integral_constant<int, NT - 1>{});
    }

    if (a.slices > 1) {
        // K slices meet in the workspace as in tile_kernel, in the registers' own order
        constexpr int kPer = kQuads * NT * 2;             // 8-byte values of a lane
        const size_t slice = (size_t)(s.M / kWideRows) * kWideWaves * kPer * kLanes;
        uint64_t* mine = (uint64_t*)a.partial + ((size_t)rb * kWideWaves + wave) * kPer * kLanes + lane;
#pragma unroll
        for (int w = 0; w < kQuads; ++w) {
#pragma unroll
            for (int n = 0; n < NT; ++n) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint64_t v = (uint64_t)__float_as_uint(acc[w][n][2 * h]) | ((uint64_t)__float_as_uint(acc[w][n][2 * h + 1]) << 32);
                    __hip_atomic_store(mine + ks * slice + ((w * NT + n) * 2 + h) * kLanes, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);      // vmcnt(0): the stores above have completed
        __syncthreads();
        uint32_t& is_last = rings[0][0];
        if (threadIdx.x == 0) {
            const uint32_t old = __hip_atomic_fetch_add(a.counters + rb, 1u, BHI_MMA_ARRIVAL_ORDER, __HIP_MEMORY_SCOPE_AGENT);
            is_last = old == (uint32_t)a.slices - 1;
            if (is_last) {
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                __hip_atomic_store(a.counters + rb, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        __syncthreads();
        if (!is_last) return;
#pragma unroll
        for (int w = 0; w < kQuads; ++w) {
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[w][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
        for (int k = 0; k < a.slices; ++k) {
#pragma unroll
            for (int w = 0; w < kQuads; ++w) {
                uint64_t v[NT * 2];
#pragma unroll
                for (int h = 0; h < NT * 2; ++h)
                    v[h] = __hip_atomic_load(mine + k * slice + (w * NT * 2 + h) * kLanes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int n = 0; n < NT; ++n) {
#pragma unroll
                    for (int i = 0; i < kGroupRows; ++i)
                        acc[w][n][i] += __uint_as_float((uint32_t)(v[2 * n + i / 2] >> (32 * (i & 1))));
                }
            }
        }
    }
    // lane 16 q + j holds rows 4 q .. 4 q + 3 of every sixteen for batch row j of every tile
#pragma unroll
    for (int w = 0; w < kQuads; ++w) {
        const int row0 = (rb * kWideQuads + quad0 + w) * 16 + kGroupRows * (lane >> 4);
        float bias[kGroupRows] = {0.f, 0.f, 0.f, 0.f};
        if (a.bias) {
#pragma unroll
            for (int i = 0; i < kGroupRows; ++i) bias[i] = __uint_as_float((uint32_t)a.bias[row0 + i] << 16);
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int batch = (tile0 + n * kParts) * kTileBatch + (lane & 15);
            if (batch < B) {
                uint2 y;
                if (B <= kMmaMaxBatch) {
                    // up to 32 rows the bias is added to the rounded product, as everywhere below that
                    const uint16_t* bp = a.bias;
                    y.x = finish_output(acc[w][n][0], bp, row0, nullptr) | (uint32_t)finish_output(acc[w][n][1], bp, row0 + 1, nullptr) << 16;
                    y.y = finish_output(acc[w][n][2], bp, row0 + 2, nullptr) | (uint32_t)finish_output(acc[w][n][3], bp, row0 + 3, nullptr) << 16;
                } else {
                    y = make_uint2(f32_to_pair(f32x2_t{acc[w][n][0] + bias[0], acc[w][n][1] + bias[1]}),
                                   f32_to_pair(f32x2_t{acc[w][n][2] + bias[2], acc[w][n][3] + bias[3]}));
                }
                *(uint2*)(a.Y + (size_t)batch * s.M + row0) = y;
            }
        }
    }
}

}  // namespace bhi

// K slices: as many as still give every block a compute unit of its own.
static inline int wide_slices(const bhi::Shape& s) {
    using namespace bhi;
    const int per_group = s.split_k * s.nc;
    int slices = 1;
    for (int d = 2; d <= kWideMaxSlices && d <= per_group; ++d)
        if (per_group % d == 0 && s.M / kWideRows * d <= kWideUnits) slices = d;
    return slices;
}

// Two halves of the weight rows (see above) where they were faster: 144 rows of 4096x12288 46.9 / 48.1 us, rANS 48.6 /
// 53.3; 192 rows 55.2 / 50.3 and 54.8 / 55.4; 256 rows 62.2 / 54.4 and 61.5 / 58.9.
static inline int wide_split(int tiles, bool huffman) { return tiles <= (huffman ? 9 : 12) ? 2 : 1; }

// Counters, X in operand order, and the partial sums of sliced launches, whose tiles are whole rounds of the wavefronts.
static inline int64_t wide_workspace_bytes(const bhi::Shape& s, int batch) {
    using namespace bhi;
    const int64_t tiles = (batch + kTileBatch - 1) / kTileBatch, held = (tiles + kWideWaves - 1) / kWideWaves * kWideWaves;
    const int slices = wide_slices(s);
    return kWideCounterBytes + tiles * kTileBatch * s.split_k * s.Ks * 2 + (slices > 1 ? held * kTileBatch * s.M * 4 * slices : 0);
}

template <class Codec, int NT, int SPLIT>
static inline void launch_wide_n(const bhi::WideArgs& a, const uint16_t* x, hipStream_t stream) {
    using namespace bhi;
    const dim3 grid((unsigned)(a.a.s.M / kWideRows * a.a.slices)), block(kWideThreads);
    hipLaunchKernelGGL((wide_kernel<Codec, NT, SPLIT>), grid, block, 0, stream, x, a);
}

template <class Codec>
static inline int launch_wide(const bhi_gemv_member* weight, const void* X, int split_k, int Ks, int batch, void* workspace,
                              int64_t workspace_bytes, int64_t table_bytes_expected, bool header_is_table, hipStream_t stream) {
    using namespace bhi;
    if (!weight || !X) return bhi_fail(BHI_EINVAL, "null pointer");
    if (batch < kWideMinBatch || batch > kWideMaxBatch) return bhi_fail(BHI_EBATCH, "the wide product takes 17 to 640 rows of X");
    WideArgs wa = {};
    MmaArgs& a = wa.a;
    if (int rc = fill_mma_member(a, *weight, split_k, Ks, batch, table_bytes_expected, header_is_table)) return rc;
    if (a.residual) return bhi_fail(BHI_EINVAL, "the wide product takes no residual");
    if (a.s.M % kWideRows != 0) return bhi_fail(BHI_EINVAL, "the wide product takes whole blocks of 64 weight rows");
    if ((uintptr_t)X % 16 != 0 || (uintptr_t)a.Y % 8 != 0) return bhi_fail(BHI_EINVAL, "X must be aligned to 16 bytes and Y to 8");
    wa.tiles = (batch + kTileBatch - 1) / kTileBatch;
    const int64_t packed_bytes = (int64_t)wa.tiles * kTileBatch * split_k * Ks * 2;
    if (packed_bytes > 0xFFFFFFFFll) return bhi_fail(BHI_EINVAL, "X takes more than 4 GB");
    if (!workspace || workspace_bytes < wide_workspace_bytes(a.s, batch))
        return bhi_fail(BHI_EINVAL, "workspace too small: see bhi_wide_workspace_bytes");
    if ((uintptr_t)workspace % 16 != 0) return bhi_fail(BHI_EINVAL, "the workspace must be aligned to 16 bytes");
    char* const packed = (char*)workspace + kWideCounterBytes;
    a.slices = wide_slices(a.s);
    a.counters = (uint32_t*)workspace;
    a.partial = (float*)(packed + packed_bytes);
    const int K = split_k * Ks, pieces = wa.tiles * (K / 32);
    // both launches before another thread's on this stream: its pack_x_kernel would write over this call's X
    const std::lock_guard<std::mutex> in_a_row(bhi_launches_mutex());
    hipLaunchKernelGGL(pack_x_kernel, dim3((unsigned)((pieces + 3) / 4)), dim3(256), 0, stream, (const uint16_t*)X, (u32x4v_t*)packed,
                       batch, K, wa.tiles);
    const uint16_t* x = (const uint16_t*)packed;
    if (wide_split(wa.tiles, Codec::kHuffman) == 2) {
        switch ((wa.tiles + kWideWaves / 2 - 1) / (kWideWaves / 2)) {
            case 1: launch_wide_n<Codec, 1, 2>(wa, x, stream); break;
            case 2: launch_wide_n<Codec, 2, 2>(wa, x, stream); break;
            default: launch_wide_n<Codec, 3, 2>(wa, x, stream); break;
        }
    } else {
        switch ((wa.tiles + kWideWaves - 1) / kWideWaves) {
            case 2: launch_wide_n<Codec, 2, 1>(wa, x, stream); break;
            case 3: launch_wide_n<Codec, 3, 1>(wa, x, stream); break;
            case 4: launch_wide_n<Codec, 4, 1>(wa, x, stream); break;
            default: launch_wide_n<Codec, 5, 1>(wa, x, stream); break;
        }
    }
    return 0;
}
