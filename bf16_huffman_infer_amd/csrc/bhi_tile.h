// Fused decode + matrix product for 17 to 128 rows of X: every wavefront decodes four row groups side
// by side and multiplies them with 16x16x32 matrix instructions.
//
// What bounds the range.  Decoding to BF16 and a library GEMM moves the BF16 weight through memory
// twice (4096x12288: 33 us to write it, 25-36 us to read and multiply it).  mma_kernel, which feeds
// 4x4x4 instructions, spends one 16-byte LDS read of X per row group, step and four rows of X; at 32
// rows those reads take as long as the decoding.  With sixteen weight rows in one A operand a read of
// X serves four row groups and four times as many multiplications.
//
// Layout.  Lane 4b + i of a row group's stream holds row i and columns 8b..8b+7 of a step; the A
// operand of the 16x16x32 instruction wants the sixteen lanes of a row of lanes to be sixteen weight
// rows of the same eight columns.  The streams of a wavefront's four groups are independent, so the
// exchange costs nothing: rows are staged as they lie in memory, and each lane then decodes the
// columns whose place in the operand is its own (TileRows).  Only the rem bytes are moved between
// lanes (24 DPP moves and 8 copies a step for four groups; read from memory in the exchanged order
// instead, 32-byte pieces, they cost 2-4 us of 40).  Exchanging the finished weights took 64.
//
// Measured on MI355X, Huffman, four clones in turn, us, before / now (before: mma_kernel up to 32
// rows, decode and library GEMM above):
//
//   M x K          17 rows       32 rows       48 rows       64 rows       96 rows       128 rows
//   4096x4096      22.2 / 16.9   28.4 / 17.1   26.9 / 18.7   27.6 / 20.9   32.4 / 25.3   34.4 / 31.0
//   12288x4096     29.4 / 27.0   36.1 / 27.8   56.3 / 30.8   56.9 / 34.6   58.1 / 40.7   60.8 / 46.5
//   4096x12288     37.4 / 30.1   45.4 / 30.6   59.2 / 34.2   63.5 / 38.5   76.2 / 47.6   84.5 / 54.5
//   18944x3584     45.9 / 36.4   57.2 / 37     65.8 / 39.9   66.1 / 45     68.8 / 60.2   71.0 / 64.3
//
// What bounds it now.  With two tiles of X the decoding: a step of four groups takes 0.83 us with one
// wavefront per SIMD and 1.1 us with two, rem bytes from cache or not.  Every further tile adds 0.13 to 0.16 us
// to a step of eight wavefronts, for which they read 32 KB of X from LDS, each of them all of it for its
// sixteen weight rows: 0.11 us at the 128 bytes a clock that LDS delivers.  At five tiles X staged and read
// is 16 of 72 us (measured with both taken out).  Decoding step t + 1 between the products of step t
// gained nothing.  Long tasks pay more per step: at 28 steps and more lanes drift out of the ring, and where the
// other kernel fills the compute units it is ahead up to 32 rows (16384x3584 at 20 rows: 29.2 there, 38.7 here;
// functional.prefers_tiles).
#pragma once
// (included by bhi_task.h users after bhi_mma.h, whose argument block and workspace it shares)

namespace bhi {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4v_t __attribute__((ext_vector_type(4)));

constexpr int kTileGroups = 4;               // row groups a wavefront decodes side by side: 16 rows
constexpr int kTileRows = kTileGroups * kGroupRows;
constexpr int kTileBatch = 16;               // rows of X per matrix instruction
constexpr int kTileSteps = 2;                // steps between two looks at the rings
constexpr int kTilePrimeRows = 8;            // rows staged before a task's first step
constexpr int tile_ring_words(int rows) { return (rows + 2) * kLanes; }
constexpr int kTileMinBatch = 17, kTileMaxBatch = 128;

// `old` with quad Q of every row of lanes replaced by quad M of `src`.
template <int Q, int M>
__device__ __forceinline__ uint32_t take_quad(uint32_t old, uint32_t src) {
    constexpr int kRotate = Q == M ? 0xE4 : 0x120 + 4 * ((Q - M) & 3);             // quad_perm:[0,1,2,3] or row_ror
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, kRotate, 0xF, 1 << Q, false);
}
// Lane 16k + 4q + i of the result holds what lane 16k + 4M + i of w[q] holds.
template <int M>
__device__ __forceinline__ uint32_t gather_quads(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3) {
    uint32_t v = M == 0 ? w0 : M == 1 ? w1 : M == 2 ? w2 : w3;
    if (M != 0) v = take_quad<0, M>(v, w0);
    if (M != 1) v = take_quad<1, M>(v, w1);
    if (M != 2) v = take_quad<2, M>(v, w2);
    if (M != 3) v = take_quad<3, M>(v, w3);
    return v;
}

// The streams of four row groups, decoded by one wavefront.  Rows are staged group by group, lane f
// of the wavefront loading column f; lane 16 kq + 4 q + i then decodes, in slot m = 0..3, column
// f = 16 kq + 4 m + i of group q: the lane that the matrix instruction wants row 4 q + i in, for the
// columns 8 (4 kq + m).  In group g's ring the four columns 4 m + i of sixteen sit at quad (m + g) % 4,
// so that the sixteen lanes that share kq read sixteen different banks in every slot.
// POS_SHIFT as in RowRingT.
template <int POS_SHIFT, int RING>
struct TileRows {
    uint32_t pos[kTileGroups];               // per slot
    const lds_u32* col[kTileGroups];         // this lane's ring column in slot m
    lds_u32* put[kTileGroups];               // this lane's ring column of group g when rows are staged
    const uint32_t* words;
    uint32_t base[kTileGroups];              // wave-uniform: the groups' task blocks
    uint32_t my_base, my_end;                // those of this lane's group
    uint32_t rhi, lim, nrows;                // wave-uniform: as in RowRingT, one for all four groups

    __device__ __forceinline__ void place(const uint32_t* words_, uint32_t* rings, int lane) {
        words = words_;
        const int kq = lane >> 4, q = (lane >> 2) & 3, i = lane & 3;
#pragma unroll
        for (int m = 0; m < kTileGroups; ++m) {
            col[m] = (const lds_u32*)(lds_u32*)rings + q * tile_ring_words(RING) + 16 * kq + 4 * ((m + q) & 3) + i;
            put[m] = (lds_u32*)rings + m * tile_ring_words(RING) + 16 * kq + 4 * ((q + m) & 3) + i;
        }
    }
    __device__ __forceinline__ void open(const TaskSpan (&span)[kTileGroups], int lane) {
        const int q = (lane >> 2) & 3;
        nrows = 0;
        my_base = my_end = 0;
#pragma unroll
        for (int g = 0; g < kTileGroups; ++g) {
            base[g] = span[g].base;
            const uint32_t n = uniform((span[g].end - span[g].base + kLanes - 1) / kLanes);
            nrows = n > nrows ? n : nrows;
            my_base = q == g ? span[g].base : my_base;
            my_end = q == g ? span[g].end : my_end;
            pos[g] = 0;
        }
    }
    // Rows past the end of a shorter block belong to the block behind it or to the zero pad that ends
    // the stream; they are staged and never decoded.  No group is staged more than a ring past its
    // slowest lane, so at most RING rows past its end: the pad has 32.
    __device__ __forceinline__ void prime_issue(uint32_t (&v)[kTileGroups][kTilePrimeRows], int lane) const {
#pragma unroll
        for (int g = 0; g < kTileGroups; ++g) {
#pragma unroll
            for (int j = 0; j < kTilePrimeRows; ++j) {
                const uint32_t r = (uint32_t)j < nrows ? (uint32_t)j : nrows - 1;
                v[g][j] = (words + base[g] + (size_t)r * kLanes)[lane];
            }
        }
    }
    __device__ __forceinline__ void prime_commit(const uint32_t (&v)[kTileGroups][kTilePrimeRows]) {
#pragma unroll
        for (int g = 0; g < kTileGroups; ++g) {
#pragma unroll
            for (int j = 0; j < kTilePrimeRows; ++j) put[g][j * kLanes] = v[g][j];
            put[g][RING * kLanes] = v[g][0];
            put[g][(RING + 1) * kLanes] = v[g][1];
        }
        rhi = kTilePrimeRows;
        set_lim();
    }
    __device__ __forceinline__ void set_lim() { lim = rhi >= nrows ? 0xFFFFFFFFu : (rhi - 2) << POS_SHIFT; }
    // Can the next two rows of every group be staged: is every lane past the rows they replace?
    __device__ __forceinline__ bool room() const {
        const uint32_t top = rhi + kTileSteps;
        const uint32_t oldest = top > (uint32_t)RING ? (top - RING) << POS_SHIFT : 0u;
        const bool still = pos[0] < oldest || pos[1] < oldest || pos[2] < oldest || pos[3] < oldest;
        return rhi < nrows && ballot(still) == 0;
    }
    __device__ __forceinline__ void prefetch(uint32_t (&v)[kTileGroups][kTileSteps], int lane) const {
#pragma unroll
        for (int g = 0; g < kTileGroups; ++g) {
            const uint32_t* p = words + base[g] + (size_t)rhi * kLanes;
#pragma unroll
            for (int j = 0; j < kTileSteps; ++j) v[g][j] = p[lane + j * kLanes];
        }
    }
    __device__ __forceinline__ void commit(const uint32_t (&v)[kTileGroups][kTileSteps]) {
        const uint32_t slot = (rhi & (RING - 1)) * kLanes;
#pragma unroll
        for (int g = 0; g < kTileGroups; ++g) {
            lds_u32* dst = put[g] + slot;
#pragma unroll
            for (int j = 0; j < kTileSteps; ++j) dst[j * kLanes] = v[g][j];
        }
        if (slot == 0) {
#pragma unroll
            for (int g = 0; g < kTileGroups; ++g) {
                put[g][RING * kLanes] = v[g][0];
                put[g][(RING + 1) * kLanes] = v[g][1];
            }
        }
        rhi += kTileSteps;
        set_lim();
    }
    __device__ __forceinline__ uint32_t column(int m, int lane) const { return (uint32_t)((lane & 0x33) + 4 * m); }
    __device__ __forceinline__ void windows(uint32_t (&lo)[kTileGroups], uint32_t (&hi)[kTileGroups], uint32_t (&nx)[kTileGroups],
                                            int lane) const {
        bool behind = false;
#pragma unroll
        for (int m = 0; m < kTileGroups; ++m) {
            uint32_t slot;
            asm("v_bfe_u32 %0, %1, %2, %3" : "=v"(slot) : "v"(pos[m]), "n"(POS_SHIFT), "n"(ring_rows_log2(RING)));
            const lds_u32* w = col[m] + slot * kLanes;
            lo[m] = w[0];
            hi[m] = w[kLanes];
            nx[m] = w[2 * kLanes];
            behind = behind || pos[m] >= lim;
        }
        if (__builtin_expect(ballot(behind) != 0, 0)) {
            // as RowRingT::fetch_behind
#pragma unroll
            for (int m = 0; m < kTileGroups; ++m) {
                const bool staged = pos[m] < lim;
                const uint32_t* p = words + my_base + (size_t)(staged ? 0u : pos[m] >> POS_SHIFT) * kLanes + column(m, lane);
                const uint32_t p0 = p[0], p1 = p[kLanes], p2 = p[2 * kLanes];
                __builtin_amdgcn_s_waitcnt(0x0F70);
                lo[m] = staged ? lo[m] : p0;
                hi[m] = staged ? hi[m] : p1;
                nx[m] = staged ? nx[m] : p2;
            }
        }
    }
};

template <int RING>
struct HuffTileCursor : TileRows<5, RING> {
    using TileRows<5, RING>::pos;
    using TileRows<5, RING>::words;
    using TileRows<5, RING>::my_end;
    uint32_t eptr;           // escape entries of this lane's group consumed so far

    __device__ __forceinline__ void start() { eptr = 0; }

    template <bool HAS_ESC>
    __device__ __forceinline__ void step(const uint32_t* __restrict__ table, uint32_t (&e)[kTileGroups][4], int lane) {
        constexpr int N = kTileGroups;
        uint32_t lo[N], hi[N], nx[N], w[N], t01[N];
        this->windows(lo, hi, nx, lane);
        const char* tb = (const char*)table;
#pragma unroll
        for (int m = 0; m < N; ++m) {
            w[m] = __builtin_amdgcn_alignbit(hi[m], lo[m], pos[m] & 31u);
            e[m][0] = table_entry(tb, w[m]);
        }
#pragma unroll
        for (int m = 0; m < N; ++m) e[m][1] = table_entry(tb, w[m] >> (e[m][0] & 31u));
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const uint32_t whi = __builtin_amdgcn_alignbit(nx[m], hi[m], pos[m] & 31u);
            t01[m] = e[m][0] + e[m][1];
            w[m] = __builtin_amdgcn_alignbit(whi, w[m], t01[m]);
            e[m][2] = table_entry(tb, w[m]);
        }
#pragma unroll
        for (int m = 0; m < N; ++m) e[m][3] = table_entry(tb, w[m] >> (e[m][2] & 31u));
        uint32_t any = 0;
#pragma unroll
        for (int m = 0; m < N; ++m) {
            pos[m] += (t01[m] + e[m][2] + e[m][3]) & 0x3Fu;
            if (HAS_ESC) any |= e[m][0] | e[m][1] | e[m][2] | e[m][3];
        }
        if (HAS_ESC && __builtin_expect(ballot((int32_t)any < 0) != 0, 0)) escapes(e, lane);
    }

    // Escaped pairs of a group are listed in (pair, column) order; its columns 16 kq + 4 m + i are
    // spread over the slots m and the lanes of quad q.
    __device__ __forceinline__ void escapes(uint32_t (&e)[kTileGroups][4], int lane) {
        const int kq = lane >> 4, q = (lane >> 2) & 3;
        const uint64_t group = 0x000F000F000F000Full << (4 * q);
        const uint64_t here = 0xFFFFull << (16 * kq), before = (1ull << (16 * kq)) - 1;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            uint32_t rank[kTileGroups], in_row = 0, in_front = 0, total = 0;
#pragma unroll
            for (int m = 0; m < kTileGroups; ++m) {
                const uint64_t mask = ballot((int32_t)e[m][d] < 0) & group;
                in_front += (uint32_t)__builtin_popcountll(mask & before);
                total += (uint32_t)__builtin_popcountll(mask);
                rank[m] = in_row + (uint32_t)__builtin_popcountll(mask & here & ((1ull << lane) - 1));
                in_row += (uint32_t)__builtin_popcountll(mask & here);
            }
#pragma unroll
            for (int m = 0; m < kTileGroups; ++m) {
                if ((int32_t)e[m][d] < 0) {
                    const uint32_t v = words[my_end - 1 - (eptr + in_front + rank[m])];
                    e[m][d] = ((v & 0xFFu) << 7) | ((v & 0xFF00u) << 15);
                }
            }
            eptr += total;
        }
    }
};

template <int RING>
struct AnsTileCursor : TileRows<0, RING> {
    using TileRows<0, RING>::pos;
    using TileRows<0, RING>::col;
    uint32_t xl[kTileGroups], xh[kTileGroups];

    // rows 0 and 1 are the initial state (call after prime_commit())
    __device__ __forceinline__ void start() {
#pragma unroll
        for (int m = 0; m < kTileGroups; ++m) {
            xl[m] = col[m][0];
            xh[m] = col[m][kLanes];
            pos[m] = 2;
        }
    }
    template <bool UNUSED>
    __device__ __forceinline__ void step(const uint32_t* __restrict__ table, uint32_t (&e)[kTileGroups][4], int lane) {
        constexpr int N = kTileGroups;
        uint32_t lo[N], hi[N], nx[N], a[N], b[N];
        bool first[N];
        this->windows(lo, hi, nx, lane);
        auto refill = [&](int m, uint32_t word) __attribute__((always_inline)) {
            const bool need = xh[m] == 0u;
            xh[m] = need ? xl[m] : xh[m];
            xl[m] = need ? word : xl[m];
            pos[m] += need ? 1u : 0u;
        };
#pragma unroll
        for (int d = 0; d < kPairsPerStep; ++d) {
#pragma unroll
            for (int m = 0; m < N; ++m) a[m] = AnsCursor::symbol(table, xl[m], xh[m]);
#pragma unroll
            for (int m = 0; m < N; ++m) b[m] = AnsCursor::symbol(table, xl[m], xh[m]);
#pragma unroll
            for (int m = 0; m < N; ++m) {
                e[m][d] = __builtin_amdgcn_perm(b[m], a[m], 0x07060302u);
                if (d == 1) {
                    first[m] = xh[m] == 0u;
                    refill(m, lo[m]);
                }
                if (d == 3) refill(m, first[m] ? hi[m] : lo[m]);
            }
        }
    }
};

// X pieces a thread carries from memory to LDS.
template <int N>
struct TilePieces {
    u32x4v_t v[N];
    uint32_t from[N];        // element of X (row and column group; window start excluded)
    uint32_t to[N];          // 16-byte unit of a window
};

// NB: tiles of sixteen rows of X.  NW wavefronts walk the same columns of NW * 16 weight rows, one step
// at a time, and share the step's X in LDS (double buffered: one barrier a step that orders LDS only;
// windows of two steps and one barrier were no faster, and up to 25 % slower on rANS weights).
// RING rows of exponents per row group: sixteen where LDS holds them; with eight, lanes drift out of the
// ring on long tasks (37 steps: 1.24 us a step instead of 0.84; up to 16 steps it makes no difference).
template <class Codec, int NB, int NW, int RING>
__global__ __launch_bounds__(NW * kLanes, NW == 4 && RING == 16 ? 1 : 2)        // wavefronts per SIMD that LDS leaves room for
void tile_kernel(const uint16_t* __restrict__ X, const MmaArgs a) {
    constexpr int kThreads = NW * kLanes;
    constexpr int kWindow = 4 * NB * kLanes;                  // 16-byte units of one step of X
    constexpr int kLoads = (kWindow + kThreads - 1) / kThreads;
    __shared__ uint32_t rings[NW * kTileGroups][tile_ring_words(RING)];
    __shared__ uint32_t lut[Codec::Table::kLdsWords];
    __shared__ u32x4v_t xbuf[2][kWindow];

    const Shape s = a.s;
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = (int)uniform(threadIdx.x / kLanes);
    const int rb = (int)blockIdx.x / a.slices, ks = (int)blockIdx.x % a.slices;
    const int G = s.M / kGroupRows;
    const int g0 = (rb * NW + wave) * kTileGroups;
    const int tpk = s.split_k * s.nc / a.slices;
    const int kc0 = ks * tpk, kc1 = kc0 + tpk;
    const int K = s.Ks * s.split_k;
    const bool variant = Codec::variant(a.header);
    const int B = a.batch;

    f32x4_t acc[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // X staging.  Piece p of a step = (batch row r, column group b), 16 consecutive threads one row's
    // 256 bytes.  Matrix product m of a step takes the column groups 4 kq + m: lane
    // 16 kq + j reads batch row j of its tile there.  The low three bits of j are XORed with those of
    // b, so that eight neighbouring threads write eight different bank groups.  Rows past the batch
    // repeat its last row.
    TilePieces<kLoads> xp;
#pragma unroll
    for (int n = 0; n < kLoads; ++n) {
        int p = (int)threadIdx.x + n * kThreads;
        p = p < kWindow ? p : kWindow - 1;                    // a thread too many repeats the last piece
        const int b = p & 15, r = p >> 4;
        const int j = r & 15, tile = r >> 4;
        xp.from[n] = (uint32_t)((r < B ? r : B - 1) * K + b * kLaneCols);
        xp.to[n] = (uint32_t)(((b & 3) * NB + tile) * kLanes + 16 * (b >> 2) + (j ^ (b & 7)));
    }
    auto x_load = [&](int k, int t) __attribute__((always_inline)) {
        const uint16_t* x0 = X + (size_t)k * s.Ks + (size_t)t * kStepCols;
#pragma unroll
        for (int n = 0; n < kLoads; ++n) xp.v[n] = *(const u32x4v_t*)(x0 + xp.from[n]);
    };
    auto x_store = [&](int par) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < kLoads; ++n) xbuf[par][xp.to[n]] = xp.v[n];
    };
    uint32_t xlane[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int kq = lane >> 4, b = 4 * kq + m;
        xlane[m] = (uint32_t)(m * NB * kLanes + 16 * kq + ((lane & 15) ^ (b & 7)));
    }

    typename Codec::template TileCursor<RING> cur;
    cur.place(a.exp, rings[wave * kTileGroups], lane);
    int par = 0;
    auto walk = [&](auto has_esc) __attribute__((always_inline)) {
        constexpr bool HAS_ESC = decltype(has_esc)::value;
        for (int kc = kc0; kc < kc1; ++kc) {
            const TaskId id = task_of(s, kc);
            const int ns = id.t1 - id.t0;
            TaskSpan span[kTileGroups];
#pragma unroll
            for (int r = 0; r < kTileGroups; ++r)
                span[r] = task_span(a.offsets, s.M, s.split_k, s.nc, id.k, g0 + r < G ? g0 + r : G - 1, id.c, s.total_words);
            const uint8_t* rem0 = a.rem + ((size_t)id.k * s.M + (size_t)kGroupRows * g0) * s.Ks + (size_t)id.t0 * kLanes * 8;
            uint2 rem[kTileSteps][kTileGroups];
            auto rem_load = [&](uint2 (&dst)[kTileGroups], int t) __attribute__((always_inline)) {
                t = t < ns ? t : ns - 1;
                const uint8_t* p = rem0 + (size_t)t * (kLanes * 8);
#pragma unroll
                for (int g = 0; g < kTileGroups; ++g)        // (past the last group: that group again)
                    dst[g] = stream_load((const uint2*)(p + (ptrdiff_t)(g0 + g < G ? g : G - 1 - g0) * (kGroupRows * s.Ks)) + lane);
            };
#pragma unroll
            for (int i = 0; i < kTileSteps; ++i) rem_load(rem[i], i);
            cur.open(span, lane);
            uint32_t first[kTileGroups][kTilePrimeRows];
            cur.prime_issue(first, lane);
            if (kc == kc0) {
                x_load(id.k, id.t0);
                Codec::Table::fill(lut, a.table);
                x_store(0);
                lds_barrier();
            }
            cur.prime_commit(first);
            cur.start();
            uint32_t rows[kTileGroups][kTileSteps];
            bool pending = false;
            const TaskId after = task_of(s, kc + 1 < kc1 ? kc + 1 : kc);
            // the X of step t, or of the next task's first step (at the very end: of any step)
            auto next_window = [&](int t) __attribute__((always_inline)) {
                const bool here = t < ns;
                x_load(here ? id.k : after.k, here ? id.t0 + t : after.t0);
            };
            auto end_window = [&]() __attribute__((always_inline)) {
                x_store(par ^ 1);
                lds_barrier();
                par ^= 1;
            };
            for (int t0 = 0; t0 < ns; t0 += kTileSteps) {
                if (pending) cur.commit(rows);
                pending = cur.room();
                if (pending) cur.prefetch(rows, lane);
#pragma unroll
                for (int i = 0; i < kTileSteps; ++i) {
                    if (i == 0 || t0 + i < ns) {
                        next_window(t0 + i + 1);
                        uint32_t e[kTileGroups][4];
                        cur.template step<HAS_ESC>(lut, e, lane);
                        const uint2 (&r)[kTileGroups] = rem[i];
                        const uint2 z[kTileGroups] = {
                            make_uint2(gather_quads<0>(r[0].x, r[1].x, r[2].x, r[3].x), gather_quads<0>(r[0].y, r[1].y, r[2].y, r[3].y)),
                            make_uint2(gather_quads<1>(r[0].x, r[1].x, r[2].x, r[3].x), gather_quads<1>(r[0].y, r[1].y, r[2].y, r[3].y)),
                            make_uint2(gather_quads<2>(r[0].x, r[1].x, r[2].x, r[3].x), gather_quads<2>(r[0].y, r[1].y, r[2].y, r[3].y)),
                            make_uint2(gather_quads<3>(r[0].x, r[1].x, r[2].x, r[3].x), gather_quads<3>(r[0].y, r[1].y, r[2].y, r[3].y))};
                        rem_load(rem[i], t0 + i + kTileSteps);
                        const u32x4v_t* xw = xbuf[par];
#pragma unroll
                        for (int m = 0; m < 4; ++m) {
                            const u32x4v_t f = {rebuild_pair(e[m][0], rem_lo_pair(z[m].x)), rebuild_pair(e[m][1], rem_hi_pair(z[m].x)),
                                                rebuild_pair(e[m][2], rem_lo_pair(z[m].y)), rebuild_pair(e[m][3], rem_hi_pair(z[m].y))};
#pragma unroll
                            for (int n = 0; n < NB; ++n)
                                acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, f),
                                                                                 __builtin_bit_cast(bf16x8_t, xw[xlane[m] + n * kLanes]), acc[n], 0, 0, 0);
                        }
                        end_window();
                    }
                }
            }
        }
    };
    if (variant) walk(std::true_type{});
    else walk(std::false_type{});

    // lane 16 q + j holds rows 0..3 of row group q for batch row j of every tile
    const int g = g0 + (lane >> 4), row0 = kGroupRows * g;
    if (a.slices > 1) {
        // K slices meet in the workspace as in mma_kernel (stores that go to the memory side, a
        // relaxed arrival, one acquire in the last block), in the registers' own order: two
        // contiguous 512-byte pieces per tile and wavefront
        const int quads = ((G + kTileGroups - 1) / kTileGroups + NW - 1) / NW * NW;
        uint64_t* mine = (uint64_t*)a.partial + ((size_t)(rb * NW + wave) * NB * 2) * kLanes + lane;
        const size_t slice = (size_t)quads * NB * 2 * kLanes;
#pragma unroll
        for (int n = 0; n < NB; ++n) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint64_t v = (uint64_t)__float_as_uint(acc[n][2 * h]) | ((uint64_t)__float_as_uint(acc[n][2 * h + 1]) << 32);
                __hip_atomic_store(mine + ks * slice + (2 * n + h) * kLanes, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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
        for (int n = 0; n < NB; ++n) acc[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < a.slices; ++k) {
            uint64_t v[NB * 2];
#pragma unroll
            for (int h = 0; h < NB * 2; ++h)
                v[h] = __hip_atomic_load(mine + k * slice + h * kLanes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int n = 0; n < NB; ++n) {
#pragma unroll
                for (int i = 0; i < kGroupRows; ++i)
                    acc[n][i] += __uint_as_float((uint32_t)(v[2 * n + i / 2] >> (32 * (i & 1))));
            }
        }
    }
    // Up to 32 rows a bias is added to the rounded product, as mma_kernel and the GEMV do; above, before
    // the one rounding, as the dense GEMM in whose place this runs.
    auto output = [&](float sum, int row, int batch) __attribute__((always_inline)) {
        if (NB * kTileBatch <= kMmaMaxBatch) return finish_output(sum, a.bias, row, a.residual ? a.residual + (size_t)batch * s.M : nullptr);
        if (a.bias) sum += __uint_as_float((uint32_t)a.bias[row] << 16);
        return finish_output(sum, nullptr, row, a.residual ? a.residual + (size_t)batch * s.M : nullptr);
    };
    if (g < G) {
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const int batch = n * kTileBatch + (lane & 15);
            if (batch < B) {
#pragma unroll
                for (int i = 0; i < kGroupRows; ++i)
                    a.Y[(size_t)batch * s.M + row0 + i] = output(acc[n][i], row0 + i, batch);
            }
        }
    }
}

}  // namespace bhi

// Shape of a launch: wavefronts per block, ring and K slices, by a cost model in microseconds.
//
// A block pays about 5.5 us of launch, first loads and last stores, 0.7 us per task and, for every step,
// a time that grows with the wavefronts on its compute unit and the tiles of X.  Fitted to 4096-column
// weights (us per step at 2 / 4 / 8 tiles: four wavefronts 0.83 / 1.05 / -, six 1.0 / 1.3 / 1.8, eight
// 1.1 / 1.45 / 2.05).  rANS steps take about 1.4 times as long throughout, which leaves the order as it
// is.  Partial sums of K slices cost 1.5 us and 0.1 us per slice and tile.
struct TilePlan { int nw, ring, slices; };

static inline double tile_step_us(int nw, int waves, int ring, int NB) {
    if (ring == 16 && nw == 4) return 0.45 + 0.15 * NB;
    if (ring == 16) return 0.80 + 0.13 * NB;
    return 0.42 + 0.05 * waves + (0.06 + 0.0125 * waves) * NB;
}

static inline TilePlan tile_plan(const bhi::Shape& s, int NB) {
    using namespace bhi;
    const int quads = (s.M / kGroupRows + kTileGroups - 1) / kTileGroups, per_group = s.split_k * s.nc;
    const double steps = (double)s.steps / s.nc;
    // the kernels that are built: what fits 160 KB of LDS (launch_tile_b)
    struct Candidate { int nw, ring, resident; };
    const Candidate candidates[3] = {NB <= 4 ? Candidate{4, 8, 2} : Candidate{4, 16, 1}, {6, NB <= 5 ? 16 : 8, 1}, {8, 8, 1}};
    TilePlan best = {0, 0, 1};
    double best_cost = 0;
    for (const Candidate& c : candidates) {
        const long long row_blocks = (quads + c.nw - 1) / c.nw;
        for (int d = 1; d <= per_group && d <= kMmaMaxSlices; ++d) {
            if (per_group % d != 0 || (d > 1 && row_blocks > kMmaCounterBytes / 4)) continue;      // one counter per row block
            const long long blocks = row_blocks * d, at_once = 256 * c.resident, rest = blocks % at_once;
            const double drift = c.ring == 8 && steps > 16 ? 1 + 0.02 * (steps - 16) : 1;
            auto walk = [&](int waves) { return per_group / d * (steps * drift * tile_step_us(c.nw, waves, c.ring, NB) + 0.7); };
            double cost = 5.5 + (double)(blocks / at_once) * walk(c.nw * c.resident);
            if (rest > 0) cost += walk(c.nw * (int)((rest + 255) / 256));
            if (d > 1) cost += 1.5 + 0.1 * d * NB;
            if (best.nw == 0 || cost < best_cost) { best = TilePlan{c.nw, c.ring, d}; best_cost = cost; }
        }
    }
    return best;
}

static inline int64_t tile_workspace_bytes(const bhi::Shape& s, int batch) {
    using namespace bhi;
    const int NB = (batch + kTileBatch - 1) / kTileBatch;
    const TilePlan plan = tile_plan(s, NB);
    const int block_rows = kTileRows * plan.nw;
    const int64_t rows = (s.M + block_rows - 1) / block_rows * (int64_t)block_rows;
    return plan.slices > 1 ? kMmaCounterBytes + rows * NB * kTileBatch * 4 * plan.slices : 0;
}

template <class Codec, int NB, int NW, int RING>
static inline void launch_tile_n(const bhi::MmaArgs& a, const uint16_t* x, hipStream_t stream) {
    using namespace bhi;
    constexpr int kBlockRows = kTileRows * NW;
    const dim3 grid((unsigned)((a.s.M + kBlockRows - 1) / kBlockRows * a.slices)), block(NW * kLanes);
    hipLaunchKernelGGL((tile_kernel<Codec, NB, NW, RING>), grid, block, 0, stream, x, a);
}

template <class Codec, int NB>
static inline void launch_tile_b(const bhi::MmaArgs& a, const TilePlan& plan, const uint16_t* x, hipStream_t stream) {
    if (plan.nw == 4) return launch_tile_n<Codec, NB, 4, NB <= 4 ? 8 : 16>(a, x, stream);
    if (plan.nw == 6) return launch_tile_n<Codec, NB, 6, NB <= 5 ? 16 : 8>(a, x, stream);
    launch_tile_n<Codec, NB, 8, 8>(a, x, stream);
}

template <class Codec>
static inline int launch_tile(const bhi_gemv_member* weight, const void* X, int split_k, int Ks, int batch, void* workspace,
                              int64_t workspace_bytes, int64_t table_bytes_expected, bool header_is_table, hipStream_t stream) {
    using namespace bhi;
    if (!weight || !X) return bhi_fail(BHI_EINVAL, "null pointer");
    if (batch < kTileMinBatch || batch > kTileMaxBatch) return bhi_fail(BHI_EBATCH, "the tiled product takes 17 to 128 rows of X");
    MmaArgs a = {};
    if (int rc = fill_mma_member(a, *weight, split_k, Ks, batch, table_bytes_expected, header_is_table)) return rc;
    if ((int64_t)batch * split_k * Ks > 0x7FFFFFFFll) return bhi_fail(BHI_EINVAL, "X has more than 2^31 elements");
    const int NB = (batch + kTileBatch - 1) / kTileBatch;
    const TilePlan plan = tile_plan(a.s, NB);
    if (plan.slices > 1) {
        if (!workspace || workspace_bytes < tile_workspace_bytes(a.s, batch))
            return bhi_fail(BHI_EINVAL, "workspace too small: see bhi_tile_workspace_bytes");
        a.slices = plan.slices;
        a.counters = (uint32_t*)workspace;
        a.partial = (float*)((char*)workspace + kMmaCounterBytes);
    }
    const uint16_t* x = (const uint16_t*)X;
    switch (NB) {
        case 2: launch_tile_b<Codec, 2>(a, plan, x, stream); break;
        case 3: launch_tile_b<Codec, 3>(a, plan, x, stream); break;
        case 4: launch_tile_b<Codec, 4>(a, plan, x, stream); break;
        case 5: launch_tile_b<Codec, 5>(a, plan, x, stream); break;
        case 6: launch_tile_b<Codec, 6>(a, plan, x, stream); break;
        case 7: launch_tile_b<Codec, 7>(a, plan, x, stream); break;
        default: launch_tile_b<Codec, 8>(a, plan, x, stream); break;
    }
    return 0;
}
