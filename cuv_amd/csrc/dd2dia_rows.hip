// The dense x dense^T projection, rows along the lanes, each wave on its own.
//
//   C_d[i] = beta * C_d[i] + alpha * sum_c A[i, c] * B[i + k_d, c]
//
// A wave owns 256 rows of one chunk: a lane keeps 4 rows x LC diagonals of running sums and, per batch column, loads
// its 4 values of A and of B (one 16-byte load each) and gets the LC - 1 values of B that follow its own from its
// neighbours through a piece of LDS that belongs to the wave; the next CU columns (2, or 4 on launches of few waves) are in
// flight meanwhile.  No barrier until the end, and 4-byte alignment is all the loads need -- the kernels that share staged
// operands between waves take 16-byte pieces from 16-byte boundaries, and fall to single-element loads where a map's width, the
// leading dimension or a pointer is no multiple of 4 -- and 64-bit addresses: no limit on the operands' sizes.  The waves of a
// workgroup take neighbouring chunks of the same rows (A's values come out of the L1) or, on launches of few tiles,
// ranges of the batch, whose sums meet in LDS.
//
// Bound: the operands' way through the L2 and the L1 (1.2 bytes per multiplication at LC = 7, 0.6 at 13: 30 - 45
// TFLOP/s), latency on small launches.  Measured against the chunk-by-chunk kernel: 1 map of 87 x 87 to 8, 9 x 9,
// batch 458 500 -> 170 us; 83 x 90, 5 x 5, 3 maps to 4, batch 192 115 -> 47; 382 x 382, 7 x 7, 1 map to 16, batch 32 (values of
// 6.5 GB: one thread per slot before) 4470 -> 377; 96 x 96, 5 x 5, 3 maps to 4, batch 14 33 -> 11.
//
// Accumulation order: range r of S sums its steps r, r + S, ... of CU columns in ascending order,
// acc = fma(a, b, acc), in blocks of DR_BLOCK columns (one running sum over a batch of a thousand loses a digit where two
// such gradients are subtracted; the blocks' sums wait in LDS); total = ((p0 + p1) + p2) + ... of blocks and ranges.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device.hpp"
#include "kernels.hpp"

namespace cuvdia {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int DR_ROWS = 256;
constexpr int DR_WAVES = 8, DR_WAVES_MOST = 16;      // waves of a workgroup, at most; ... with the batch in 16 ranges,
constexpr int DR_LC_MOST = 8;                        // ... for whose sums LDS has the place up to here
constexpr int DR_COLS = 2, DR_COLS_FEW = 4;          // batch columns in flight per wave; ... of launches of few waves
// 16 waves leave 128 registers to each: 4 columns of 7 and 8 diagonals do not fit (8 and 12 registers spilled)
constexpr int dr_cols_few(int lc, int waves) { return waves == DR_WAVES_MOST && lc > 6 ? DR_COLS : DR_COLS_FEW; }
constexpr int DR_BLOCK = 128;                        // batch columns per running sum
constexpr int dr_halo(int lc) { return lc > 1 ? (lc + 2) / 4 : 1; }

// 4 consecutive rows from `row` of a column of n rows.  `plain`: the 16 bytes lie inside the allocation (rows outside
// the column then hold a neighbour's values, for slots that are not stored); else element by element.
__device__ __forceinline__ f4 dr_rows(const float *col, int row, int n, bool plain)
{
    if (plain) return *reinterpret_cast<const f4u *>(col + row);
    f4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = col[min(max(row + i, 0), n - 1)];
    return v;
}
// The first of the 4 rows to load for a lane whose rows start at `row`: itself as long as one of them exists.
__device__ __forceinline__ int dr_start(int row, int n) { return row <= -4 ? 0 : row >= n ? n - 4 : row; }

template <int LC, int CU, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void dd2dia_rows_kernel(
    const Chunk *__restrict__ chunks, int nchunks, float *__restrict__ C, int stride, const float *__restrict__ A,
    long long lda, const float *__restrict__ B, long long ldb, int h, int w, int batch, float alpha, float beta,
    int row_blocks, int unit_groups, int splits, int blocks_at)
{
    constexpr int NQ = (LC + 6) / 4, HQ = dr_halo(LC), PITCH = DR_ROWS + 4 * HQ;
    static_assert(CU * HQ <= 64, "the halo is one piece per lane");
    extern __shared__ __attribute__((aligned(16))) float lds[];

    // each XCD takes a contiguous stretch of row blocks, the chunks of a block side by side
    const int nblk = row_blocks * unit_groups, q = nblk / 8, rest = nblk % 8;
    const int xcd = blockIdx.x % 8, tile = xcd * q + min(xcd, rest) + blockIdx.x / 8;
    const int rb = tile / unit_groups, ug = tile - rb * unit_groups;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;
    const int split = wave % splits, unit = ug * ((int)blockDim.x / 64 / splits) + wave / splits;
    const int row0 = rb * DR_ROWS, row = row0 + 4 * lane;
    const Chunk &ch = chunks[min(unit, nchunks - 1)];
    const int slot = ch.slot[min(lane, CHUNK_SLOTS - 1)];       // lane j: the j-th diagonal's position in the table
    const int s0 = ch.s0, len = unit < nchunks ? min(ch.len, LC) : 0, x0 = row0 + s0;
    const bool live = len > 0 && x0 + DR_ROWS + LC > 0 && x0 < w;
    const bool edge = row0 + DR_ROWS > h || x0 < 0 || x0 + PITCH > w;

    f4 acc[LC];
#pragma unroll
    for (int j = 0; j < LC; ++j) acc[j] = f4{0.f, 0.f, 0.f, 0.f};

    if (live) {
        float *const own = lds + wave * CU * PITCH;
        const int arow = dr_start(row, h), brow = dr_start(row + s0, w);
        // this lane's piece of the halo: column hc of a group, rows hk ...
        const int hc = lane / HQ, hk = DR_ROWS + 4 * (lane % HQ), hrow = dr_start(x0 + hk, w);
        const bool halo = NQ > 1 && hc < CU;

        f4 a[CU], b[CU], hv = {0.f, 0.f, 0.f, 0.f};
        auto request = [&](int c0) {
#pragma unroll
            for (int u = 0; u < CU; ++u) {
                const int c = min(c0 + u, batch - 1);
                const bool plain = !edge || (c > 0 && c < batch - 1);
                a[u] = dr_rows(A + (long long)c * lda, plain ? arow : row, h, plain);
                b[u] = dr_rows(B + (long long)c * ldb, plain ? brow : row + s0, w, plain);
            }
            if (halo) {
                const int c = min(c0 + hc, batch - 1);
                const bool plain = !edge || (c > 0 && c < batch - 1);
                hv = dr_rows(B + (long long)c * ldb, plain ? hrow : x0 + hk, w, plain);
            }
        };
        // blocks_at: where in LDS the blocks' sums are (0: a range is one block)
        f4 *const total = reinterpret_cast<f4 *>(lds + blocks_at) + wave * LC * 64 + lane;
        int steps = 0, blocks = 0;
        int c0 = split * CU;
        if (c0 < batch) request(c0);
        for (; c0 < batch; c0 += splits * CU) {
            f4 now[CU];
            wave_lds_fence();
#pragma unroll
            for (int u = 0; u < CU; ++u) {
                now[u] = a[u];
                *reinterpret_cast<f4 *>(own + u * PITCH + 4 * lane) = b[u];
            }
            if (halo) *reinterpret_cast<f4 *>(own + hc * PITCH + hk) = hv;
            wave_lds_fence();
            if (c0 + splits * CU < batch) request(c0 + splits * CU);
#pragma unroll
            for (int u = 0; u < CU; ++u) {
                if (c0 + u < batch) {
                    f4 x[NQ];
#pragma unroll
                    for (int k = 0; k < NQ; ++k) x[k] = *reinterpret_cast<const f4 *>(own + u * PITCH + 4 * lane + 4 * k);
#pragma unroll
                    for (int j = 0; j < LC; ++j)
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[j][i] = __builtin_fmaf(now[u][i], x[(i + j) / 4][(i + j) % 4], acc[j][i]);
                }
            }
            if (blocks_at != 0 && ++steps == DR_BLOCK / CU) {
#pragma unroll
                for (int j = 0; j < LC; ++j) {
                    total[j * 64] = blocks == 0 ? acc[j] : total[j * 64] + acc[j];
                    acc[j] = f4{0.f, 0.f, 0.f, 0.f};
                }
                steps = 0;
                ++blocks;
            }
        }
        if (blocks > 0) {
#pragma unroll
            for (int j = 0; j < LC; ++j) acc[j] = total[j * 64] + acc[j];
        }
    }

    // Results: the diagonals this wave stores are first, first + step, ...; all their old values are requested before
    // the first of them is needed.
    const int first = splits == 1 ? 0 : split, step = splits;
    auto whole = [&](int k) { return row + 3 < h && row + k >= 0 && row + k + 3 < w; };
    auto exists = [&](int k, int i) { return row + i < h && row + i + k >= 0 && row + i + k < w; };
    auto place = [&](int j) { return C + (long long)__builtin_amdgcn_readlane(slot, j) * stride + row; };
    auto old_values = [&](int j) {
        f4 old = {0.f, 0.f, 0.f, 0.f};
        if (beta == 0.f || j >= len) return old;
        const float *c = place(j);
        if (whole(s0 + j)) return static_cast<f4>(*reinterpret_cast<const f4u *>(c));
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (exists(s0 + j, i)) old[i] = c[i];
        return old;
    };
    auto store = [&](int j, f4 v, f4 old) {
        if (j >= len) return;
        float *c = place(j);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = beta == 0.f ? alpha * v[i] : beta * old[i] + alpha * v[i];
        if (whole(s0 + j)) {
            stream_store4(c, v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (exists(s0 + j, i)) c[i] = v[i];
        }
    };
    if (splits == 1) {
        if (live) {
            f4 old[LC];
#pragma unroll
            for (int j = 0; j < LC; ++j) old[j] = old_values(j);
#pragma unroll
            for (int j = 0; j < LC; ++j) store(j, acc[j], old[j]);
        }
        return;
    }
    // the ranges' sums meet in LDS
    constexpr int MOST = (LC + 1) / 2;
    f4 old[MOST];
#pragma unroll
    for (int t = 0; t < MOST; ++t) old[t] = live && first + t * step < LC ? old_values(first + t * step) : f4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();
    f4 *const meet = reinterpret_cast<f4 *>(lds) + (wave - split) * LC * 64 + lane;
#pragma unroll
    for (int j = 0; j < LC; ++j) meet[(split * LC + j) * 64] = acc[j];
    __syncthreads();
    if (!live) return;
#pragma unroll
    for (int t = 0; t < MOST; ++t) {
        const int j = first + t * step;
        if (j >= LC) break;
        f4 sum = meet[j * 64];
        for (int s = 1; s < splits; ++s) sum += meet[(s * LC + j) * 64];
        store(j, sum, old[t]);
    }
}

struct DrLaunch {
    const Chunk *chunks;
    int nchunks;
    float *C;
    int stride;
    const float *A;
    long long lda;
    const float *B;
    long long ldb;
    int h, w, batch;
    float alpha, beta;
    hipStream_t stream;
};

template <int LC>
hipError_t dr_launch(const DrLaunch &L)
{
    constexpr int PITCH = DR_ROWS + 4 * dr_halo(LC);
    const long long row_blocks = ((long long)L.h + DR_ROWS - 1) / DR_ROWS, tiles = row_blocks * L.nchunks;
    // Ranges of the batch side by side: what fills the chip (4096 waves) even if a range then is one step of DR_COLS
    // columns -- a step takes about 1 us whatever the launch's size --, and up to four rounds of waves where each still
    // has 16 columns (one round and a bit takes as long as two: 4851 tiles, batch 544 take 181 us in 4 ranges, 216 in 2).
    int splits = 1;
    while (splits < 8 && ((2 * splits * tiles <= 4096 && 2 * splits * DR_COLS <= L.batch) ||
                          (2 * splits * tiles <= 16384 && 32 * splits <= L.batch)))
        splits *= 2;
    // 16 where each still has 16 columns (and blocks' sums need no place beside the 16 waves' columns): 28 x 28, 7 x 7, 2 maps to
    // 2, batch 864 38 -> 28 us, 32 x 32, 1 map to 8, batch 931 41 -> 30; 8 x 8, 48 x 48, batch 1024 38 -> 33.  With few waves a
    // step is a trip to memory, and 4 columns of one take as long as 2: 8 waves of 7 and 8 diagonals 59 x 59, batch 4096 188 ->
    // 153 us, 61 x 61, batch 224 12.8 -> 12.4.  (One bound of 16 waves for all launches, 4 columns with spilled registers in
    // them: 198 and 13.4, and 48 x 48 36.)
    if (LC <= DR_LC_MOST && splits == 8 && 16 * tiles <= 4096 && L.batch >= 256 && L.batch <= 16 * DR_BLOCK) splits = 16;
    const int waves = splits > 4 ? splits : 4, per = waves / splits;
    const long long groups = (L.nchunks + per - 1) / per;
    if (row_blocks * groups > 0x7fffffffLL) return hipErrorInvalidValue;
    const bool blocks = L.batch > splits * DR_BLOCK;
    const bool few = splits * tiles <= 2048 && 2 * splits * DR_COLS_FEW <= L.batch;
    auto go = [&](auto cu_, auto most_) {
        constexpr int CU = decltype(cu_)::value, MOST = decltype(most_)::value;
        const size_t staged = (size_t)waves * CU * PITCH * sizeof(float), sums = (size_t)waves * LC * 1024;
        const size_t stage = blocks ? staged + sums : staged, meet = splits > 1 ? sums : 0;
        note_kernel("dd2dia_rows_kernel<%d, %d, %d>", LC, CU, MOST);
        launch_kernel((dd2dia_rows_kernel<LC, CU, MOST>), dim3((unsigned)(row_blocks * groups)), dim3(64 * waves),
                      stage > meet ? stage : meet, L.stream, L.chunks, L.nchunks, L.C, L.stride, L.A, L.lda, L.B, L.ldb, L.h, L.w,
                      L.batch, L.alpha, L.beta, (int)row_blocks, (int)groups, splits, blocks ? (int)(staged / sizeof(float)) : 0);
    };
    auto with_waves = [&](auto most) {
        constexpr int FEW = dr_cols_few(LC, decltype(most)::value);
        if (few) go(std::integral_constant<int, FEW>{}, most);
        else go(std::integral_constant<int, DR_COLS>{}, most);
    };
    if constexpr (LC <= DR_LC_MOST) {
        if (waves == DR_WAVES_MOST) with_waves(std::integral_constant<int, DR_WAVES_MOST>{});
    }
    if (waves <= DR_WAVES) with_waves(std::integral_constant<int, DR_WAVES>{});
    return hipGetLastError();
}

}  // namespace

bool dd2dia_rows_ok(const DiaView &C) { return C.rf == 1 && C.h >= 4 && C.w >= 4; }

bool dd2dia_rows_by_size(const DiaView &C, int batch, bool aligned, bool windowed)
{
    if (!aligned) return true;
    // 16-byte pieces fit: the kernels that stage for several waves at a time share more and win with the batch.
    // Measured on 130 random layers (time of the kernel otherwise taken / time of this one): window tables in the
    // plane's kernel 1.0 - 1.8 up to batch 8 where its tiles of 64 positions are not full, 0.6 - 1.1 else; tables of 14
    // chunks or more (several maps) 1.1 - 3 up to batch 64, 0.65 - 1.1 above; pairs in a band of more than 128 rows
    // 1.3 - 1.7 up to batch 128; bands and single windows 0.7 - 1.
    // Measured again with 4 columns in flight and up to 16 ranges, on 1800 gradients of these kinds that had gone elsewhere:
    // More than 1024 tiles of 256 rows and a chunk, batch up to 16: 1.2 - 4.7; windows of one map, whose few chunks share little
    // there, 0.85 - 1.1 above 8 columns of rows up to 4 wide and above 12 of 5 and 6 (5 x 5, 396 x 278, batch 15 11.5 and 13.5 us).
    // Pairs of chunks on up to 256 tiles: 1.1 - 1.5 up to batch 128 (rows 5 wide 0.96 - 1.05 above 96), 0.9 - 1 up to 256, 1.05 -
    // 1.25 where 16 ranges run, up to batch 2048, 0.79 - 0.95 above (8 x 8, 28 x 28, batch 4096 130 and 153 us), 0.9 - 0.96 for
    // 3 columns, two steps of one wave; up to 1024 tiles 1.0 - 1.5 up to batch 48, of bands of a few chunks up to 64 (mean
    // 1.25; a band of 15 on 262 x 262, batch 64 16.4 -> 11.9), of rows 5 and 6 wide up to 16 (5 x 5, 128 x 128, batch 64 6.8 and
    // 8.2).
    // 9 to 12 wide window rows in the plane's kernel: 1.1 - 1.6 up to batch 20, 0.6 - 0.85 above 32.
    // Of 1583 gradients that the lines without these distinctions had sent here 230 are left out, at 0.79 - 1.5 (mean 0.92); the
    // others are at a mean of 1.25, 1 % below 1.0, the least 0.94.
    const long long tiles = (long long)((C.h + DR_ROWS - 1) / DR_ROWS) * C.n_chunks_n;
    const int run = C.max_len_n;
    if (windowed) return C.walk_n.period % 64 != 0 && batch <= (C.walk_n.lck > CHUNK_MAX && C.walk_n.lck < 13 ? 20 : 8);
    const int short_batch = run >= 7 || C.n_chunks_n > run ? 16 : run >= 5 ? 12 : 8;
    if (tiles > 1024 && run <= CHUNK_MAX && C.n_chunks_n > 1 && batch <= short_batch) return true;
    if (C.n_units < C.n_chunks_p && run <= CHUNK_MAX && run >= 5 && tiles <= 1024 && (batch != 3 || tiles > 256)) {
        const int most = tiles <= 256 && C.n_chunks_n < 14 ? (run == 5 ? 96 : 128) : run < 7 ? 16 : C.n_chunks_n < run ? 64 : 48;
        if (batch <= most || (tiles <= 256 && batch > 256 && batch <= DR_WAVES_MOST * DR_BLOCK)) return true;
    }
    if (C.n_chunks_n >= 14) return batch <= 64;
    const bool wide = C.n_units < C.n_chunks_p && C.max_len_n <= CHUNK_MAX && C.pair_delta_max > PAIR_NARROW_DELTA &&
                      C.pair_delta_max <= PAIR_BAND_DELTA;
    return wide && C.max_len_p >= 4 && batch <= 128;
}

hipError_t launch_dd2dia_rows(const DiaView &C, float *vals, const float *A, long long lda, const float *B, long long ldb,
                              int batch, float alpha, float beta, hipStream_t stream)
{
    const DrLaunch L{C.chunks_n_dev, C.n_chunks_n, vals, C.stride, A, lda, B, ldb, C.h, C.w, batch, alpha, beta, stream};
    switch (C.max_len_n) {
        case 1: return dr_launch<1>(L);
        case 2: return dr_launch<2>(L);
        case 3: return dr_launch<3>(L);
        case 4: return dr_launch<4>(L);
        case 5: return dr_launch<5>(L);
        case 6: return dr_launch<6>(L);
        case 7: return dr_launch<7>(L);
        case 8: return dr_launch<8>(L);
        case 9: return dr_launch<9>(L);
        case 10: return dr_launch<10>(L);
        case 11: return dr_launch<11>(L);
        case 12: return dr_launch<12>(L);
        case 13: return dr_launch<13>(L);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace cuvdia
