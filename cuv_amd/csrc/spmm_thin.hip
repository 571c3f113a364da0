// The product for few batch columns, and for few tiles of many chunks: rows along the lanes, chunks dealt to the waves.
//
//   dst[r, c] = sum over chunks, over their diagonals j:  A(slot_j)[r] * X[r + s0 + j, c]
//
// With few columns the diagonals' values are (nearly) all of the traffic, and a kernel that keeps one batch column on
// each of 64 lanes spends most of its lanes on columns that do not exist.  Here a lane owns 4 consecutive output rows
// and CB columns (4 * CB running sums): a diagonal's values are one 16-byte load per lane, coalesced along the rows,
// and serve CB columns from registers; a chunk's dense rows are a window of 4 + LC - 1 values per column: NQ 16-byte
// loads that overlap the neighbouring lanes', or -- STAGED -- one load per lane and column, passed on to the
// neighbours through a piece of LDS that belongs to the wave.  No wave waits for another until the end.  4-byte
// alignment is all these loads need: any map width, any leading dimension; addresses are 64 bits wide.
//
// Parallelism comes from the chunks: the waves of a workgroup (and, with G = 4, the four 16-lane groups of each wave)
// take every n-th chunk of the table and their sums meet in LDS, in slice order.  G = 4 gives workgroups of 64 rows
// for products whose rows alone would leave most of the chip idle.
//
// Bound: HBM on large tables (the values once, 3.7 TB/s on the 1024-diagonal layer below), with the L1 path close
// behind (a 16-byte load instruction occupies it for 12 - 20 clocks); latency on small ones.  Measured against the
// kernel with one thread per output row that served these products before: 65536 x 1048576, 1024 diagonals, batch 14
// 1360 -> 91 us; 3 maps of 288 x 288 to 4, 13 x 13, batch 6, transposed 1795 -> 185; 1 map of 33 x 38 to 8, 11 x 11,
// batch 21 715 -> 12; a vector through 4096 rows and 33 diagonals 14 -> 5.
//
// Accumulation order: slice i of S sums its chunks lo + i, lo + i + S, ... (lo: the first chunk with dense rows inside
// the operand) in ascending shift order, diagonals ascending within a chunk, acc = fma(a, x, acc);
// total = ((p0 + p1) + p2) + ...
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device.hpp"
#include "kernels.hpp"

namespace cuvdia {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f4 load4(const float *p) { return *reinterpret_cast<const f4u *>(p); }

// Whether a column's dense rows go through LDS: with 4 or more columns per lane on 256 rows, where the L1 path is busy
// (a window of overlapping 16-byte loads occupies it NQ times); for the small shapes the round trip costs more.
constexpr bool thin_staged(int lc, int cb, int g) { return lc > 1 && cb >= 4 && g == 1; }

template <int LC, int CB, int G>
__global__ __launch_bounds__(64 * (CB == 4 ? 16 : 8)) void spmm_thin_kernel(
    const Chunk *__restrict__ chunks, int nchunks, const float *__restrict__ vals, int stride, int ashift,
    const float *__restrict__ X, long long ldx, float *__restrict__ Y, long long ldy, int n_out, int n_in, int batch,
    int row_blocks, int col_groups, int s_min, int s_max, float alpha, float beta, SpEpilogue ep)
{
    constexpr int LANES = 64 / G;                    // lanes of one chunk slice
    constexpr int ROWS = 4 * LANES;                  // output rows of the workgroup
    constexpr int NQ = (4 + LC - 1 + 3) / 4;         // 16-byte pieces of a window
    constexpr bool STAGED = thin_staged(LC, CB, G);
    constexpr int HQ = NQ > 1 ? NQ - 1 : 1, PITCH = STAGED ? ROWS + 4 * HQ : ROWS;
    static_assert(!STAGED || CB * HQ <= LANES, "the halo is one piece per lane");
    extern __shared__ __attribute__((aligned(16))) float part[];     // [slices][CB][ROWS]

    // Workgroup ids go to the 8 XCDs in turn: each XCD takes a contiguous stretch of row blocks, the column groups of
    // a block side by side, so that a block's values and the rows of neighbouring blocks are found in that XCD's L2.
    const int nblk = row_blocks * col_groups, q = nblk / 8, rest = nblk % 8;
    const int xcd = blockIdx.x % 8, tile = xcd * q + min(xcd, rest) + blockIdx.x / 8;
    const int rb = tile / col_groups, cg = tile - rb * col_groups;
    const int first_row = rb * ROWS, col0 = cg * CB;
    // the last block is moved up to end with the matrix (rows below first_row are computed again and not stored)
    const int row0 = max(0, min(first_row, n_out - ROWS));

    const int waves = blockDim.x / 64;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;
    const int group = G == 1 ? 0 : lane / LANES, l4 = 4 * (lane % LANES);
    const int slices = waves * G;

    f4 acc[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) acc[c] = f4{0.f, 0.f, 0.f, 0.f};
    long long colat[CB];                             // (columns past the batch repeat the last one)
#pragma unroll
    for (int c = 0; c < CB; ++c) colat[c] = (long long)min(col0 + c, batch - 1) * ldx;
    // this slice's dense rows in LDS: a column's ROWS rows and HALO more behind them
    float *const own = part + (wave * G + group) * CB * PITCH;
    const int hc = (lane % LANES) / HQ, hk = ROWS + 4 * ((lane % LANES) % HQ);      // this lane's piece of the halo
    const bool halo = STAGED && hc < CB;
    const long long halo_at = (long long)min(col0 + hc, batch - 1) * ldx + hk;

    // the chunks with dense rows inside the operand: a contiguous range, the table being sorted by shift
    int c_lo = 0, c_hi = nchunks;
    if (!((row0 + s_min + ROWS > 0) & (row0 + s_max < n_in))) {
        c_hi = 0;
        for (int base = 0; base < nchunks; base += 64) {
            const int idx = base + lane, x0 = row0 + chunks[min(idx, nchunks - 1)].s0;
            const unsigned long long before = __builtin_amdgcn_ballot_w64(idx < nchunks && x0 + ROWS + LC - 1 <= 0);
            const unsigned long long upto = __builtin_amdgcn_ballot_w64(idx < nchunks && x0 < n_in);
            c_lo = base == 0 || before ? base + (int)__builtin_popcountll(before) : c_lo;
            c_hi += (int)__builtin_popcountll(upto);
        }
    }

    int ci = c_lo + wave * G + group;
    Chunk next = chunks[min(ci, nchunks - 1)];
    for (; ci < c_hi; ci += slices) {
        const Chunk ch = next;
        next = chunks[min(ci + slices, nchunks - 1)];                // (in flight while this chunk is worked on)
        const int len = min(ch.len, LC), x0 = row0 + ch.s0;
        f4 a[LC], x[CB][STAGED ? 1 : NQ], hq = {0.f, 0.f, 0.f, 0.f};
        constexpr int NX = STAGED ? 1 : NQ;
        if (row0 + ROWS <= n_out && x0 >= 0 && x0 + ROWS + 4 * (NQ - 1) <= n_in) {
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
                for (int k = 0; k < NX; ++k) x[c][k] = load4(X + colat[c] + x0 + l4 + 4 * k);
            if (halo) hq = load4(X + halo_at + x0);
#pragma unroll
            for (int j = 0; j < LC; ++j) {
                const int jj = min(j, len - 1);                      // (a diagonal the chunk does not have: not used)
                a[j] = load4(vals + (long long)ch.slot[j < len ? j : 0] * stride + ashift * (ch.s0 + jj) + row0 + l4);
            }
        } else {
            // a chunk that crosses an end: element by element, what does not exist is 0 (never its padding)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int xr = x0 + l4 + i;
#pragma unroll
                for (int c = 0; c < CB; ++c)
#pragma unroll
                    for (int k = 0; k < NX; ++k)
                        x[c][k][i] = xr + 4 * k >= 0 && xr + 4 * k < n_in ? X[colat[c] + xr + 4 * k] : 0.f;
                if (halo) hq[i] = x0 + hk + i >= 0 && x0 + hk + i < n_in ? X[halo_at + x0 + i] : 0.f;
#pragma unroll
                for (int j = 0; j < LC; ++j) {
                    const float *v = vals + (long long)ch.slot[j < len ? j : 0] * stride;
                    a[j][i] = j < len && xr + j >= 0 && xr + j < n_in && row0 + l4 + i < n_out ? v[ashift ? xr + j : row0 + l4 + i] : 0.f;
                }
            }
        }
        if (STAGED) {
            wave_lds_fence();
#pragma unroll
            for (int c = 0; c < CB; ++c) *reinterpret_cast<f4 *>(own + c * PITCH + l4) = x[c][0];
            if (halo) *reinterpret_cast<f4 *>(own + hc * PITCH + hk) = hq;
            wave_lds_fence();
        }
        auto column = [&](int c, bool whole) {
            f4 win[NQ];
#pragma unroll
            for (int k = 0; k < NQ; ++k)
                win[k] = k < NX ? x[c][k < NX ? k : 0] : *reinterpret_cast<const f4 *>(own + c * PITCH + l4 + 4 * k);
#pragma unroll
            for (int j = 0; j < LC; ++j)
                if (whole || j < len) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[c][i] = __builtin_fmaf(a[j][i], win[(i + j) / 4][(i + j) % 4], acc[c][i]);
                }
        };
        if (len == LC) {
#pragma unroll
            for (int c = 0; c < CB; ++c) column(c, true);
        } else {
            // a chunk shorter than the table's longest: only the diagonals it has (0 * Inf would be a NaN)
#pragma unroll
            for (int c = 0; c < CB; ++c) column(c, false);
        }
    }

    __syncthreads();
    // the slices' sums meet: slice by slice
    const int slice = wave * G + group;
#pragma unroll
    for (int c = 0; c < CB; ++c) *reinterpret_cast<f4 *>(part + (slice * CB + c) * ROWS + l4) = acc[c];
    __syncthreads();
    auto total = [&](int e) {
        float sum = part[e];
        for (int s = 1; s < slices; ++s) sum += part[s * CB * ROWS + e];
        return sum;
    };
    // Sampled: a thread takes as many neighbouring columns of a row as leave every thread some, up to the four that a block of the
    // generator serves.  (With a block for every element -- and its word by index, from memory -- samples took longer than all
    // else: 452 x 452, 3 x 3, 4 maps to 4, batch 28, transposed 194 -> 123 us; 160 x 160, 7 x 7, 1 to 8, batch 33, transposed
    // 67 -> 43; 64 x 64, a band of 9, batch 16 8.4 -> 5.9.)
    auto sampled = [&](auto q_) {
        constexpr int Q = decltype(q_)::value;
        for (int e = threadIdx.x; e < CB / Q * ROWS; e += blockDim.x) {
            const int c = e / ROWS * Q, r = e % ROWS, row = row0 + r, col = col0 + c;
            if (row < first_row || row >= n_out || col >= batch) continue;
            const SpRand4 w = sp_philox((unsigned)row, (unsigned)col >> 2, ep.seed_lo, ep.seed_hi);
            const unsigned upper = 0u - (((unsigned)col >> 1) & 1u), odd = 0u - ((unsigned)col & 1u);    // the first column's place
            const float bias = ep.bias ? ep.bias[row] : 0.f;
#pragma unroll
            for (int i = 0; i < Q; ++i) {
                if (col + i >= batch) break;
                unsigned word = w.w[i];
                if (Q == 2) word = (w.w[i] & ~upper) | (w.w[(2 + i) & 3] & upper);
                if (Q == 1) word = (((w.w[0] & ~upper) | (w.w[2] & upper)) & ~odd) | (((w.w[1] & ~upper) | (w.w[3] & upper)) & odd);
                const float sum = total((c + i) * ROWS + r);
                float *y = Y + (long long)(col + i) * ldy + row;
                stream_store(y, sp_finish(beta == 0.f ? alpha * sum : beta * (*y) + alpha * sum, bias, 2, word));
            }
        }
    };
    if (ep.act == 2) {
        const int share = CB * ROWS / (int)blockDim.x;
        if (CB >= 4 && share >= 4) sampled(std::integral_constant<int, CB >= 4 ? 4 : 1>{});
        else if (CB >= 2 && share >= 2) sampled(std::integral_constant<int, CB >= 2 ? 2 : 1>{});
        else sampled(std::integral_constant<int, 1>{});
        return;
    }
    for (int e = threadIdx.x; e < CB * ROWS; e += blockDim.x) {
        const int c = e / ROWS, r = e - c * ROWS, row = row0 + r, col = col0 + c;
        if (row < first_row || row >= n_out || col >= batch) continue;
        const float sum = total(e);
        float *y = Y + (long long)col * ldy + row;
        const float v = (beta == 0.f) ? alpha * sum : beta * (*y) + alpha * sum;
        stream_store(y, sp_finish(v, ep.bias ? ep.bias[row] : 0.f, ep.act));
    }
}

struct ThinLaunch {
    const Chunk *chunks;
    int nchunks;
    const float *vals;
    int stride, ashift;
    const float *X;
    long long ldx;
    float *Y;
    long long ldy;
    int n_out, n_in, batch, s_min, s_max;
    float alpha, beta;
    SpEpilogue ep;
    hipStream_t stream;
};

template <int LC, int CB, int G>
hipError_t launch_one(const ThinLaunch &L, int waves)
{
    constexpr int ROWS = 4 * (64 / G);
    const long long row_blocks = ((long long)L.n_out + ROWS - 1) / ROWS, col_groups = (L.batch + CB - 1) / CB;
    if (row_blocks * col_groups > 0x7fffffffLL) return hipErrorInvalidValue;
    const size_t lds = (size_t)waves * G * CB * (ROWS + (thin_staged(LC, CB, G) ? 4 * ((LC + 2) / 4) : 0)) * sizeof(float);
    note_kernel("spmm_thin_kernel<%d, %d, %d>", LC, CB, G);
    launch_kernel((spmm_thin_kernel<LC, CB, G>), dim3((unsigned)(row_blocks * col_groups)), dim3(64 * waves), lds, L.stream,
                       L.chunks, L.nchunks, L.vals, L.stride, L.ashift, L.X, L.ldx, L.Y, L.ldy, L.n_out, L.n_in, L.batch,
                       (int)row_blocks, (int)col_groups, L.s_min, L.s_max, L.alpha, L.beta, L.ep);
    return hipGetLastError();
}
template <int LC>
hipError_t launch_lc(const ThinLaunch &L, int cb, int g, int waves)
{
    if (g == 1)
        return cb == 1 ? launch_one<LC, 1, 1>(L, waves) : cb == 2 ? launch_one<LC, 2, 1>(L, waves)
               : cb == 4 ? launch_one<LC, 4, 1>(L, waves) : launch_one<LC, 8, 1>(L, waves);
    return cb == 1 ? launch_one<LC, 1, 4>(L, waves) : launch_one<LC, 2, 4>(L, waves);
}

// Few chunks per row block (launch_spmm_thin): 8 columns per lane only from so many workgroups of them on.
bool thin_few_chunks(int nchunks, double chunks) { return chunks <= (nchunks < 16 ? 18 : 9); }
constexpr int THIN_EIGHT_FROM = 4000;

}  // namespace

bool spmm_thin_ok(const DiaView &A, bool trans)
{
    return A.rf == 1 && (trans ? A.n_chunks_t : A.n_chunks_n) <= NOALLOC_MAX_CHUNKS;
}

bool spmm_thin_by_size(const DiaView &A, bool trans, int batch)
{
    const int n_out = trans ? A.w : A.h, lc = trans ? A.max_len_t : A.max_len_n;
    if (!spmm_thin_ok(A, trans) || lc < 3) return false;
    // The tile-by-tile kernel works through a tile's chunks one after another, 1 - 2 us apart, and always for 64 columns;
    // here eight waves share the chunks and the columns are the ones that exist.  So few tiles of many chunks belong here,
    // and many where a good part of their columns is not there.  Measured on 33500 products of windows of 3 x 3 to 13 x 13,
    // square maps up to 300 wide, batch 24 to 300, with and without the fused layer update: 1.1 - 4 times the tile-by-tile
    // kernel's rate where the tiles' number decides (median 1.8; 0.1 % below 0.97), 0.93 - 2 where the columns do (1st
    // percentile; median 1.37, 2.1 % below 0.97, most of them maps whose width is a multiple of 4); one step beyond these
    // lines a tenth of the products falls below 0.9.  On 2400 products of maps of any shape up to 640 wide, batch up to 640:
    // none and 1.5 % below 0.97, the least 0.90.
    // Up to 35 columns of many tiles: measured on 2742 products and layers of maps up to 520 wide that meet fewer than 14 chunks.
    // Rows 6 and 13 long are behind with 8 columns per lane (337 at a mean of 0.94, the least 0.65; 340 x 340, 6 x 6, 2 maps to 5,
    // batch 25, transposed 184 us tile by tile, 217 here); from 7 on 33 - 35 columns with 8 per lane are a fifth group nearly empty
    // (0.83 - 1.2).  Where a table holds twice the chunks that a row block meets -- one map to more, transposed -- the results are
    // most of the traffic: of rows from 7 on and fewer than 1000 tiles 25 - 28 columns are ahead with an odd length (1.20; 0.88 at
    // the least), not with 8 and 12 (0.71 - 1.3), and more are not (29 - 35: 1.02, a third below 0.97;
    // 32 x 410, 8 x 8, 1 map to 8, batch 30, transposed 32 us tile by tile, 49 here).  The 1945 that come here are at 0.82 - 2.9
    // (mean 1.32, 2 % below 0.97), the 797 left out at a mean of 1.00, half of them below 0.97.  (A second column tile that is
    // nearly empty: 448 x 448, a band of 25, batch 67 59 and 85 us.)
    const double tiles = (n_out + 63) / 64 * (batch / 64.0);     // of the columns that exist
    const double chunks = (double)A.nnz / n_out / lc;            // per tile, those outside the operand left out
    const double there = batch / 64.0 / ((batch + 63) / 64);
    const double most = chunks < 6 ? 40 : chunks < 9.5 ? 56 : chunks < 14 ? 115 : chunks < 40 ? 130 : 250;
    if (batch <= 35 && chunks >= 4 && tiles >= (chunks < 6 ? 1000 : 300)) {
        const int nchunks = trans ? A.n_chunks_t : A.n_chunks_n;
        const long long groups = (n_out + 255) / 256 * (long long)((batch + 7) / 8);
        const bool eight = !thin_few_chunks(nchunks, chunks) || groups >= THIN_EIGHT_FROM, wide = nchunks >= 1.9 * chunks;
        const int most_columns = lc <= 5 ? 35 : !wide ? (eight ? 32 : 35) : tiles >= 1000 ? 32 : lc % 2 == 1 ? 28 : 24;
        if (!(eight && (lc == 6 || lc == 13)) && batch <= most_columns) return true;
    }
    return tiles < most || (chunks >= 14 && there <= (lc <= 5 ? 0.8 : 0.7));
}

hipError_t launch_spmm_thin(const DiaView &A, const float *vals, const float *B, long long ldb,
                            float *dst, long long ldd, int batch, bool trans,
                            float alpha, float beta, SpEpilogue ep, hipStream_t stream)
{
    const ThinLaunch L{trans ? A.chunks_t_dev : A.chunks_n_dev, trans ? A.n_chunks_t : A.n_chunks_n, vals, A.stride,
                       trans ? 1 : 0, B, ldb, dst, ldd, trans ? A.w : A.h, trans ? A.h : A.w, batch,
                       trans ? A.s_min_t : A.s_min_n, trans ? A.s_max_t : A.s_max_n, alpha, beta, ep, stream};
    const int lc = trans ? A.max_len_t : A.max_len_n;
    // The shape, from the products of 24 random layers (measured against every other shape, this choice within a few
    // per cent of the best): as many columns per lane as leave the chip enough workgroups -- every halving reads the
    // values once more --, and where even 2 columns do not, 64 rows per workgroup.  Tables of a chunk per wave are
    // one round of loads whatever the shape: fewer of them per wave end sooner.
    auto wgs = [&](int rows, int cb) { return (((long long)L.n_out + rows - 1) / rows) * ((batch + cb - 1) / cb); };
    const double chunks = (double)A.nnz / L.n_out / lc;         // per row block, those outside the operand left out
    int cb = batch <= 2 ? batch : (batch > 4 && wgs(256, 8) >= 384) ? 8 : wgs(256, 4) >= 128 ? 4 : 2;
    if (L.nchunks <= 8 && cb > 2 && wgs(256, 2) <= 2048) cb = 2;
    int g = 1, waves = L.nchunks < 8 ? L.nchunks : 8;
    if (L.nchunks >= 16 && wgs(256, 2) <= 160) {
        g = 4;
        if (cb > 2) cb = 2;
    } else if (cb == 8 && thin_few_chunks(L.nchunks, chunks)) {
        // Few chunks per row block, however many the table has: 8 waves have nothing to share, and their sums' place in LDS
        // lets two workgroups into a CU.  Measured on 170 random products, up to 16 maps, batch 1 to 140, every shape: of those
        // that come here the choice below is at 1.00 - 2.4 times the rate of 8 columns by 4 or 8 waves (mean 1.35), within 1.2 of
        // the best.  Of 260 others (batch 1 to 139) 33 come here to 4 columns per lane: 0.94 - 2.0 times (median 1.30; the one below
        // 0.99 is 144 x 144, 5 x 5, 2 maps to 1, batch 17: 8.4 -> 9.0 us).  448 x 448, 3 x 3, 1 map to 4, batch 23, transposed 94 -> 45 us; 388 x 388,
        // 7 x 7, batch 12, transposed 33 -> 17.  Tables of 16 chunks and more had 4 waves before: beyond 9 chunks a row block
        // 0.89 - 1.1.
        if (wgs(256, 8) < THIN_EIGHT_FROM) cb = 4;
        const long long n = wgs(256, cb);
        waves = n >= 16000 ? 1 : n >= 3000 || chunks <= 3 ? 2 : 4;
    } else if (cb == 8 && L.nchunks >= 16) {
        waves = 4;
    } else if (cb == 4 && L.nchunks >= 64 && wgs(256, 4) <= 256) {
        waves = 16;
    }
    switch (lc) {
        case 1: return launch_lc<1>(L, cb, g, waves);
        case 2: return launch_lc<2>(L, cb, g, waves);
        case 3: return launch_lc<3>(L, cb, g, waves);
        case 4: return launch_lc<4>(L, cb, g, waves);
        case 5: return launch_lc<5>(L, cb, g, waves);
        case 6: return launch_lc<6>(L, cb, g, waves);
        case 7: return launch_lc<7>(L, cb, g, waves);
        case 8: return launch_lc<8>(L, cb, g, waves);
        case 9: return launch_lc<9>(L, cb, g, waves);
        case 10: return launch_lc<10>(L, cb, g, waves);
        case 11: return launch_lc<11>(L, cb, g, waves);
        case 12: return launch_lc<12>(L, cb, g, waves);
        case 13: return launch_lc<13>(L, cb, g, waves);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace cuvdia
