// The dense x dense^T projection of square windows of 9 and 11 rows, on the matrix cores.
//
//   C_d[i] = beta * C_d[i] + alpha * sum_c A[i, c] * B[i + k_d, c]
//
// A tile is 64 map positions of 8 map rows, a wave per map row.  v_mfma_f32_4x4x1 makes 16 outer products of 4 x 4: block
// b takes rows 4 b .. 4 b + 3 of A and, for each window row and t = 0 .. T - 1, rows 4 (b + t) .. + 3 of B's map row, and
// adds one batch column to 4 x 4 sums, of which those with 0 <= 4 t + j - v < LC are slots of the window: 75 % at 9 (T =
// 3), 69 % at 11 (T = 4).  The others are sums of their own that nobody reads, so no value of theirs, infinite or not,
// reaches a slot.  A lane is a row in both operands, so a fragment of B for 4 columns is one 16-byte LDS read per lane
// where the columns lie side by side: the staging transposes 4 rows x 4 columns in registers.
//
// Per stage of 4 columns the loads of the next but one stage are on their way, the next one's pass from registers to LDS,
// and there is one barrier.  Nothing in the loop is behind a branch: a wait for loads that may or may not have been issued
// takes the ones just issued with it, which cost a load's whole latency per stage (512 x 512, 11 x 11, batch 64: 89 -> 83 us).
//
// Bound: the matrix cores' issue (a 4x4x1 every 14 clocks per SIMD, two waves on it, where 8 is the instruction's own
// time) and whole rounds of a workgroup per CU.  Measured against the kernel with a wave per window row (vector FMAs, 85 %
// of their rate): 4 maps of 256 x 256 to 4, 9 x 9, batch 128 480 -> 426 us; 512 x 512, 9 x 9, batch 128 145 -> 118;
// 256 x 256 to 2, 11 x 11, batch 512 353 -> 249; 300 x 300, 2 maps to 2, 11 x 11, batch 200 393 -> 337.  Not for 13 x 13, whose
// 208 sums per lane leave too few registers (416 per lane on half the waves: 1012 us on the large layer, 975 by window
// rows), nor for 7 x 7 (58 % of the sums are slots: 332 us, 282 by the window's plane on 512 x 512, batch 512).
//
// Accumulation order, that of the kernel with a wave per window row: batch columns ascending, acc = fma(a, b, acc).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "device.hpp"
#include "kernels.hpp"

namespace cuvdia {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t dp_rsrc(const void *base, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00020000);
}
__device__ __forceinline__ float dp_load(__amdgpu_buffer_rsrc_t r, unsigned off)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

constexpr int DP_XT = 64;                            // map positions of a tile: a lane each
constexpr int DP_COLS = 4;                           // batch columns per stage

// Where row r of a stage lies (in rows of 4 columns): rows of a quad change places with the quad, which spreads the
// staging writes -- a lane's 4 rows one after another -- over the banks.
__device__ __forceinline__ int dp_place(int r) { return (r & ~3) | ((r ^ (r >> 2)) & 3); }

constexpr int DP_YT = 8;                             // map rows of a tile: a wave each
constexpr int DP_MAX_GROUPS = 32;

// The tiles that have slots: those of group g's map-row blocks first_block[g] ..., first_tile[g] tiles before them.
struct DpTiles {
    int first_tile[DP_MAX_GROUPS + 1], first_block[DP_MAX_GROUPS];
};

template <int LC, int K>
struct DpShape {
    static constexpr int T = (LC + 3 + 3) / 4;       // quads of B rows that a quad of A rows meets
    static constexpr int NBR = DP_YT + K - 1;        // map rows of B
    // quads staged per map row: T - 1 behind the tile's own, one for s0 % 4; a multiple of 4, so that a row's place in its
    // quad (dp_place) is the same in every map row
    static constexpr int QPR = (DP_XT / 4 + T + 3) / 4 * 4;
    static constexpr int TASKS = NBR * QPR, NTASK = (TASKS + 64 * DP_YT - 1) / (64 * DP_YT);
    static constexpr int STAGE = NTASK * 64 * DP_YT * 16;        // floats (the last threads' share past the rows is not read)
    static constexpr int RING = 2;                   // window rows whose B is in registers or on their way
    static constexpr int PITCH = DP_XT + 1;          // of a slot's 64 results on their way out
    static_assert(DP_YT * LC * PITCH <= 2 * STAGE, "the results leave through the stages' place");
};

template <int LC, int K>
__global__ __launch_bounds__(64 * DP_YT, 2) void dd2dia_plane_kernel(
    const int *__restrict__ tab, int ngroups, int period, int s0, int astep, float *__restrict__ C,
    const float *__restrict__ A, long long lda, const float *__restrict__ B, long long ldb, int h, int w, int batch,
    float alpha, float beta, unsigned a_bytes, unsigned b_bytes, unsigned c_bytes, int txn, DpTiles tiles)
{
    using S = DpShape<LC, K>;
    constexpr int THREADS = 64 * DP_YT;
    __shared__ __attribute__((aligned(16))) float lds[2 * S::STAGE];
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);

    // each XCD takes a contiguous stretch of the tiles: neighbours share rows of A and B
    const int each = gridDim.x / 8, more = gridDim.x % 8, xcd = blockIdx.x % 8;
    const int tile = xcd * each + min(xcd, more) + blockIdx.x / 8;
    int g = 0;
    while (g + 1 < ngroups && tile >= tiles.first_tile[g + 1]) ++g;
    const int in_group = tile - tiles.first_tile[g], ty = tiles.first_block[g] + in_group / txn, tx = in_group % txn;
    const int i_tile = ty * DP_YT * period + tx * DP_XT;         // the tile's first row of A
    const int s_g = s0 + tab[g];

    const int sh = s_g & 3;                                      // (pieces of B start at multiples of 4 rows)
    const __amdgpu_buffer_rsrc_t ar = dp_rsrc(A, a_bytes), br = dp_rsrc(B, b_bytes), cr = dp_rsrc(C, c_bytes);
    const unsigned lda4 = (unsigned)lda * 4u, ldb4 = (unsigned)ldb * 4u;
    const int row = i_tile + wave * period + lane;               // this lane's row of A
    unsigned b_off[S::NTASK];
#pragma unroll
    for (int k = 0; k < S::NTASK; ++k) {
        const int p = (int)threadIdx.x + THREADS * k, r = p / S::QPR, q = p - r * S::QPR;
        b_off[k] = p < S::TASKS ? (unsigned)(i_tile + s_g - sh + r * period + 4 * q) * 4u : OOB_OFFSET;
    }

    // Columns past the batch and rows outside the operands lie out of the resources' range (0) or in a neighbouring
    // column (slots that are not stored).
    f4 st[S::NTASK][DP_COLS];
    auto request = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < S::NTASK; ++k)
#pragma unroll
            for (int u = 0; u < DP_COLS; ++u) {
                const bool have = (THREADS * (k + 1) <= S::TASKS || (int)threadIdx.x + THREADS * k < S::TASKS) && c + u < batch;
                st[k][u] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(br, have ? b_off[k] + (unsigned)(c + u) * ldb4 : OOB_OFFSET, 0, 0));
            }
    };
    auto place = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < S::NTASK; ++k) {
            const int p = (int)threadIdx.x + THREADS * k;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                *reinterpret_cast<f4 *>(lds + buf * S::STAGE + 4 * dp_place(4 * p + e)) = f4{st[k][0][e], st[k][1][e], st[k][2][e], st[k][3][e]};
        }
    };
    float a_next[DP_COLS];
    auto request_a = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < DP_COLS; ++u) a_next[u] = dp_load(ar, c + u < batch ? (unsigned)row * 4u + (unsigned)(c + u) * lda4 : OOB_OFFSET);
    };

    f4 acc[K][S::T];
#pragma unroll
    for (int d = 0; d < K; ++d)
#pragma unroll
        for (int t = 0; t < S::T; ++t) acc[d][t] = f4{0.f, 0.f, 0.f, 0.f};

    const int stages = (batch + DP_COLS - 1) / DP_COLS;
    request(0);
    request_a(0);
    place(0);
    request(DP_COLS);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const float *const mine = lds + 4 * (wave * 4 * S::QPR);
    int from[S::T];                                  // this lane's row behind each quad
#pragma unroll
    for (int t = 0; t < S::T; ++t) from[t] = 4 * dp_place(lane + sh + 4 * t);
    for (int s = 0; s < stages; ++s) {
        float a[DP_COLS];
#pragma unroll
        for (int u = 0; u < DP_COLS; ++u) {
            a[u] = a_next[u];
            asm volatile("" : "+v"(a[u]));               // (a copy: the wait for it belongs here)
        }
        const float *const st_b = mine + (s & 1) * S::STAGE;
        f4 b[S::RING][S::T];
        auto fetch = [&](int d) __attribute__((always_inline)) {
            if (d < K)
#pragma unroll
                for (int t = 0; t < S::T; ++t) b[d % S::RING][t] = *reinterpret_cast<const f4 *>(st_b + from[t] + 16 * d * S::QPR);
        };
        fetch(0);
        // (no branch, past the last column either: the waits for what is in flight would have to allow for both ways)
        place((s + 1) & 1);
        request_a((s + 1) * DP_COLS);
        request((s + 2) * DP_COLS);
#pragma unroll
        for (int d = 0; d < K; ++d) {
            __builtin_amdgcn_sched_barrier(0);
            fetch(d + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < DP_COLS; ++u)
#pragma unroll
                for (int t = 0; t < S::T; ++t)
                    acc[d][t] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[u], b[d % S::RING][t][u], acc[d][t], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }
    // Results: acc[d][t][v] of lane 4 b + j is slot dx = 4 t + j - v of row 4 b + v; through LDS to a row per lane.
    float *const out = lds + wave * LC * S::PITCH;
    const int j = lane % 4, b4 = lane - j;
    const bool row_ok = tx * DP_XT + lane < period && row < h;
#pragma unroll
    for (int d = 0; d < K; ++d) {
        __builtin_amdgcn_sched_barrier(0);
        wave_lds_fence();
#pragma unroll
        for (int t = 0; t < S::T; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int dx = 4 * t + j - v;
                if ((4 * t - v >= 0 && 4 * t + 3 - v < LC) || (dx >= 0 && dx < LC)) out[dx * S::PITCH + b4 + v] = acc[d][t][v];
            }
        wave_lds_fence();
        const int e0 = tab[ngroups + g * K + d] / 4 + row, in0 = row + s_g + d * period;
        unsigned off[LC];
        float old[LC];
#pragma unroll
        for (int dx = 0; dx < LC; ++dx) {
            off[dx] = row_ok && (unsigned)(in0 + dx) < (unsigned)w ? (unsigned)(e0 + dx * astep) * 4u : OOB_OFFSET;
            old[dx] = 0.f;
            if (beta != 0.f) old[dx] = dp_load(cr, off[dx]);
        }
#pragma unroll
        for (int dx = 0; dx < LC; ++dx) {
            const float sum = out[dx * S::PITCH + lane];
            const float r = beta == 0.f ? alpha * sum : beta * old[dx] + alpha * sum;
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, r), cr, off[dx], 0, 2);
        }
    }
}

template <int LC, int K>
hipError_t dp_launch(const DiaView &C, float *vals, const float *A, long long lda, const float *B, long long ldb, int batch,
                     float alpha, float beta, hipStream_t stream, int txn, const DpTiles &tiles)
{
    const WalkView &wk = C.walk_n;
    note_kernel("dd2dia_plane_kernel<%d, %d>", LC, K);
    launch_kernel((dd2dia_plane_kernel<LC, K>), dim3((unsigned)tiles.first_tile[wk.ngroups]), dim3(64 * DP_YT), 0, stream,
                  wk.tab_dev, wk.ngroups, wk.period, wk.s0, wk.astep4 / 4, vals, A, lda, B, ldb, C.h, C.w, batch, alpha, beta,
                  (unsigned)((((long long)batch - 1) * lda + C.h) * 4), (unsigned)((((long long)batch - 1) * ldb + C.w) * 4),
                  (unsigned)((long long)C.nd * C.stride * 4), txn, tiles);
    return hipGetLastError();
}

// Fills in the launch's tiles; false: another table, operands that 16-byte pieces do not fit, or (not force) a launch on
// which the kernel would not be ahead.
bool dp_plan(const DiaView &C, const float *B, long long lda, long long ldb, int batch, bool force, DpTiles &tiles)
{
    const WalkView &wk = C.walk_n;
    if (wk.tab_dev == nullptr || wk.lck != wk.k || (wk.k != 9 && wk.k != 11) || wk.ngroups > DP_MAX_GROUPS || batch < 1 ||
        !wk.rows4 || wk.period % 4 != 0 || C.h % 4 != 0 || C.w % 4 != 0 || wk.astep4 % 4 != 0 || lda % 4 != 0 || ldb % 4 != 0 ||
        reinterpret_cast<unsigned long long>(B) % 16 != 0)
        return false;
    const long long block = (long long)DP_YT * wk.period, txn = (wk.period + DP_XT - 1) / DP_XT, tyn = (C.h + block - 1) / block;
    // every byte offset, those of rows past the operands' ends included, on its side of 2^32
    long long far = 0;
    for (int g = 0; g < wk.ngroups; ++g) far = std::max(far, std::abs((long long)wk.s0 + wk.rows_host[g]));
    const long long reach = far + tyn * block + 64 * txn + (wk.k + 8LL) * wk.period;
    if ((((long long)batch + 12) * std::max(lda, ldb) + reach) * 4 >= (1LL << 32) || reach >= (1LL << 29) || txn * tyn * wk.ngroups > 0x7fffffffLL)
        return false;
    long long n = 0;
    for (int g = 0; g < wk.ngroups; ++g) {
        // the blocks whose first dense row lies before the operand's end and whose last one not before its start
        const long long first = (long long)wk.s0 + wk.rows_host[g], before = -first - block - (wk.k - 1LL) * wk.period - wk.lck + 2;
        const long long lo = before > 0 ? (before + block - 1) / block : 0;
        const long long hi = std::min(tyn, std::max(0LL, C.w - first + block - 1) / block);
        tiles.first_tile[g] = (int)n;
        tiles.first_block[g] = (int)lo;
        n += std::max(0LL, hi - lo) * txn;
    }
    tiles.first_tile[wk.ngroups] = (int)n;
    if (n == 0) return false;
    // A tile takes a CU to itself for the whole batch, so a launch comes in rounds of 32 tiles per XCD: taken where at least
    // three quarters of the rounds' positions are the map's.  Measured on 16 layers that the kernel with a wave per window
    // row serves otherwise, batch 30 to 1024: 1.0 - 1.4 times its rate where taken, 0.6 - 1.2 elsewhere.
    const long long rounds = ((n + 7) / 8 + 31) / 32;
    return force || (batch >= 24 && 4 * n * wk.period >= 3 * rounds * 256 * txn * DP_XT);
}

}  // namespace

hipError_t launch_dd2dia_plane(const DiaView &C, float *vals, const float *A, long long lda, const float *B, long long ldb,
                               int batch, float alpha, float beta, hipStream_t stream, bool force)
{
    DpTiles tiles;
    if (!dp_plan(C, B, lda, ldb, batch, force, tiles)) return hipErrorNotSupported;
    const int txn = (C.walk_n.period + DP_XT - 1) / DP_XT;
    return C.walk_n.k == 9 ? dp_launch<9, 9>(C, vals, A, lda, B, ldb, batch, alpha, beta, stream, txn, tiles)
                           : dp_launch<11, 11>(C, vals, A, lda, B, ldb, batch, alpha, beta, stream, txn, tiles);
}

}  // namespace cuvdia
