// The tile-by-tile product of small window tables, a tile being a patch of the window's plane.
//
// A window table of one group pairs output row (y, x) = (i / period, i mod period) with dense rows (y + dy, x + dx), K window
// rows of K diagonals.  A workgroup owns 4 map rows x 32 positions x 32 batch columns and stages, once, all that they need: the
// 4 + K - 1 map rows around them and the K * K diagonals' values.  The kernel that takes 64 rows in a line (spmm_tiled_kernel in
// kernels.hip, of which this is the form for such tables) stages 76 rows x 64 columns anew for every window row, 7 steps with a
// barrier each where this one has 4, and twice the bytes (2.7 times the dense rows, half the values); 1.76 times the accesses of
// the L1 were counted.  A half of a wave owns a group of 8 positions, a lane a column:
// its window is read by 16 bytes, the values are broadcast by DPP in every 16 lanes (fma16_dpp).
//
// Bound: on one round of workgroups (the 16384-unit layer at batch 128: 512) everything happens at once on all CUs -- 1400
// clocks until the first request, 4700 for the requests (a load that writes LDS costs 2.3 clocks per 128-byte line that it
// touches, a column's map row of 38 values touches 3), 5200 of products, 1500 for the exit.  So only what the first two window
// rows need is waited for; the rest is requested between their products.  Kernel arguments that the requests need come preloaded
// in registers (the compiler switch in the Makefile; the prologue takes 1900 clocks otherwise).  Tried: a wait for every window
// row, all requests in front (level, 9.5 us for 9.3); patches of 8 x 16 positions (9.5; 7.3 for 6.9 on 5 x 5 windows); priorities
// for every other workgroup (level); several groups (maps) in turn with one staging buffer (0.7 - 1.15 of the kernels that serve
// them: a CU's two workgroups load and multiply in step); a map row's pieces of all columns dealt to the lanes (13.3: 600
// instructions of addresses).
//
// Measured, us, 15 sets of operands in turn (in a line -> this): 128 x 128, 7 x 7, batch 128 10.4 -> 9.6, with a sigmoid 10.3 -> 9.9,
// added to half of the old values, transposed 11.2 -> 10.7; 96 x 96, 5 x 5, batch 200 11.0 -> 6.6; 64 x 64, 5 x 5, batch 512 9.3 ->
// 6.9; 128 x 128, 3 x 3, batch 128 6.4 -> 5.6; (rows along the lanes) 384 x 384, 7 x 7, batch 32 28.6 -> 22.2.
//
// Accumulation order per output element: window rows ascending, diagonals ascending, acc = fma(a, x, acc).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device.hpp"
#include "kernels.hpp"

namespace cuvdia {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int PT_WAVES = 8, PT_THREADS = 64 * PT_WAVES, PT_COLS = 32;

// n / d by a multiplication, n * d < 2^32
struct PtDiv {
    unsigned d, magic;
    explicit PtDiv(unsigned divisor) : d(divisor), magic(divisor > 1 ? (unsigned)(((1ull << 32) + divisor - 1) / divisor) : 0u) {}
    __device__ static __forceinline__ int of(int n, unsigned magic) { return magic ? (int)__umulhi((unsigned)n, magic) : n; }
};

// A patch: PYG map rows of PXG groups of 8 positions, 32 columns.
template <int K>
struct PtShape {
    static constexpr int LC = K, PXG = 4, PYG = 4, G = PXG * PYG, WIDTH = 8 * PXG;
    static_assert(G == 2 * PT_WAVES, "a group for every half of a wave");
    static constexpr int XW = (8 + LC - 1 + 3) / 4;      // pieces of a lane's window
    static constexpr int NQ = (LC + 1) / 2;              // registers of values: 2 diagonals each
    // Dense rows: [4 columns: a wave's][map row][column][piece], a column's pieces an odd number
    static constexpr int QX = 2 * PXG + (LC - 1 + 3) / 4, XC = PT_COLS / PT_WAVES, XQ = QX | 1, XROW = XC * XQ, R = PYG + K - 1;
    static constexpr int XWAVE = R * XROW + (R * XROW % 8 == 4 ? 0 : 4);     // (4 or 12 modulo 16: no bank conflicts)
    static_assert(XWAVE % 8 == 4, "");
    static_assert(XROW <= 64, "a map row of a wave's columns by one instruction");
    static constexpr int V0 = PT_WAVES * XWAVE;          // the values: [window row][diagonal][group][position]
    static constexpr int VROW = LC * 2 * G;
    static constexpr int BYTES = 16 * (V0 + K * VROW);
    static constexpr int PER_ROW = (LC + 1) / 2;         // value loads of a window row: two diagonals each
    static_assert(2 * PER_ROW <= PT_WAVES, "one of a pair of window rows for every wave at most");
    // What window rows 2 p and 2 p + 1 need beyond those before: dense map rows from rows_to(p - 1) to rows_to(p), value loads
    static constexpr int PAIRS = (K + 1) / 2;
    static constexpr int rows_to(int p) { return p < 0 ? 0 : R < PYG + 2 * p + 1 ? R : PYG + 2 * p + 1; }
    static constexpr int loads(int p) { return (K - 2 * p < 2 ? K - 2 * p : 2) * PER_ROW; }
    static constexpr int OPITCH = WIDTH * PYG + 4;
    static constexpr int LDS = BYTES > 4 * PT_COLS * OPITCH ? BYTES : 4 * PT_COLS * OPITCH;
    static constexpr int PER_CU = 160 * 1024 / LDS < 4 ? 160 * 1024 / LDS : 4;
};

template <int K, bool EP>
__global__ __launch_bounds__(PT_THREADS, 2 * PtShape<K>::PER_CU) void spmm_tiled_kernel(
    const float *__restrict__ X, unsigned ldx, int period, int tiles, unsigned group_tiles, unsigned group_magic,
    unsigned col_group, unsigned col_magic, unsigned tx_count, unsigned tx_magic, int s0, int n_in, int batch, int map_rows,
    const int *__restrict__ tab, const float *__restrict__ vals, unsigned a_bytes, int astep4, int n_out,
    unsigned last_group, unsigned last_magic, int whole_groups,
    float *__restrict__ Y, long long ldy, float alpha, float beta, SpEpilogue ep)
{
    using S = PtShape<K>;
    constexpr int LC = S::LC, PXG = S::PXG, PYG = S::PYG;
    __shared__ __attribute__((aligned(16))) float lds[S::LDS / 4];
    int tile = xcd_tile(blockIdx.x, tiles), coltile;
    {
        // column tiles of a group side by side, then the patches of a map row
        const int cg = PtDiv::of(tile, group_magic);
        tile -= cg * (int)group_tiles;
        const bool last = cg >= whole_groups;
        const int patch = PtDiv::of(tile, last ? last_magic : col_magic);
        coltile = tile - patch * (int)(last ? last_group : col_group) + cg * (int)col_group;
        tile = patch;
    }
    const int ty = PtDiv::of(tile, tx_magic), tx = tile - ty * (int)tx_count;
    constexpr int width = S::WIDTH;
    const int y0 = ty * PYG, rows = min(PYG, map_rows - y0), xrows = rows + K - 1;
    const int xs = max(0, min(tx * width, period - width)), skip = tx * width - xs, xend = min(width, period - xs);
    const int row0 = y0 * period + xs;
    const int col0 = coltile * PT_COLS, cols = min(PT_COLS, batch - col0);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;

    const unsigned x_bytes = ((unsigned)(cols - 1) * ldx + (unsigned)n_in) * 4u;
    const float *const xbase = X + (unsigned long long)ldx * (unsigned)col0;
    const sp_int4 xrsrc = raw_rsrc(xbase, x_bytes);
    const sp_int4 arsrc = raw_rsrc(vals, a_bytes);
    const unsigned ldx4 = ldx * 4u, period4 = 4u * (unsigned)period;
    const unsigned lds0 = (unsigned)(unsigned long long)(__attribute__((address_space(3))) float *)&lds[0];

    // this lane's share of the requests: a piece of a column's map row, a piece of one of two diagonals' values
    const int lc = lane / S::XQ, lq = lane % S::XQ, xcol = S::XC * wave + lc;
    const bool x_lane = lane < S::XROW && lq < S::QX;
    const unsigned x_off = xcol < cols ? (unsigned)xcol * ldx4 + 16u * lq : OOB_OFFSET;
    const unsigned x_to = lds0 + 16u * (unsigned)(wave * S::XWAVE);
    const int vj = lane / (2 * S::G), ve = lane % (2 * S::G), vy = ve / 2 / PXG, vx = 8 * (ve / 2 % PXG) + 4 * (ve % 2);
    const int amin = min(0, astep4 * (LC - 1));
    const unsigned v_off = (unsigned)(astep4 * vj - amin) + period4 * (unsigned)vy + 4u * vx;

    const int gid = 2 * wave + lane / 32, gy = gid / PXG, gx = gid % PXG;
    float acc[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) acc[r] = 0.f;
    const int my_col = lane % 32;
    const f4 *const x_from = reinterpret_cast<const f4 *>(lds) + (my_col / S::XC * S::XWAVE + gy * S::XROW + my_col % S::XC * S::XQ + 2 * gx);
    const float *const v_from = lds + 4 * S::V0 + 4 * (lane / 8 % 2 * 2 * S::G + 2 * gid) + lane % 8;
    const float *const v_last = lds + 4 * S::V0 + 4 * (LC % 2 ? 2 * gid : lane / 8 % 2 * 2 * S::G + 2 * gid) + lane % 8;    // (no diagonal behind the last one)

    // This thread's results: four positions of two columns, 16 bytes each where the patch lies in the map as a whole, else element
    // by element (what does not exist is out of the resource's range).  Old values and biases are asked for here.
    static_assert(PT_THREADS % (2 * PXG * PYG) == 0 && 2 * PT_THREADS >= PT_COLS * 2 * S::G, "two columns' for every thread");
    constexpr int O_STEP = PT_THREADS / (2 * S::G);
    const int o_x = (int)threadIdx.x % (2 * PXG) * 4, o_y = (int)threadIdx.x / (2 * PXG) % PYG, o_col = (int)threadIdx.x / (2 * S::G);
    const __amdgpu_buffer_rsrc_t ybuf = __builtin_amdgcn_make_buffer_rsrc(
        Y + (long long)col0 * ldy, 0, ((unsigned)(cols - 1) * (unsigned)ldy + (unsigned)n_out) * 4u, 0x00020000);
    const bool some = o_y < rows && o_x + 4 > skip && o_x < xend, whole = some && o_x >= skip && o_x + 4 <= xend, part = some && !whole;
    auto place = [&](int k) __attribute__((always_inline)) { return ((unsigned)(o_col + O_STEP * k) * (unsigned)ldy + (unsigned)(o_y * period + o_x)) * 4u; };
    auto column = [&](int k) __attribute__((always_inline)) { return o_col + O_STEP * k < cols; };
    auto element = [&](int i) __attribute__((always_inline)) { return o_x + i >= skip && o_x + i < xend; };
    f4 old[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, bias = {0.f, 0.f, 0.f, 0.f};
    if (beta != 0.f && !(EP && ep.act == 2)) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
            old[k] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(ybuf, whole && column(k) ? place(k) : OOB_OFFSET, 4u * (unsigned)row0, 0));
        if (part) {
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    old[k][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ybuf, column(k) && element(i) ? place(k) + 4u * i : OOB_OFFSET, 4u * (unsigned)row0, 0));
        }
    }
    if (EP && ep.bias && ep.act != 2 && some) {
        const float *const from = ep.bias + row0 + o_y * period + o_x;
        if (whole) bias = *reinterpret_cast<const f4u *>(from);
        else
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (element(i)) bias[i] = from[i];
    }

    auto barrier = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    typedef const int __attribute__((address_space(4))) *Scalars;            // (loads through scalar registers)
    const Scalars table = (Scalars)(unsigned long long)tab;
    const Scalars starts = table + 1;                // (behind the only group's rows)
    const int x0 = row0 + s0, xlast = x0 + (xrows - 1) * period;             // the first and the last map row's first dense row
    if (xlast + width + LC - 1 > 0 && x0 < n_in) {
        const bool inside = x0 >= 0 && xlast + 4 * S::QX <= n_in && row0 + (rows - 1) * period + width <= n_out;
        // a whole patch inside the operand: what the later window rows need is requested between the first ones' products
        const bool staged = inside && rows == PYG;
        auto request_x = [&](int r) __attribute__((always_inline)) {
            if (x_lane) lds_load_b128_scalar(xrsrc, x_to + 16u * (unsigned)(r * S::XROW), x_off, 4u * (unsigned)x0 + (unsigned)r * period4);
        };
        // values: diagonals 2 j, 2 j + 1 of window row d
        auto request_values = [&](int p) __attribute__((always_inline)) {
            if (wave >= S::loads(p)) return;
            const int d = 2 * p + wave / S::PER_ROW, j = wave % S::PER_ROW;
            if (vy < rows && vj < min(2, LC - 2 * j))
                lds_load_b128_scalar(arsrc, lds0 + 16u * (unsigned)(S::V0 + d * S::VROW + j * 4 * S::G), v_off + (unsigned)(2 * j * astep4), (unsigned)(starts[d] + 4 * row0 + amin));
        };
        f4 mend[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        if (inside) {
            static_for<0, S::PAIRS>([&](auto p_) __attribute__((always_inline)) {
                constexpr int p = decltype(p_)::value;
                if (p > 0 && staged) return;
                for (int r = S::rows_to(p - 1); r < min(S::rows_to(p), xrows); ++r) request_x(r);
                request_values(p);
            });
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        } else {
#pragma nounroll
            for (int r = 0; r < xrows; ++r) {
                const int row = x0 + r * period + 4 * lq;
                if (x_lane) lds_load_b128_scalar(xrsrc, x_to + 16u * (unsigned)(r * S::XROW), row >= 0 && row + 4 <= n_in && xcol < cols ? (unsigned)xcol * ldx4 + 4u * (unsigned)row : OOB_OFFSET, 0u);
            }
            // values: element by element, 0 where the dense row does not exist
            constexpr int E = 8 * S::G;
#pragma nounroll
            for (int v = wave; v < K * ((LC * E + 63) / 64); v += PT_WAVES) {
                const int d = v / ((LC * E + 63) / 64), p = 64 * (v % ((LC * E + 63) / 64)) + lane;
                const int dx = p / E, e = p % E, y = e / 8 / PXG, x = 8 * (e / 8 % PXG) + e % 8, row = x0 + (y + d) * period + x + dx;
                if (p < LC * E)
                    lds_load_b32(arsrc, lds0 + 16u * (unsigned)(S::V0 + d * S::VROW) + 256u * (unsigned)(v % ((LC * E + 63) / 64)),
                                 y < rows && row >= 0 && row < n_in && row0 + y * period + x < n_out
                                     ? (unsigned)(starts[d] + 4 * row0 + astep4 * dx + 4 * (y * period + x)) : OOB_OFFSET);
            }
            // pieces that cross an end of the operand: element by element, one column per lane of each half
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int r = wave + PT_WAVES * k, row = x0 + r * period, to = (lane < 32 ? 0 : n_in) - row, q = to / 4;
                if (r < xrows && to > 0 && to % 4 != 0 && q < S::QX && my_col < cols) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int xr = row + 4 * q + e;
                        if (xr >= 0 && xr < n_in) mend[k][e] = xbase[(unsigned)my_col * ldx + (unsigned)xr];
                    }
                }
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            barrier();
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int r = wave + PT_WAVES * k, row = x0 + r * period, to = (lane < 32 ? 0 : n_in) - row, q = to / 4;
                if (r < xrows && to > 0 && to % 4 != 0 && q < S::QX && my_col < cols)
                    *reinterpret_cast<f4 *>(lds + 4 * (my_col / S::XC * S::XWAVE + r * S::XROW + my_col % S::XC * S::XQ + q)) = mend[k];
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        barrier();

        f4 x[2][S::XW];
        float a[2][S::NQ];
        auto read = [&](auto d_) __attribute__((always_inline)) {
            constexpr int d = decltype(d_)::value;
#pragma unroll
            for (int q = 0; q < S::XW; ++q) x[d % 2][q] = x_from[d * S::XROW + q];
#pragma unroll
            for (int q = 0; q < S::NQ; ++q) a[d % 2][q] = (q + 1 < S::NQ ? v_from : v_last)[4 * (d * S::VROW + 2 * q * 2 * S::G)];
        };
        // request n of the later window rows': of every pair a map row, values, a map row
        auto request = [&](auto n_) __attribute__((always_inline)) {
            constexpr int n = decltype(n_)::value, p = 1 + n / 3;
            if constexpr (p < S::PAIRS) {
                if (!staged) return;
                if constexpr (n % 3 == 1) request_values(p);
                else if constexpr (S::rows_to(p - 1) + n % 3 / 2 < S::rows_to(p)) request_x(S::rows_to(p - 1) + n % 3 / 2);
            }
        };
        // the next pair's has come; of this wave's requests the later pairs' may be under way
        auto arrive = [&](auto p_) __attribute__((always_inline)) {
            constexpr int p = decltype(p_)::value;
            if (!staged) return;
            int more = 0;
            static_for<p + 1, S::PAIRS>([&](auto s_) __attribute__((always_inline)) { more += wave < S::loads(decltype(s_)::value); });
            static_for<0, S::PAIRS - p>([&](auto n_) __attribute__((always_inline)) {
                if (more == decltype(n_)::value) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(S::R - S::rows_to(p) + decltype(n_)::value) : "memory");
            });
            barrier();
        };
        read(std::integral_constant<int, 0>{});
        static_for<0, K>([&](auto d_) __attribute__((always_inline)) {
            constexpr int d = decltype(d_)::value;
            static_for<0, S::NQ>([&](auto q_) __attribute__((always_inline)) {
                constexpr int q = decltype(q_)::value;
                if constexpr (q == (d % 2 == 0 ? 0 : S::NQ - 1) && d + 1 < K) {
                    if constexpr (d % 2 == 1) arrive(std::integral_constant<int, (d + 1) / 2>{});
                    read(std::integral_constant<int, d + 1>{});
                }
                float w[4 * S::XW];
#pragma unroll
                for (int i = 0; i < 4 * S::XW; ++i) w[i] = x[d % 2][i / 4][i % 4];
                if constexpr (2 * q + 1 < LC) fma16_dpp(acc, a[d % 2][q], w + 2 * q);
                else fma8_dpp(acc, a[d % 2][q], w + 2 * q);
                // between the first pair's products the requests, all of them before the first wait
                constexpr int at = d * S::NQ + q, slots = 2 * S::NQ - 1, items = 3 * (S::PAIRS - 1);
                if constexpr (at < slots)
                    static_for<(at * items + slots - 1) / slots, ((at + 1) * items + slots - 1) / slots>([&](auto n_) __attribute__((always_inline)) { request(n_); });
            });
        });
    }

    // the sums meet in LDS, in the place of the operands: a column's map rows one after the other
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
#pragma unroll
    for (int r = 0; r < 8; r += 4)
        *reinterpret_cast<f4 *>(lds + my_col * S::OPITCH + 8 * gid + r) = f4{acc[r], acc[r + 1], acc[r + 2], acc[r + 3]};
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
    if (EP && ep.act == 2) {
        // sampled: a thread takes a position and 4 columns, a block of the generator
        constexpr int positions = width * PYG;
#pragma nounroll
        for (int e = threadIdx.x; e < positions * (PT_COLS / 4); e += PT_THREADS) {
            const int c0 = e / positions * 4, pos = e % positions, y = pos / width, x = pos - y * width;
            if (y >= rows || x < skip || x >= xend || c0 >= cols) continue;
            const int row = row0 + y * period + x;
            const float bias = ep.bias ? ep.bias[row] : 0.f;
            const SpRand4 w = sp_philox((unsigned)row, (unsigned)(col0 + c0) / 4u, ep.seed_lo, ep.seed_hi);
            float *const to = Y + (long long)(col0 + c0) * ldy + row;
            float before[4] = {0.f, 0.f, 0.f, 0.f};
            if (beta != 0.f)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (c0 + j < cols) before[j] = to[j * ldy];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (c0 + j >= cols) break;
                const float t = alpha * lds[(c0 + j) * S::OPITCH + pos];
                stream_store(to + j * ldy, sp_finish(beta == 0.f ? t : beta * before[j] + t, bias, 2, w.w[j]));
            }
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        f4 s = *reinterpret_cast<const f4 *>(lds + (o_col + O_STEP * k) * S::OPITCH + o_y * width + o_x);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s[j] = beta == 0.f ? alpha * s[j] : beta * old[k][j] + alpha * s[j];
            if (EP) s[j] = sp_finish(s[j], bias[j], ep.act);
        }
        constexpr int NT = 2;                        // streamed past the caches, as stream_store does (through them: 9.9 us for 9.1)
        buffer_store4<NT>(s, ybuf, whole && column(k) ? place(k) : OOB_OFFSET, 4u * (unsigned)row0);
        if (part) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float e = s[j];
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(e), ybuf, column(k) && element(j) ? place(k) + 4u * j : OOB_OFFSET, 4u * (unsigned)row0, NT);
            }
        }
    }
}

template <int K>
hipError_t patch_launch_one(const PlaneLaunch &L)
{
    using S = PtShape<K>;
    const int map_rows = L.n_out / L.period, tx = (L.period + S::WIDTH - 1) / S::WIDTH, ty = (map_rows + S::PYG - 1) / S::PYG;
    // Column tiles of up to 256 columns side by side, of a wider batch 128: the patches of an XCD stay neighbours.
    const int col_tiles = (L.batch + PT_COLS - 1) / PT_COLS, in_group = col_tiles <= 8 ? col_tiles : 4, rest = col_tiles % in_group;
    const PtDiv row(tx), group(tx * ty * in_group), columns(in_group), last(rest ? rest : in_group);
    const bool fused = L.ep.bias != nullptr || L.ep.act != 0;
    note_kernel("spmm_tiled_kernel<%d, %s>", K, fused ? "true" : "false");
    auto go = [&](auto kernel) {
        launch_kernel(kernel, dim3((unsigned)(tx * ty * col_tiles)), dim3(PT_THREADS), 0, L.stream, L.B, (unsigned)L.ldb, L.period,
                      tx * ty * col_tiles, group.d, group.magic, columns.d, columns.magic, row.d, row.magic, L.s0, L.n_in, L.batch,
                      map_rows, L.tab, L.vals, L.a_bytes, L.astep4, L.n_out, last.d, last.magic, col_tiles / in_group, L.dst, L.ldd,
                      L.alpha, L.beta, L.ep);
    };
    if (fused) go(spmm_tiled_kernel<K, true>);
    else go(spmm_tiled_kernel<K, false>);
    return hipGetLastError();
}

}  // namespace

hipError_t spmm_patch_launch(const PlaneLaunch &L)
{
    switch (L.k) {
        case 3: return patch_launch_one<3>(L);
        case 5: return patch_launch_one<5>(L);
        case 7: return patch_launch_one<7>(L);
        default: return hipErrorNotSupported;
    }
}

// Measured on 16500 random products and layers of one map, 20 to 400 wide, batch 24 to 1024, against the kernels that would run.
//
// In place of the one that takes rows in a line, what counts is how many workgroups of either a CU gets one after the other, as a
// round costs the same whether it is full: 7 x 7 1.10 of its rate where it is not more than there, 0.93 where it is (0.79 on 513 -
// 768 patches, a third workgroup on a few CUs); with so few that every CU has one at most, or two, the other's are ahead on maps
// from 72 wide whose ends its 16-byte pieces fit (one: 0.95; two: sampled ones 0.96, of a bias and widths that are no multiples of 4
// 0.99, the others 1.01).  3 x 3 and 5 x 5, which fit a CU three and four times: 1.25 and 1.23; with more workgroups than there 1.05 - 1.2,
// but on a third, sampled ones on a second one too, 0.92 on maps from 65 wide (1.04 on others, sampled 5 x 5 ones 0.99).  3 x 3 that only
// write a map whose rows are no multiples of 16 bytes leave half lines to memory: 0.92 from a fourth workgroup on, unless the other
// has a quarter more of them, 1.02 - 1.16 on old values, which bring the lines into the caches.  Of 7650 others 6100 come here, at
// 1.16 on average, 3.4 % below 0.97 (the least 0.84); of those left out two thirds are below 0.97, 0.94 on average.
// In place of rows along the lanes, which have a column of
// their own for each: at 1.22 (1.05 - 1.57) on one column tile of 320 patches and more that the map's width fills; 0.7 - 1.1 on
// fewer, 0.8 - 1.0 on a second column tile that is nearly empty.  The plane's walk is ahead where it runs (0.90).
bool spmm_patch_plan(const WalkView &wk, long long n_out, long long n_in, int batch, float beta, const SpEpilogue &ep, bool thin)
{
    if (wk.tab_dev == nullptr || wk.spans == nullptr || wk.spans->work == 0 || wk.ngroups != 1 || wk.lck != wk.k) return false;
    if (wk.k != 3 && wk.k != 5 && wk.k != 7) return false;
    using S = PtShape<7>;
    const long long tx = (wk.period + S::WIDTH - 1) / S::WIDTH, col_tiles = (batch + PT_COLS - 1) / PT_COLS;
    const long long tiles = tx * ((n_out / wk.period + S::PYG - 1) / S::PYG) * col_tiles;
    if (tiles > 0xffff) return false;                // (PtDiv)
    if (thin) return col_tiles == 1 && tiles >= 320 && 20 * wk.period >= 19 * S::WIDTH * tx;
    constexpr int CUS = 256;
    const long long in_a_line = ((n_out + 63) / 64) * ((batch + 63) / 64);     // tiles there
    const long long rounds = (tiles + CUS - 1) / CUS, rounds_there = (in_a_line + CUS - 1) / CUS;
    const bool sampled = ep.act == 2, fused = ep.bias != nullptr || ep.act != 0, quads = wk.period % 4 == 0;
    if (wk.k == 7) {
        if (rounds > rounds_there) return false;
        if (wk.period < 72 || n_in % 4 != 0 || rounds_there > 2) return true;
        return rounds_there == 2 && !sampled && (quads || !fused);
    }
    if (rounds > rounds_there && (rounds == 3 || (rounds == 2 && sampled)) && (wk.period > 64 || (wk.k == 5 && sampled))) return false;
    if (wk.k == 3 && rounds > 3 && !quads && !sampled) return beta == 0.f ? 5 * tiles <= 4 * in_a_line : rounds <= rounds_there;
    return true;
}

}  // namespace cuvdia
