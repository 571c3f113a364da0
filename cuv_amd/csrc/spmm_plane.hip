// The product with a window table on the matrix cores: the window's plane, walked down column by column.
//
// A window table pairs output row i = (y, x) = (i / period, i mod period) with dense rows (y + dy, x + dx) for K window
// rows dy of LC diagonals dx.  A workgroup owns 32 output positions x of 64 batch columns and walks down the map rows of
// a segment.  At step u it has dense row block u in LDS -- the 32 + LC - 1 rows of map row y0 + u + (first dy) -- which all
// of the K tiles u - K + 1 .. u use, tile m with its window row u - m.  Those tiles are what the matrix instruction's four
// rows are: v_mfma_f32_4x4x1 multiplies four values (of four tiles, for one x and dx, from 4 lanes that its ABID field
// names) with 64 values (dense row x + dx, a batch column per lane) and adds to 4 x 64 sums.  Every product that it makes
// is one that the table has -- a band tiled along x instead would multiply zeros, and a zero times an infinity of the
// dense operand is a NaN --; a slot whose tile has not started or has left only collects values nobody reads.  Of K = 5,
// 9 and 13 tiles one is left over by groups of four: its FMAs go to the vector unit, the value broadcast by DPP.
//
// Per step and wave (8 rows): LC * 8 * ceil(K / 4) matrix instructions of 8 clocks for LC * K * 8 * 64 multiplications,
// 22 - 26 per clock and SIMD where the DPP form of the tile-by-tile kernel does 15, and one staging of the dense rows for
// K window rows.  The walk costs K - 1 steps in which not all tiles are alive (groups of four without any are skipped).
//
// A block's requests follow each other without waiting for anything: the chunks' starts are in LDS, a tile's place comes from
// one of them, blocks at the operand's ends are fetched 4 bytes per lane with what does not exist out of the resource's range
// (element by element, with a wait for each, the few such blocks at a segment's ends held up the launch), and the next block's
// place is worked out behind the requests.  Old values and results go through buffer accesses, their 32-bit offsets in few
// registers: a fourth workgroup per CU for 7 and 8 window rows.  Before -> with all of that, the segments cut for it:
// 7 x 7, 150 x 150, 4 maps to 6, batch 200 346 -> 257 us; 96 x 64, batch 512 183 -> 154; 475 x 475, 1 map, batch 213 177 -> 156;
// 9 x 9, 343 x 343, batch 288 154 -> 139; 5 x 5, 152 x 152, 4 to 4, batch 256 131 -> 119, with a sigmoid on 352 x 352, batch 832
// 283 -> 268.  Three blocks in LDS instead of two: 318 for 302 with three workgroups per CU either way.
//
// Bound: on large windows the matrix cores (13 x 13: two thirds of a launch's time), on small ones the dense rows' way
// from memory; with few steps per segment the walk's ends.  Measured (tile-by-tile kernel -> this one): 4 channels of
// 13 x 13 on 256 x 256, batch 256 1131 -> 800 us (50 -> 71 TFLOP/s); 9 x 9 on 475 x 475, batch 213 264 -> 193; 8 x 8, 1 map of
// 448 x 448 to 2, batch 372 582 -> 354; 9 x 9, 4 maps of 256 x 256 to 4, batch 114 494 -> 300; 7 x 7 on 475 x 475, batch 213
// 202 -> 156; level or behind where the rule below says no.  Of 13 x 13 windows it has the products without bias and activation
// that spmm_split.hip's rule leaves (the bound there on filled tiles).
//
// Accumulation order per output element: window rows ascending, groups in table order within a window row, diagonals
// ascending, acc = fma(a, x, acc).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "device.hpp"
#include "kernels.hpp"

namespace cuvdia {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// A workgroup's tile: 32 rows x 64 columns, 8 rows per wave.  Up to four workgroups share a CU, each with barriers of its
// own: while one waits for its block the others multiply.
constexpr int PLANE_XT = 4;
constexpr int PLANE_WAVES = 4, PLANE_ROWS = 8 * PLANE_WAVES;
constexpr int PLANE_TAB = 256;                       // chunks of a table, at most

template <int LC, int K>
struct PlaneShape {
    static constexpr int TAIL = K % 4 == 1 ? 1 : 0;  // a tile on its own: its FMAs go to the vector unit
    static constexpr int NG = (K - TAIL + 3) / 4;    // groups of 4 tiles
    static constexpr int NQX = (PLANE_ROWS + LC - 1 + 3) / 4;       // 16-byte pieces of a column
    static constexpr int XQ = NQX | 1;                              // ... and from column to column (odd: no bank conflicts)
    static constexpr int XW = (8 + LC - 1 + 3) / 4;                 // pieces of a lane's window
    static constexpr int AROW = PLANE_ROWS, AQ = AROW / 4;          // floats from diagonal to diagonal: 32 banks on ...
    static constexpr int AIT = (AQ * LC + 63) / 64;                 // load instructions per tile
    static constexpr int ASLOT = std::max(LC * AROW, AIT == 1 ? 256 : 0) + 8;   // ... and from tile to tile 8 or 40 (a whole
                                                                                // instruction fits: no lane sits it out)
    static constexpr int NQ = (LC + 1) / 2;                         // registers of values per group: 2 diagonals each
    static constexpr int X_FLOATS = 64 * XQ * 4, STAGE = X_FLOATS + K * ASLOT;
    // The last slot's last register of an odd window row holds a diagonal that does not exist in its upper half: its lanes read
    // on behind the slot, 24 floats behind the last block's of 9, 11 and 13 diagonals.
    static constexpr int LAST_READ = X_FLOATS + (K - 1) * ASLOT + (2 * NQ - 1) * AROW + PLANE_ROWS - 1;
    static constexpr int LDS_FLOATS = STAGE + std::max(STAGE, LAST_READ + 1);
    static constexpr int XIT = (XQ + PLANE_WAVES - 1) / PLANE_WAVES;    // load instructions per wave
    static constexpr int FIT = 160 * 1024 / ((4 * LDS_FLOATS + 4 * PLANE_TAB + 1279) / 1280 * 1280);
    // Workgroups per CU, a wave per SIMD each: as many as fit in LDS and, with the registers that a wave needs, on a SIMD (fused
    // 9 x 9 windows spill 4 there, and are faster all the same: `AHEAD`).
    static constexpr int per_cu(bool fused)
    {
        const int most = K <= 5 ? 4 : K <= 8 ? (fused ? 3 : 4) : 3;
        return FIT < most ? FIT : most;
    }
};

template <int LC, int K, bool EP>
__global__ __launch_bounds__(64 * PLANE_WAVES, (PlaneShape<LC, K>::per_cu(EP))) void spmm_plane_kernel(
    const int *__restrict__ tab, int ngroups, int period, int s0, int astep4, int tp, int nseg, PlaneCuts cuts,
    const float *__restrict__ vals, const float *__restrict__ X, long long ldx, float *__restrict__ Y, long long ldy,
    int n_out, int n_in, int batch, float alpha, float beta, int col_tiles, unsigned a_bytes, SpEpilogue ep)
{
    using S = PlaneShape<LC, K>;
    __shared__ __attribute__((aligned(16))) float lds[S::LDS_FLOATS];
    __shared__ int starts[PLANE_TAB];                // where the chunks' values start

    // A unit -- a segment of PLANE_XT neighbouring walks -- stays on one XCD with all its column tiles: they share the
    // diagonals' values, and the cache lines that tiles side by side have in common.  The last walks of a map row, where
    // there are fewer, are units of their own behind the full ones, without gaps: an XCD deals its workgroups out to its
    // four shader engines in turn, idle ones among them, and with gaps in step with that two of the engines got more than
    // fit into one round (13 x 13, 3 maps of 258 x 258 to 4, batch 72, 9 walks: 927 us with gaps, 559 without).
    const int xcd = blockIdx.x % 8, k8 = blockIdx.x / 8, xgroups = tp / PLANE_XT, full_unit = PLANE_XT * col_tiles;
    const int full_slots = (nseg * xgroups + 7) / 8 * full_unit;
    const bool full = k8 < full_slots;
    const int size = full ? full_unit : tp % PLANE_XT * col_tiles, at = full ? k8 : k8 - full_slots;
    const int unit = at / size * 8 + xcd, within = at % size;
    const int xg = full ? unit / nseg : xgroups, seg = full ? unit - xg * nseg : unit;
    if (full ? xg >= xgroups : seg >= nseg) return;
    const int xt = xg * PLANE_XT + within / col_tiles, coltile = within % col_tiles;
    constexpr int waves = PLANE_WAVES, rows = PLANE_ROWS, nqx = S::NQX;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;
    const int xs = min(xt * rows, period - rows), skip = xt * rows - xs;       // (the last tile of a row is moved up)
    const int seg0 = cuts.at[seg], tiles = cuts.at[seg + 1] - seg0;
    if (tiles <= 0) return;
    const int row_first = xs + seg0 * period;
    const int col0 = coltile * 64, cols = min(64, batch - col0);
    const float *const xbase = X + (long long)col0 * ldx;
    const sp_int4 xrsrc = raw_rsrc(xbase, (unsigned)(((long long)(cols - 1) * ldx + n_in) * 4));
    const sp_int4 arsrc = raw_rsrc(vals, a_bytes);
    const __amdgpu_buffer_rsrc_t yrsrc = __builtin_amdgcn_make_buffer_rsrc(
        Y + (long long)col0 * ldy, 0, (unsigned)(((long long)(cols - 1) * ldy + n_out) * 4), 0x00020000);
    const int amin = min(0, astep4 * (LC - 1));
    const unsigned lds0 = (unsigned)(unsigned long long)(__attribute__((address_space(3))) float *)&lds[0];

    for (int i = threadIdx.x; i < ngroups * K; i += 64 * PLANE_WAVES) starts[i] = tab[ngroups + i];
    const int group_rows = lane < ngroups ? tab[lane] : 0;          // (5 window rows at least: 51 groups at most)

    // this lane's share of a block's requests: byte offsets that stay the same for the whole walk
    unsigned x_off[S::XIT], a_off[S::AIT];
#pragma unroll
    for (int it = 0; it < S::XIT; ++it) {
        const int p = 64 * (wave + waves * it) + lane, col = p / S::XQ, q = p - col * S::XQ;
        x_off[it] = q < nqx ? (unsigned)min(col, cols - 1) * ((unsigned)ldx * 4u) + 16u * q : OOB_OFFSET;
    }
#pragma unroll
    for (int it = 0; it < S::AIT; ++it) {
        const int p = 64 * it + lane, dx = p / S::AQ, q = p - dx * S::AQ;
        a_off[it] = dx < LC ? (unsigned)(astep4 * dx - amin) + 16u * q : OOB_OFFSET;
    }
    auto block_row = [&](int u, int g) { return row_first + s0 + __builtin_amdgcn_readlane(group_rows, g) + u * period; };

    // requests the block of step u (u % K: `slot`) whose dense rows start at x0: those rows, and the values of the tiles that
    // use them; lane d of `first` has where the group's chunk of window row d starts
    auto issue = [&](int u, int slot, int first, int x0, int buf) {
        const unsigned base = lds0 + (unsigned)(buf * S::STAGE * 4);
        const bool inside = x0 >= 0 && x0 + 4 * nqx <= n_in;
        if (inside) {
#pragma unroll
            for (int it = 0; it < S::XIT; ++it) {
                const int i = wave + waves * it;
                if (i < S::XQ) lds_load_b128(xrsrc, base + 1024u * i, x_off[it], (unsigned)x0 * 4u);
            }
        } else {
            // the block crosses an end of the operand: element by element, what does not exist is 0
            for (int i = wave; i < 4 * S::XQ; i += waves) {
                const int p = 64 * i + lane, col = p / (4 * S::XQ), r = p - col * (4 * S::XQ), row = x0 + r;
                const bool there = r < 4 * nqx && (unsigned)row < (unsigned)n_in;
                lds_load_b32(xrsrc, base + 256u * i,
                             there ? (unsigned)min(col, cols - 1) * ((unsigned)ldx * 4u) + 4u * row : OOB_OFFSET);
            }
        }
        for (int s = wave; s < K; s += waves) {
            const int d = slot - s + (slot < s ? K : 0), m = u - d;  // the tile in slot s, and its window row
            if (m < 0 || m >= tiles) continue;
            const int at = __builtin_amdgcn_readlane(first, d) + 4 * (row_first + m * period);
            const unsigned to = base + (unsigned)((S::X_FLOATS + s * S::ASLOT) * 4);
            if (inside) {
#pragma unroll
                for (int it = 0; it < S::AIT; ++it)
                    if (256 * (it + 1) <= S::ASLOT || 256 * it + 4 * lane < S::ASLOT)
                        lds_load_b128(arsrc, to + 1024u * it, a_off[it], (unsigned)(at + amin));
            } else {
                for (int it = 0; it < (LC * S::AROW + 63) / 64; ++it) {
                    const int p = 64 * it + lane, dx = p / S::AROW, r = p % S::AROW;
                    const bool there = (unsigned)(x0 + r + dx) < (unsigned)n_in;
                    if (dx < LC)
                        lds_load_b32(arsrc, to + 256u * it, there ? (unsigned)(at + astep4 * dx + 4 * r) : OOB_OFFSET);
                }
            }
        }
    };

    f4 acc[S::NG][8];                                // tiles 4 g + i of rows r in acc[g][r][i]; a lane is a column
    float tail[8];                                   // the tile that no group has
#pragma unroll
    for (int r = 0; r < 8; ++r) {
#pragma unroll
        for (int g = 0; g < S::NG; ++g) acc[g][r] = f4{0.f, 0.f, 0.f, 0.f};
        tail[r] = 0.f;
    }
    // where this lane reads values: lane 4 b + i of a group's register: row b % 8, diagonal 2 q + b / 8, tile i
    const int lane_a = (lane % 4) * S::ASLOT + (lane / 32) * S::AROW + (lane / 4) % 8 + 8 * wave;
    const int lane_last = lane_a - std::max(0, 4 * (S::NG - 1) + lane % 4 - (K - 1)) * S::ASLOT;
    const int lane_t = (S::NG * 4) * S::ASLOT + (lane % 16 / 8) * S::AROW + lane % 8 + 8 * wave;

    auto multiply = [&](int u, int buf) {
        const float *const st = lds + buf * S::STAGE;
        float x[4 * S::XW];
#pragma unroll
        for (int q = 0; q < S::XW; ++q) {
            const f4 v = *reinterpret_cast<const f4 *>(st + lane * (4 * S::XQ) + 8 * wave + 4 * q);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[4 * q + e] = v[e];
        }
        auto value = [&](int g, int q) {
            // (slots past the last tile, diagonals past the last one: any value of the array, never used)
            return st[S::X_FLOATS + (4 * g + 3 < K ? lane_a : lane_last) + 4 * g * S::ASLOT + 2 * q * S::AROW];
        };
        // tiles alive at this step: max(0, u - K + 1) .. min(u, tiles - 1)
        const int lo = max(0, u - K + 1), n = min(u, tiles - 1) - lo + 1, s_lo = lo % K;
        const unsigned ones = (1u << n) - 1u, alive = (ones << s_lo) | (ones >> (K - s_lo));
        static_for<0, S::NG>([&](auto g_) {
            constexpr int g = decltype(g_)::value;
            if (!((alive >> (4 * g)) & 15u)) return;
            static_for<0, S::NQ>([&](auto q_) {
                constexpr int q = decltype(q_)::value;
                const float v = value(g, q);
                static_for<0, 16>([&](auto b_) {
                    constexpr int b = decltype(b_)::value, r = b % 8, dx = 2 * q + b / 8;
                    if constexpr (dx < LC) acc[g][r] = __builtin_amdgcn_mfma_f32_4x4x1f32(v, x[r + dx], acc[g][r], 4, b, 0);
                });
            });
        });
        if constexpr (S::TAIL) {
            if ((alive >> (4 * S::NG)) & 1u) {
                static_for<0, S::NQ>([&](auto q_) {
                    constexpr int q = decltype(q_)::value;
                    const float v = st[S::X_FLOATS + lane_t + 2 * q * S::AROW];
                    if constexpr (2 * q + 1 < LC) fma16_dpp(tail, v, x + 2 * q);
                    else fma8_dpp(tail, v, x + 2 * q);
                });
            }
        }
    };

    // A finished tile leaves through LDS, in the place of a block that is done with, so that a column's 32 rows are
    // written together: lane (c, q) holds rows 4 q .. 4 q + 3 of columns 16 wave + c and 16 wave + 8 + c.
    constexpr int OPITCH = PLANE_ROWS + 4;
    static_assert(64 * OPITCH <= S::STAGE, "a tile fits a block's place");
    const int my_row = 4 * (lane % 8), my_col = 16 * wave + lane / 8;
    // (what lies past the batch or before the rows of this walk is out of the resource's range)
    auto place = [&](int c, int r) { return c < cols && r >= skip ? (unsigned)c * ((unsigned)ldy * 4u) + 4u * r : OOB_OFFSET; };
    const int sample_row = lane % 32, sample_col = 16 * wave + 8 * (lane / 32);   // sampled: a lane takes a row and 8 columns
    const bool reads_old = beta != 0.f;
    f4 old[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    auto read_old = [&](int m) {
        const unsigned tile_at = (unsigned)(row_first + m * period) * 4u;
        // (sampled: all before the first store; one by one between the stores each waited for memory: 5 x 5, 272 x 63, 1 map to 8,
        // batch 670, transposed 404 us like that, 276 now; 8 x 8, 364 x 364, batch 273 279 and 185; 9 x 9, 467 x 467, batch 860
        // 1410 and 984; 11 x 11, 128 x 251, 1 to 8, batch 898 1955 and 1233)
        if (EP && ep.act == 2) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                old[i / 4][i % 4] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(yrsrc, place(sample_col + i, sample_row), tile_at, 0));
            return;
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (skip == 0) {
                old[k] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(yrsrc, place(my_col + 8 * k, my_row), tile_at, 0));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    old[k][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(yrsrc, place(my_col + 8 * k, my_row + i), tile_at, 0));
            }
        }
    };
    auto finish = [&](int m, const float (&v)[8], float *out) {
        const unsigned tile_at = (unsigned)(row_first + m * period) * 4u;
        __builtin_amdgcn_s_barrier();                // nobody reads the block any more
        asm volatile("" ::: "memory");
#pragma unroll
        for (int r = 0; r < 8; r += 4) *reinterpret_cast<f4 *>(out + lane * OPITCH + 8 * wave + r) = f4{v[r], v[r + 1], v[r + 2], v[r + 3]};
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (EP && ep.act == 2) {
            // sampled: two blocks of the generator
            const int r = sample_row, c0 = sample_col, row = row_first + m * period + r;
            const float bias = ep.bias ? ep.bias[row] : 0.f;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const SpRand4 w = sp_philox((unsigned)row, (unsigned)(col0 + c0) / 4u + h, ep.seed_lo, ep.seed_hi);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int c = c0 + 4 * h + i;
                    const float t = alpha * out[c * OPITCH + r];
                    const float p = sp_finish(beta == 0.f ? t : beta * old[h][i] + t, bias, 2, w.w[i]);
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(p), yrsrc, place(c, r), tile_at, 0);
                }
            }
            return;
        }
        float bias[4] = {0.f, 0.f, 0.f, 0.f};
        if (EP && ep.bias) {
#pragma unroll
            for (int i = 0; i < 4; ++i) bias[i] = ep.bias[row_first + m * period + my_row + i];
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            f4 s = *reinterpret_cast<const f4 *>(out + (my_col + 8 * k) * OPITCH + my_row);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[i] = beta == 0.f ? alpha * s[i] : beta * old[k][i] + alpha * s[i];
                if (EP) s[i] = sp_finish(s[i], bias[i], ep.act);
            }
            if (skip == 0) {
                buffer_store4<0>(s, yrsrc, place(my_col + 8 * k, my_row), tile_at);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s[i]), yrsrc, place(my_col + 8 * k, my_row + i), tile_at, 0);
            }
        }
    };

    // The blocks (u, g) in order, one requested ahead.  Of the groups only those with rows anywhere in the segment are
    // looked through at its steps (group rows ascend): with one map to 16, transposed, looking through all of them took
    // longer than multiplying (7 x 7, 134 x 134, batch 321: 524 us so, 351 as it is; tile by tile 369).
    const int steps = tiles + K - 1;
    int g0 = 0, g1 = ngroups;
    while (g0 < g1 && block_row(steps - 1, g0) + rows + LC - 1 <= 0) ++g0;
    while (g0 < g1 && block_row(0, g1 - 1) >= n_in) --g1;
    // the block to be requested next: its step, step % K, group, first dense row, and where its chunks' values start
    int nu = g0 < g1 ? 0 : steps, nslot = 0, ng = g0 - 1, nx0 = 0, first = 0;
    auto advance = [&]() {
        do {
            if (++ng >= g1) {
                ng = g0;
                ++nu;
                nslot = nslot + 1 == K ? 0 : nslot + 1;
            }
            nx0 = block_row(nu, ng);
        } while (nu < steps && (nx0 + rows + LC - 1 <= 0 || nx0 >= n_in));
        first = starts[ng * K + (lane < K ? lane : 0)];
    };
    __syncthreads();                                 // (the starts are in place)
    if (nu < steps) advance();
    int pu = nu;                                     // the step of the block that was requested last
    int buf = 0;                                     // its place
    auto request = [&](int to) {
        pu = nu;
        if (nu >= steps) return;
        issue(nu, nslot, first, nx0, to);
        advance();
    };
    request(0);
    // A tile's old values are requested with the last of its blocks and held for its length, or requested at its exit; the code for
    // the first is the faster one also where none are read.  11 x 11, 402 x 310, batch 477, transposed 348 us held, 395 at the
    // exit; 9 x 9 with a sigmoid, 512 x 563, batch 86 116 and 132 (held, 4 registers are spilled; with two workgroups per CU none
    // are, and 132); 5 x 5 with a sigmoid, 352 x 352, batch 832 268 and 293.  Without bias and activation four workgroups of 5, 7
    // and 8 window rows have no registers to hold them (level).
    constexpr bool AHEAD = S::per_cu(EP) < 4 || (EP && K == 5);
    int slot = 0;                                    // u % K
    for (int u = 0; u < steps; ++u) {
        static_for<0, K>([&](auto s_) {
            constexpr int s = decltype(s_)::value;
            if (slot == s && u < tiles) {
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    if constexpr (s < 4 * S::NG) acc[s / 4][r][s % 4] = 0.f;
                    else tail[r] = 0.f;
                }
            }
        });
        const int done = u - (K - 1);                // the tile that ends with this step
        bool old_read = !reads_old || done < 0;
        while (pu == u) {
            // (for a finished tile's stores as well: to leave them under way took a branch on whether there are any, and cost more
            // than their wait: 7 x 7, 475 x 475, batch 213, with a sigmoid 188 us with it, 169 without, plain 162 and 156; 9 x 9,
            // 256 x 256, 4 maps to 4, batch 114 340 and 300)
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            request(buf ^ 1);
            if (AHEAD && !old_read) {
                read_old(done);
                old_read = true;
            }
            multiply(u, buf);
            buf ^= 1;
        }
        if (done >= 0) {
            if (AHEAD && !old_read) read_old(done);
            const int leaving = slot + 1 == K ? 0 : slot + 1;
            float v[8];
            static_for<0, K>([&](auto s_) {
                constexpr int s = decltype(s_)::value;
                if (leaving == s) {
#pragma unroll
                    for (int r = 0; r < 8; ++r) {
                        if constexpr (s < 4 * S::NG) v[r] = acc[s / 4][r][s % 4];
                        else v[r] = tail[r];
                        asm volatile("" : "+v"(v[r]));       // (keeps the compiler from indexing the sums in memory)
                    }
                }
            });
            if (!AHEAD) {
                old[0] = old[1] = f4{0.f, 0.f, 0.f, 0.f};            // (not held in between)
                if (!old_read) read_old(done);
            }
            finish(done, v, lds + (buf ^ 1) * S::STAGE);
        }
        slot = slot + 1 == K ? 0 : slot + 1;
    }
}

template <int LC, int K>
hipError_t plane_launch_one(const PlaneLaunch &L)
{
    const bool fused = L.ep.bias != nullptr || L.ep.act != 0;
    const long long full = (long long)L.nseg * (L.tp / PLANE_XT), part = L.nseg;       // units (the kernel's head)
    const unsigned grid = (unsigned)(((full + 7) / 8 * PLANE_XT + (part + 7) / 8 * (L.tp % PLANE_XT)) * 8 * L.col_tiles);
    note_kernel("spmm_plane_kernel<%d, %d, %s>", LC, K, fused ? "true" : "false");
    auto go = [&](auto kernel) {
        launch_kernel(kernel, dim3(grid), dim3(64 * PLANE_WAVES), 0, L.stream, L.tab, L.ngroups, L.period, L.s0, L.astep4, L.tp,
                      L.nseg, L.cuts, L.vals, L.B, L.ldb, L.dst, L.ldd, L.n_out, L.n_in, L.batch, L.alpha, L.beta,
                      L.col_tiles, L.a_bytes, L.ep);
    };
    if constexpr (K < 13) {
        if (fused) go(spmm_plane_kernel<LC, K, true>);
        else go(spmm_plane_kernel<LC, K, false>);
    } else {
        go(spmm_plane_kernel<LC, K, false>);         // (fused: spmm_plane_plan leaves them to spmm_split.hip)
    }
    return hipGetLastError();
}

}  // namespace

hipError_t spmm_plane_launch(const PlaneLaunch &L)
{
    switch (L.k) {
        case 5: return plane_launch_one<5, 5>(L);
        case 7: return plane_launch_one<7, 7>(L);
        case 8: return plane_launch_one<8, 8>(L);
        case 9: return plane_launch_one<9, 9>(L);
        case 11: return plane_launch_one<11, 11>(L);
        case 13: return plane_launch_one<13, 13>(L);
        default: return hipErrorNotSupported;
    }
}

// Every segment walks (its map rows + k - 1) steps of as many blocks as groups have rows there: the map rows are cut where that
// work divides evenly, at multiples of `every` from the segment's first (plane_cut).  Between two ends of groups' ranges the
// groups are the same.  How many: workgroups run on 32 CUs per XCD, a unit of `unit` walks with its column tiles on one XCD;
// shares[n] is how long a CU takes for n workgroups at once, in workgroups of a CU that holds as many as it can, the last entry
// (plane_over, which returns the time, in steps of such workgroups, over the segments' own).
double plane_over(const PlaneSpans &spans, int walk_len, int unit, int per_cu, const double *shares, double walk_ends, PlaneLaunch &L)
{
    const long long work = spans.work;
    const int full = L.tp / unit, part = L.tp % unit;
    auto time = [&](int segs) {
        const int wgs = ((segs * full + 7) / 8 * unit + (segs * (part > 0) + 7) / 8 * part) * L.col_tiles, n = (wgs + 31) / 32;
        return n / per_cu * shares[per_cu] + shares[n % per_cu];
    };
    double best = -1;
    int n = 1;
    for (int i = 1; i <= PLANE_MAX_SEGMENTS && i <= walk_len; ++i) {
        const double t = time(i);
        if (best >= 0 && t * walk_ends >= best) break;       // (more segments never run in less)
        const double cost = t * ((double)work / i + walk_ends);
        if (best < 0 || cost < best) {
            best = cost;
            n = i;
        }
    }
    L.nseg = n;
    return best * 8 * 32 / std::max(1.0, (double)work * L.tp * L.col_tiles);
}

void plane_cut(const PlaneSpans &spans, int walk_len, int every, PlaneLaunch &L)
{
    const std::vector<int> &ends = spans.ends, &groups = spans.groups;
    const long long work = spans.work;
    const int n = L.nseg;
    L.nseg = 0;
    long long done = 0;
    size_t i = 0;
    L.cuts.at[0] = 0;
    for (int s = 1; s < n; ++s) {
        const long long want = work * s / n;
        while (i + 2 < ends.size() && done + (long long)groups[i] * (ends[i + 1] - ends[i]) <= want) {
            done += (long long)groups[i] * (ends[i + 1] - ends[i]);
            ++i;
        }
        const int at = groups[i] ? ends[i] + (int)((want - done) / groups[i]) : ends[i], last = L.cuts.at[L.nseg];
        const int cut = last + (at - last + every / 2) / every * every;
        if (cut > last && cut < walk_len) L.cuts.at[++L.nseg] = cut;
    }
    L.cuts.at[++L.nseg] = walk_len;
}

bool spmm_plane_plan(const WalkView &wk, long long n_out, int batch, const SpEpilogue &ep, bool force, PlaneLaunch &L)
{
    const bool fused = ep.bias != nullptr || ep.act != 0;
    if (wk.tab_dev == nullptr || wk.spans == nullptr || wk.lck != wk.k || wk.ngroups * wk.k > PLANE_TAB) return false;
    if (wk.period < PLANE_ROWS || (wk.k == 13 && fused)) return false;
    const PlaneSpans &spans = *wk.spans;
    if (spans.work == 0) return false;
    L.col_tiles = (batch + 63) / 64;
    int per_cu = 1;
    switch (wk.k) {
        case 5: per_cu = PlaneShape<5, 5>::per_cu(fused); break;
        case 7: per_cu = PlaneShape<7, 7>::per_cu(fused); break;
        case 8: per_cu = PlaneShape<8, 8>::per_cu(fused); break;
        case 9: per_cu = PlaneShape<9, 9>::per_cu(fused); break;
        case 11: per_cu = PlaneShape<11, 11>::per_cu(fused); break;
        case 13: per_cu = PlaneShape<13, 13>::per_cu(fused); break;
        default: return false;
    }
    L.tp = (wk.period + PLANE_ROWS - 1) / PLANE_ROWS;
    const int walk_len = (int)(n_out / wk.period);

    // A CU with fewer workgroups than it holds takes as long as a full one, but for 7 and 8 window rows, four workgroups of which
    // hold each other up: 7 x 7, 96 x 64, 4 maps to 6, batch 512 154 us with these shares, 187 with full rounds; 8 x 8, 128 x 128,
    // 3 to 4, batch 203 115 and 122.  Not so 5 x 5 windows, bound by memory and by the tiles' exits: 400 x 400, 4 to 4, batch 82
    // 456 and 441.  With three 9 x 9 ones it is level: 475 x 475, batch 213 196 and 194.
    static const double PART[] = {0, 1.9, 2.6, 3.1, 4};
    double shares[5];
    for (int n = 0; n <= per_cu; ++n) shares[n] = n == 0 ? 0 : per_cu == 4 && wk.k != 5 ? PART[n] : per_cu;
    const double over = plane_over(spans, walk_len, PLANE_XT, per_cu, shares, 0.9 * (wk.k - 1) * spans.most, L);
    // Taken by the steps, with the positions that only fill tiles up, over the work: up to these lines, for plain products,
    // with a bias and a sigmoid, and with a sample (on the vector unit, a few workgroups at a time).  Columns that only fill
    // tiles up are the tile-by-tile kernel's as well; where they are more than half of those that exist the kernel with rows
    // along the lanes does without them, and is ahead on a single column tile (and, with a sample, up to 76 columns of 15 chunks
    // and more: 0.72 - 0.95 of its rate, 310 x 310, 5 x 5, 3 maps to 4, batch 71 204 us here and 152).
    // Fitted to random products and layers of 1 to 16 maps, 28 to 520 wide, batch 24 to 1024, all kernels timed on each; of 10700
    // others within these lines the mean is 1.29 times the better other kernel's rate, 5 % are below 0.99, 3.6 % below 0.97 (2.0 %
    // without samples added to old values, whose exit was slower then, and of up to 76 columns; the least, 0.63, on 5 x 5 windows
    // of maps 32 wide).  A sample is taken at every exit, on the vector unit, and with one map there is
    // an exit for every block: 9 x 9 1.05 on average from 1.4 to 1.5, 0.98 from there to 1.8; with several 1.19 and 1.17 around 1.7;
    // 11 x 11 with several 1.22 from 1.4 to 1.5 and 1.18 to 1.6, with one 1.02 and 0.98.  7 x 7 with a sigmoid are at 1.1 - 1.6 up to
    // 1.8, but their steps alone are looked at beyond 1.5; plain ones at 1.11 on average from 2.0 to 2.1, 1.06 to 2.2, 0.99 from
    // there to 2.4, two fifths below 0.97 (56 x 152, batch 897 41 us here and 33).
    static const struct { int k; double plain, fused, sample, sample_one; } LINES[] = {{5, 1.8, 1.85, 1.75, 1.75},
                                                                                       {7, 2.2, 1.5, 1.55, 1.45},
                                                                                       {8, 2.5, 2.2, 1.8, 1.8},
                                                                                       {9, 2.2, 2.4, 1.7, 1.5},
                                                                                       {11, 2.0, 1.8, 1.55, 1.3}};
    double line = 0;
    for (const auto &l : LINES)
        if (l.k == wk.k) line = ep.act != 2 ? (fused ? l.fused : l.plain) : wk.ngroups > 1 ? l.sample : l.sample_one;
    if (wk.k == 7 && fused && ep.act != 2 && over <= 1.4) line = 1.8;
    if (L.col_tiles * 64 > batch + batch / 2) line = L.col_tiles > 1 ? std::min(line, wk.k >= 8 ? 1.65 : 1.45) : 0;
    if (ep.act == 2 && batch <= 76 && L.col_tiles == 2 && (long long)spans.work * wk.k >= 15LL * walk_len) line = 0;
    bool ahead = over * L.tp * PLANE_ROWS / wk.period <= line;
    // (13 x 13: of what spmm_split.hip's rule leaves; with one column tile the values are most of the traffic, and the
    // tile-by-tile kernel fetches them in pieces twice as long)
    if (wk.k == 13) ahead = L.col_tiles >= 2 && over <= 1.65;
    if (!force && !ahead) return false;
    plane_cut(spans, walk_len, 1, L);
    return true;
}

}  // namespace cuvdia
