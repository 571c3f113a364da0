// The product with a window table of 13 rows: fp32 products as bfloat16 ones on the matrix cores.
//
// A workgroup owns a strip of 16 output positions x of 64 batch columns and walks down the map rows of a segment, two at a time.
// Its 4 waves are 4 patches of 4 x 4 positions side by side; a patch needs the 16 x 16 dense rows around it (66 % of what is
// multiplied is in the table, the rest are zeros in the values' place), 2 x 16 a step, and lives 8 steps: at any time 4 of them,
// begun 2 steps apart, use the same dense rows, two pairs of 32 rows for v_mfma_f32_32x32x16_bf16.  Dense rows and values are
// split into three bfloat16 numbers (split.hpp), the rows on their way to LDS, the values on their way from it, between the
// products; six of the nine products of parts are made, and only the three of the rows' first parts where no row of a step
// has others (a binary layer's units).  What the split does not hold exactly (an infinity, a NaN, a number below 2^-110) is
// seen there, and the step that has it is multiplied in fp32 on the vector unit: 6 times as long where every step has some (4
// channels of 256 x 256 maps, batch 256, every eighth column around 2^-126: 4.4 ms), 1.06 where one number in 65536 is one.
//
// Two workgroups share a CU, so that one multiplies while the other waits: a step is a chain of waits (its values and rows from
// LDS, the first pair's split, two barriers) of which a wave alone hides nothing.  Tried: one workgroup of 128 columns with 512
// registers, its work interleaved by hand (720 - 770 us on the first case below), the values and not the rows in two buffers (780).
//
// Bound: that chain, 7500 - 8500 clocks a step where the products take 1600 (rows of bfloat16 numbers) or 3200 of a SIMD's.
// Measured against the kernels that served it: 4 channels of 256 x 256 maps, batch 256, binary rows 815 -> 667 us, uniform ones
// 752 (six products of parts instead of three); 200 x 200, 2 maps to 4, batch 256 556 -> 385 and 450; 448 x 448, 2 maps to 3,
// batch 64 560 -> 358 and 425.  (Parts cut off instead of rounded: 689, 407 and 367 with binary rows.)
// Windows of 11 rows use 47 % of a patch's products: level with the fp32 kernel.
//
// Accumulation order: of every 32 dense rows (16 of two map rows) the products of parts, smallest first, rounded as the matrix
// core does (split.hpp); these sums in fp32, map rows ascending.  Error against 64 bits (2-norm, relative), normal values, one
// map's sums of 1, 2, 3, 7, 19 and 169 uniform rows that are not 0: 3.3, 4.2, 4.4, 4.8, 5.7 and 6.4e-8, where a chain of fp32 FMAs
// has 2.6, 3.6, 4.0, 5.0, 8.0 and 22.6e-8; of binary rows 0.5, 3.6, 4.1, 4.7, 5.7 and 6.3e-8, the chain 0.5, 3.6, 4.0, 5.3, 8.0 and
// 23.5e-8.  (First parts' products as a sum of their own: 2.6, 3.4, 3.6, 4.1, 5.2 and 7.0e-8, and 2 - 5 % more time.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "device.hpp"
#include "kernels.hpp"
#include "split.hpp"

namespace cuvdia {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f16 __attribute__((ext_vector_type(16)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

constexpr int PS_WAVES = 4, PS_THREADS = 64 * PS_WAVES;

template <int LC, int K>
struct PsShape {
    static constexpr int NT = 2, COLS = 32 * NT;                    // batch columns, in tiles of 32
    static constexpr int PX = 4, PY = 4;                            // a patch: PX x PY output positions
    static_assert(PX + LC - 1 <= 16, "a patch's dense rows fit 16 positions");
    static constexpr int XS = PX * PS_WAVES;                        // positions of a workgroup's strip
    static constexpr int EVERY = PY / 2;                            // steps (of two map rows) from patch to patch
    static constexpr int NS = (PY + K) / 2;                         // steps that a patch lives
    static constexpr int NA = (NS + EVERY - 1) / EVERY;             // patches alive at once
    static_assert(NA == 4, "two pairs of patches");
    // Dense rows, twice: [part][map row][quad of positions][column], 8 bytes each, quads 40 bytes further for the banks
    static constexpr int NQ = (XS + 16 - PX) / 4;
    static constexpr int XQB = 8 * COLS + 40;
    static constexpr int XRB = NQ * XQB;
    static constexpr int XSB = 2 * XRB, X_BYTES = 3 * XSB;
    static constexpr int XLANES = 2 * NQ, XC = 64 / XLANES;         // a column's pieces of 4 positions; columns per wave and request
    static constexpr int PIECES = COLS / (XC * PS_WAVES);           // ... requests per wave
    static_assert(PIECES == 4 && XC * PS_WAVES * PIECES == COLS, "two requests for each pair of patches");
    // Values: [map row][window row][diagonal][position], fp32, zeros behind the last diagonal (a lane reads from diagonal -3 to 15)
    static constexpr int ROWB = 4 * XS, SLOTB = 16 * ROWB + 16, HALFB = K * SLOTB;
    static constexpr int A_BYTES = 2 * HALFB;
    static constexpr int SLOTS = (K + 1) / 2;                       // slots (of a map row and a window row) per wave
    static constexpr int ZERO = 2 * X_BYTES, ZERO_BYTES = 8 * ROWB; // what lanes without a window row read; in front of the first slot
    static constexpr int A0 = ZERO + ZERO_BYTES;
    static constexpr int NOWHERE = A0 + A_BYTES;                    // where the loads of a slot that there is not go
    static constexpr int TAB = NOWHERE + 1024;                      // (tables of up to 256 chunks come here)
    static constexpr int FLAGS = TAB + 1024;
    static constexpr int LDS = FLAGS + 2 * 4 * PS_WAVES;
    static constexpr int OPITCH = XS + 4;                           // a finished patch row's column, floats
    static_assert(PY * COLS * OPITCH * 4 <= X_BYTES, "a finished row of patches fits the dense rows' place");
    static constexpr int OQ = XS / 4, OIT = PY * COLS * OQ / PS_THREADS;           // its pieces of 4 positions
    static_assert(2 * LDS <= 160 * 1024, "two workgroups per CU");
};

// A pair of numbers on its way into three parts, a step at a time
struct PsPair {
    float x0, x1;
    unsigned p;
    __device__ __forceinline__ unsigned first(float v0, float v1)
    {
        x0 = v0; x1 = v1;
        return p = split_near(x0, x1);
    }
    __device__ __forceinline__ unsigned second(const SplitConst &k)
    {
        split_rest(p, k, x0, x1);
        return p = split_near(x0, x1);
    }
    __device__ __forceinline__ unsigned third(const SplitConst &k, unsigned &low)
    {
        split_rest(p, k, x0, x1);
        const unsigned last = split_last(x0, x1, low);
        asm volatile("" : "+v"(low));
        return last;
    }
};

template <int LC, int K, bool EP>
__global__ __launch_bounds__(PS_THREADS, 2) void spmm_split_kernel(
    const int *__restrict__ tab, int ngroups, int period, int s0, int astep4, int tp, int nseg, PlaneCuts cuts,
    const float *__restrict__ vals, const float *__restrict__ X, long long ldx, float *__restrict__ Y, long long ldy,
    int n_out, int n_in, int batch, float alpha, float beta, int col_tiles, unsigned a_bytes, SpEpilogue ep)
{
    using S = PsShape<LC, K>;
    constexpr int XT = 128 / S::XS, PX = S::PX, PY = S::PY, NT = S::NT, NA = S::NA, PIECES = S::PIECES;
    __shared__ __attribute__((aligned(16))) unsigned char lds[S::LDS];

    // (a unit -- a segment of XT neighbouring walks -- stays on one XCD, the last walks of a map row are units behind the full
    // ones: as in spmm_plane_kernel)
    const int xcd = blockIdx.x % 8, k8 = blockIdx.x / 8, xgroups = tp / XT, full_unit = XT * col_tiles;
    const int full_slots = (nseg * xgroups + 7) / 8 * full_unit;
    const bool full = k8 < full_slots;
    const int size = full ? full_unit : tp % XT * col_tiles, at_ = full ? k8 : k8 - full_slots;
    const int unit = at_ / size * 8 + xcd, within = at_ % size;
    const int xg = full ? unit / nseg : xgroups, seg = full ? unit - xg * nseg : unit;
    if (full ? xg >= xgroups : seg >= nseg) return;
    const int xt = xg * XT + within / col_tiles, coltile = within % col_tiles;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;
    const int xs = min(xt * S::XS, period - S::XS), skip = xt * S::XS - xs;       // (the last tile of a row is moved up)
    const int seg0 = cuts.at[seg], rows = cuts.at[seg + 1] - seg0;
    if (rows <= 0) return;
    const int row_first = xs + seg0 * period;
    const int col0 = coltile * S::COLS, cols = min(S::COLS, batch - col0);
    const float *const xbase = X + (long long)col0 * ldx;
    const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(xbase), 0, (unsigned)(((long long)(cols - 1) * ldx + n_in) * 4), 0x00020000);
    const __amdgpu_buffer_rsrc_t yrsrc = __builtin_amdgcn_make_buffer_rsrc(Y + (long long)col0 * ldy, 0, (unsigned)(((long long)(cols - 1) * ldy + n_out) * 4), 0x00020000);
    const sp_int4 arsrc = raw_rsrc(vals, a_bytes);
    const int amin = min(0, astep4 * (LC - 1));
    const unsigned lds0 = (unsigned)(unsigned long long)(__attribute__((address_space(3))) unsigned char *)&lds[0];

    // this lane's share of a block's dense rows: a piece of 4 positions of PIECES columns (the last
    // lanes do as the first ones do)
    const int x_i = lane < S::XC * S::XLANES ? lane : lane - S::XC * S::XLANES, x_lane_c = x_i / S::XLANES, x_lane_r = x_i % S::XLANES / S::NQ, x_lane_q = x_i % S::NQ;
    const int x_col = wave * S::XC + x_lane_c;
    const unsigned ldx4 = (unsigned)ldx * 4u, x_step = (unsigned)(S::XC * PS_WAVES) * ldx4;
    const unsigned x_off = (unsigned)x_col * ldx4 + (unsigned)(x_lane_r * period + 4 * x_lane_q) * 4u;
    unsigned char *const x_to = lds + x_lane_r * S::XRB + x_lane_q * S::XQB + x_col * 8;
    // ... and of a slot's values
    const int slot_r = wave & 1, slot_d = wave >> 1;               // this wave's slots: map row slot_r, window rows slot_d, + 2, ...
    const unsigned a_off = lane / 4 < LC ? (unsigned)(astep4 * (lane / 4) - amin) + 16u * (lane % 4) : OOB_OFFSET;
    // The tables: group i's first row in lane i; in LDS, byte offsets of every window row's values for the output row as far
    // above the segment's first as the window row lies down.
    const int group_lane = tab[min(lane, ngroups - 1)];          // (not more than 256 / K)
    int *const window_tab = reinterpret_cast<int *>(lds + S::TAB);
    for (int i = threadIdx.x; i < ngroups * K; i += PS_THREADS) window_tab[i] = tab[ngroups + i] + 4 * (row_first - i % K * period) + amin;
    for (int i = threadIdx.x; i < (S::NOWHERE - S::ZERO) / 4; i += PS_THREADS) *reinterpret_cast<float *>(lds + S::ZERO + 4 * i) = 0.f;
    auto block_row = [&](int u, int g) { return row_first + s0 + __builtin_amdgcn_readlane(group_lane, g) + 2 * u * period; };
    auto outside = [&](int x0) { return x0 + period + S::XS + LC - 1 <= 0 || x0 >= n_in; };
    auto inside = [&](int x0) { return x0 >= 0 && x0 + period + 4 * S::NQ <= n_in; };
    const SplitConst split_const;
    unsigned *const flags = reinterpret_cast<unsigned *>(lds + S::FLAGS);

    // The blocks (u, g) in order: one multiplied, the next one split, the one after that requested.  Of the groups only those
    // with rows anywhere in the segment are looked through at its steps (group rows ascend).
    const int patches = (rows + PY - 1) / PY, steps = (patches - 1) * S::EVERY + S::NS;
    int g0 = 0, g1 = ngroups;
    while (g0 < g1 && block_row(steps - 1, g0) + period + S::XS + LC - 1 <= 0) ++g0;
    while (g0 < g1 && block_row(0, g1 - 1) >= n_in) --g1;
    // (a look at 64 of them at once, one per lane)
    struct Block { int u, g, x0; };
    const int groups = g1 - g0, candidates = groups > 0 ? steps * groups : 0;
    int looked = 0, lane_u = 0, lane_g = 0, lane_x0 = 0;
    unsigned long long found = 0;
    auto look = [&]() __attribute__((always_inline)) {
        while (found == 0 && looked < candidates) {
            const int i = looked + here(lane);
            lane_u = i / groups;
            lane_g = g0 + i - lane_u * groups;
            lane_x0 = row_first + s0 + tab[min(lane_g, ngroups - 1)] + 2 * lane_u * period;
            found = __ballot(i < candidates && !outside(lane_x0));
            looked += 64;
        }
    };
    auto advance = [&]() __attribute__((always_inline)) -> Block {
        if (found == 0) look();
        const int i = found ? __builtin_ctzll(found) : 0;
        const int bu = found ? __builtin_amdgcn_readlane(lane_u, i) : steps;
        found &= found - 1;
        return Block{bu, __builtin_amdgcn_readlane(lane_g, i), __builtin_amdgcn_readlane(lane_x0, i)};
    };

    f4 xst[PIECES];                                  // the requested dense rows
    // the requests' scalars
    int window_lane = 0, values_up = 0, values_top = -1;
    unsigned x_soff = 0, x_at = 0;
    const unsigned values_to = lds0 + (unsigned)(S::A0 + slot_r * S::HALFB + slot_d * S::SLOTB);
    // (a block that crosses an end of the operand is staged by itself)
    auto request = [&](const Block &b) __attribute__((always_inline)) {
        x_at = x_off;
        x_soff = b.u < steps && inside(b.x0) ? (unsigned)b.x0 * 4u : 0u;
    };
    auto request_values_of = [&](const Block &b) __attribute__((always_inline)) {
        window_lane = window_tab[b.g * K + min(slot_d + 2 * lane, K - 1)];
        values_up = 4 * (2 * b.u + slot_r) * period;
        values_top = b.u < steps && inside(b.x0) ? 2 * b.u + slot_r - slot_d : -1;
    };
    auto request_x = [&](auto n_) __attribute__((always_inline)) {
        constexpr int n = decltype(n_)::value;
        xst[n] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(xrsrc, x_at, x_soff, 0));
        x_at += x_step;
        asm volatile("" : "+v"(x_at));
    };
    auto request_values = [&](auto i_) __attribute__((always_inline)) {
        constexpr int i = decltype(i_)::value;
        if constexpr (i < S::SLOTS) {
            // (a slot whose output row is not of the segment, or that there is not: zeros)
            const bool have = 2 * i + 1 < K || slot_d == 0, alive = have && (unsigned)(values_top - 2 * i) < (unsigned)rows;
            const int at = __builtin_amdgcn_readlane(window_lane, i) + values_up;
            lds_load_b128_scalar(arsrc, have ? values_to + 2 * i * S::SLOTB : lds0 + S::NOWHERE, alive ? a_off : OOB_OFFSET, (unsigned)at);
        }
    };

    f16 acc[NA / 2][NT];
#pragma unroll
    for (int a = 0; a < NA / 2; ++a)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[a][n][i] = 0.f;

    // As the matrix instruction has its operands: lane (m, kg) holds positions 8 kg .. 8 kg + 7 of a map row for output position
    // (mx, my) of patch mp of a pair, or for column m; of the sums, elements 4 i .. 4 i + 3 for positions 0 .. 3 of patch row
    // 2 (i % 2) + kg of patch i / 2, column m
    const int m32 = lane % 32, kg = lane / 32, mx = m32 % PX, my = m32 / PX % PY, mp = m32 / 16;
    const int a_lane = S::A0 - my * S::SLOTB + (8 * kg - mx) * S::ROWB + 16 * wave + 4 * mx;
    const int x_lane = (wave * PX / 4 + 2 * kg) * S::XQB + m32 * 8;
    // the step (0 .. PERIOD - 1; NS and above: none) that patch slot a is in at step u
    constexpr int PERIOD = NA * S::EVERY;
    auto step_of = [&](int a, int u) { const int t = (u - a * S::EVERY) % PERIOD; return t < 0 ? t + PERIOD : t; };

    u4 af[NA / 2][2][3];
    // the raw values of a pair's map row r; a pair of them
    const unsigned char *a_from = lds;
    auto values_at = [&](auto a_, int r, int u) __attribute__((always_inline)) {
        constexpr int a = decltype(a_)::value;
        const int t0 = step_of(2 * a, u), t1 = step_of(2 * a + 1, u), d = 2 * (mp ? t1 : t0) + r;
        a_from = lds + ((unsigned)(d - my) < (unsigned)K ? a_lane + r * S::HALFB + d * S::SLOTB : S::ZERO);
    };
    auto values_of = [&](auto j_, float (&v)[2]) __attribute__((always_inline)) {
        constexpr int j = decltype(j_)::value;
#pragma unroll
        for (int i = 0; i < 2; ++i) v[i] = *reinterpret_cast<const float *>(a_from + (2 * j + i) * S::ROWB);
    };
    auto barrier = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    // A row of patches that is done leaves through LDS, in the place of dense rows that are done with, so that a column's
    // positions are written together.
    auto finish = [&](int y0, int leaving, int buf) __attribute__((always_inline)) {
        float *const out = reinterpret_cast<float *>(lds + buf * S::X_BYTES);
        static_for<0, NA>([&](auto a_) __attribute__((always_inline)) {
            constexpr int a = decltype(a_)::value;
            if (leaving != a) return;
            asm volatile("" :: "n"(a));              // (four ways through, not one with an index)
            float *const to = out + (kg * S::COLS + m32) * S::OPITCH + wave * PX;
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                asm volatile("" : "+v"(acc[a / 2][n]));
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    f4 s;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        s[i] = acc[a / 2][n][8 * (a % 2) + 4 * h + i];
                        acc[a / 2][n][8 * (a % 2) + 4 * h + i] = 0.f;
                    }
                    *reinterpret_cast<f4 *>(to + (2 * h * S::COLS + 32 * n) * S::OPITCH) = s;
                }
                asm volatile("" : "+v"(acc[a / 2][n]));
            }
        });
        barrier();
        const int thread = here(threadIdx.x), q = thread % S::OQ, x = 4 * q, c = thread / S::OQ;
        constexpr int CSTEP = PS_THREADS / S::OQ, PER_ROW = S::COLS / CSTEP;
        if (EP && ep.act == 2) {
            // sampled: a lane takes a position and 4 columns, a block of the generator
            static_assert(S::COLS / 4 * S::XS == PS_THREADS, "a patch row at a time");
            const int sx = thread % S::XS, c0 = thread / S::XS * 4;
#pragma nounroll
            for (int y = 0; y < PY; ++y) {
                if (sx < skip || y0 + y >= rows || c0 >= cols) continue;
                const int row = row_first + (y0 + y) * period + sx;
                const float bias = ep.bias ? ep.bias[row] : 0.f;
                const SpRand4 w = sp_philox((unsigned)row, (unsigned)(col0 + c0) / 4u, ep.seed_lo, ep.seed_hi);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (c0 + i >= cols) continue;
                    float *const p = Y + (long long)(col0 + c0 + i) * ldy + row;
                    const float sum = out[(y * S::COLS + c0 + i) * S::OPITCH + sx];
                    *p = sp_finish(beta == 0.f ? alpha * sum : beta * *p + alpha * sum, bias, 2, w.w[i]);
                }
            }
            barrier();
            return;
        }
        f4 s[S::OIT];
        unsigned at[S::OIT];
#pragma unroll
        for (int it = 0; it < S::OIT; ++it) {
            const int col = c + it % PER_ROW * CSTEP;
            s[it] = *reinterpret_cast<const f4 *>(out + (it / PER_ROW * S::COLS + col) * S::OPITCH + x);
            at[it] = col < cols && y0 + it / PER_ROW < rows ? (unsigned)col * ((unsigned)ldy * 4u) + 4u * x : OOB_OFFSET;
        }
        const unsigned first = (unsigned)(row_first + y0 * period) * 4u, step = (unsigned)period * 4u;
        if (beta == 0.f) {
#pragma unroll
            for (int it = 0; it < S::OIT; ++it) s[it] = f4{alpha * s[it][0], alpha * s[it][1], alpha * s[it][2], alpha * s[it][3]};
        } else {
            f4 old[S::OIT];
#pragma unroll
            for (int it = 0; it < S::OIT; ++it) old[it] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(yrsrc, at[it], first + it / PER_ROW * step, 0));
#pragma unroll
            for (int it = 0; it < S::OIT; ++it)
#pragma unroll
                for (int i = 0; i < 4; ++i) s[it][i] = beta * old[it][i] + alpha * s[it][i];
        }
        if (EP) {
#pragma unroll
            for (int it = 0; it < S::OIT; ++it) {
                f4 bias = {0.f, 0.f, 0.f, 0.f};
                if (ep.bias && at[it] != OOB_OFFSET) bias = *reinterpret_cast<const f4u *>(ep.bias + row_first + (y0 + it / PER_ROW) * period + x);
#pragma unroll
                for (int i = 0; i < 4; ++i) s[it][i] = sp_finish(s[it][i], bias[i], ep.act);
            }
        }
        if (skip == 0) {
#pragma unroll
            for (int it = 0; it < S::OIT; ++it) buffer_store4<0>(s[it], yrsrc, at[it], first + it / PER_ROW * step);
        } else {
#pragma unroll
            for (int it = 0; it < S::OIT; ++it)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float e = s[it][i];
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, e), yrsrc, x + i >= skip ? at[it] + 4u * i : OOB_OFFSET, first + it / PER_ROW * step, 0);
                }
        }
        barrier();
    };

    // The first block's rows and values come by stage(), the next one's rows are on their way.
    Block cur = advance(), next = advance(), third = advance();
    __syncthreads();                                 // (the tables, the zeros)
    request(next);
    static_for<0, PIECES>([&](auto n_) __attribute__((always_inline)) { request_x(n_); });


    // A block's flags: 1: not all of its dense rows are held exactly; 2: not all are bfloat16 numbers
    auto raise = [&](int buf, unsigned low, unsigned more) __attribute__((always_inline)) {
        const bool bad = split_inexact<PIECES / 2>(low, [&](int i) __attribute__((always_inline)) {
            const unsigned char *const at = x_to + buf * S::X_BYTES + 2 * S::XSB + 2 * i * (8 * S::XC * PS_WAVES);
            const u2 p0 = *reinterpret_cast<const u2 *>(at), p1 = *reinterpret_cast<const u2 *>(at + 8 * S::XC * PS_WAVES);
            return u4{p0[0], p0[1], p1[0], p1[1]};
        });
        const unsigned f = (bad ? 1u : 0u) | (__any(more != 0u) ? 2u : 0u);
        if (lane == 0) flags[4 * buf + wave] = f;
    };
    // The values of a block that crosses an end of the operand, and such a block's or the first one's dense rows: element by
    // element, what does not exist is 0.
    auto stage = [&](int buf) __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        barrier();                                   // (what was requested has come)
        const int l = here(lane), li = l < S::XC * S::XLANES ? l : l - S::XC * S::XLANES, r = li % S::XLANES / S::NQ, q = li % S::NQ, c0 = wave * S::XC + li / S::XLANES;
        unsigned low = 0, more = 0;
#pragma nounroll
        for (int it = 0; it < PIECES; ++it) {
            const int c = c0 + it * S::XC * PS_WAVES;
            f4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int xr = cur.x0 + r * period + 4 * q + e;
                x[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrsrc, c < cols && xr >= 0 && xr < n_in ? (unsigned)c * ldx4 + 4u * xr : OOB_OFFSET, 0, 0));
            }
            u2 p[3];
            low |= split4(x, split_const, p);
            more |= p[1][0] | p[1][1];
#pragma unroll
            for (int s = 0; s < 3; ++s) *reinterpret_cast<u2 *>(lds + buf * S::X_BYTES + s * S::XSB + r * S::XRB + q * S::XQB + c * 8) = p[s];
        }
#pragma nounroll
        for (int i = 0; i < S::SLOTS; ++i) {
            const int d = slot_d + 2 * i, m = 2 * cur.u + slot_r - d;
            if (d >= K || l / 4 >= LC) continue;
            const int at = window_tab[cur.g * K + d] + 4 * (2 * cur.u + slot_r) * period - amin;
            f4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int x = 4 * (l % 4) + e, xr = cur.x0 + slot_r * period + x + l / 4;
                v[e] = (unsigned)m < (unsigned)rows && xr >= 0 && xr < n_in ? vals[(long long)(at / 4) + (long long)(astep4 / 4) * (l / 4) + x] : 0.f;
            }
            *reinterpret_cast<f4 *>(lds + (S::A0 + slot_r * S::HALFB + d * S::SLOTB) + 16 * l) = v;
        }
        raise(buf, low, more);
        barrier();
    };
    // An operand that the split does not hold exactly -- an infinity, a NaN, a number next to the smallest ones --: the
    // block's products for a pair of patches one by one, those that the table has and no others; then zeros in its place.
    // A lane takes a column's dense rows 4 at a time, for all the patch rows that use them.
    auto exact = [&](auto p_) __attribute__((always_inline)) {
        constexpr int p = decltype(p_)::value;
        const int l = here(lane), sx = wave * PX;            // this lane's sums: positions sx .. sx + 3 of patch rows l / 32, + 2
        static_for<0, NT>([&](auto n_) __attribute__((always_inline)) {
            constexpr int n = decltype(n_)::value;
            const unsigned col = (unsigned)min(32 * n + l % 32, cols - 1) * ldx4;
            auto piece = [&](int xr) __attribute__((always_inline)) {
                if (xr >= 0 && xr + 4 <= n_in) return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(xrsrc, col, 4 * xr, 0));
                f4 x;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    x[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrsrc, xr + e >= 0 && xr + e < n_in ? col + 4u * (xr + e) : OOB_OFFSET, 0, 0));
                return x;
            };
#pragma nounroll
            for (int r = 0; r < 2; ++r) {
                const int x0 = cur.x0 + r * period + sx;
                f4 x = piece(x0);
#pragma nounroll
                for (int q = 0; q < LC; q += 4) {
                    const f4 more = piece(x0 + min(q + 4, LC - 1));
                    const float xs[7] = {x[0], x[1], x[2], x[3], more[0], more[1], more[2]};
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        const int t = step_of(2 * p + i4 / 2, cur.u), y0 = 2 * (cur.u - t), sy = 2 * (i4 % 2) + l / 32, d = 2 * t + r - sy;
                        if (t >= S::NS || y0 < 0 || d < 0 || d >= K || y0 + sy >= rows) continue;
                        const unsigned char *const from = lds + S::A0 + r * S::HALFB + d * S::SLOTB + 4 * sx + q * S::ROWB;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            if (q + e >= LC) continue;
                            const f4 w = *reinterpret_cast<const f4 *>(from + e * S::ROWB);
#pragma unroll
                            for (int i = 0; i < 4; ++i) acc[p][n][4 * i4 + i] = fmaf(w[i], xs[e + i], acc[p][n][4 * i4 + i]);
                        }
                    }
                    x = more;
                }
            }
        });
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int s = 0; s < 3; ++s) af[p][r][s] = u4{0u, 0u, 0u, 0u};
    };

    int buf = 0, u = -1;
    bool staged = false;
    for (;;) {
        // the patches that end before this step
        while (u < cur.u) {
            const int first = u - (S::NS - 1);
            if (first >= 0 && first % S::EVERY == 0) finish(first / S::EVERY * PY, first / S::EVERY % NA, buf ^ 1);
            ++u;
        }
        if (u >= steps) break;
        if (!staged || !inside(cur.x0)) stage(buf);
        staged = true;
        const unsigned char *const x_from = lds + x_lane + buf * S::X_BYTES;
        unsigned char *const x_next = x_to + (buf ^ 1) * S::X_BYTES;
        u4 xf[NT][2][3];
        const unsigned x_flag = flags[4 * buf + lane % PS_WAVES];
        const bool x_bad = __any(x_flag & 1u), x_more = __any(x_flag & 2u);
        unsigned low_x = 0, more_x = 0;
        float v[8][2];
        if (x_bad) {
            // (no product of theirs comes from the matrix cores)
            exact(std::integral_constant<int, 0>{});
            exact(std::integral_constant<int, 1>{});
            barrier();                               // (everybody has read the values)
            for (int i = here(threadIdx.x); i < S::X_BYTES / 8; i += PS_THREADS) *reinterpret_cast<u2 *>(lds + buf * S::X_BYTES + 8 * i) = u2{0u, 0u};
            for (int i = here(threadIdx.x); i < S::A_BYTES / 8; i += PS_THREADS) *reinterpret_cast<u2 *>(lds + S::A0 + 8 * i) = u2{0u, 0u};
            barrier();
        }
        // the first pair's values
        {
            unsigned low = 0;
            static_for<0, 2>([&](auto r_) __attribute__((always_inline)) {
                constexpr int r = decltype(r_)::value;
                values_at(std::integral_constant<int, 0>{}, r, u);
                static_for<0, 4>([&](auto j_) __attribute__((always_inline)) { values_of(j_, v[4 * r + decltype(j_)::value]); });
            });
            auto rows_of = [&](auto s_) __attribute__((always_inline)) {
                constexpr int s = decltype(s_)::value;
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        const unsigned char *const from = x_from + s * S::XSB + r * S::XRB + n * 256;
                        const u2 q0 = *reinterpret_cast<const u2 *>(from), q1 = *reinterpret_cast<const u2 *>(from + S::XQB);
                        xf[n][r][s] = u4{q0[0], q0[1], q1[0], q1[1]};
                        __builtin_amdgcn_sched_barrier(0);       // (both quads by one instruction)
                    }
            };
            if (x_more) {                            // (read in any case: 686 us for 667 on the large layer's binary rows)
                rows_of(std::integral_constant<int, 2>{});
                rows_of(std::integral_constant<int, 1>{});
            }
            rows_of(std::integral_constant<int, 0>{});
            static_for<0, 8>([&](auto j_) __attribute__((always_inline)) {
                constexpr int j = decltype(j_)::value;
                unsigned p0, p1, p2;
                split2(v[j][0], v[j][1], split_const, p0, p1, p2, low);
                af[0][j / 4][0][j % 4] = p0; af[0][j / 4][1][j % 4] = p1; af[0][j / 4][2][j % 4] = p2;
            });
            if (split_inexact<2>(low, [&](int i) __attribute__((always_inline)) { return af[0][i][2]; })) exact(std::integral_constant<int, 0>{});
        }
        request(third);
        static_for<0, 2>([&](auto pass_) __attribute__((always_inline)) {
            constexpr int pass = decltype(pass_)::value;
            unsigned low = 0;
            if constexpr (pass == 0) {
                values_at(std::integral_constant<int, 1>{}, 0, u);
                values_of(std::integral_constant<int, 0>{}, v[0]);
                values_of(std::integral_constant<int, 1>{}, v[1]);
            }
            f16 t[NT];
            u2 xq[3];
            PsPair ap, aq, xp;
            __builtin_amdgcn_sched_barrier(0);
            auto product = [&](auto i_, auto pa_, auto pb_, auto first_) __attribute__((always_inline)) {
                constexpr int r = decltype(i_)::value / 2 % 2, n = decltype(i_)::value % 2, pa = decltype(pa_)::value, pb = decltype(pb_)::value;
                t[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(split_b8, af[pass][r][pa]), __builtin_bit_cast(split_b8, xf[n][r][pb]), decltype(first_)::value ? f16{} : t[n], 0, 0, 0);
            };
            // (dense rows of bfloat16 numbers, as a layer's binary units are, have no other parts to multiply; the first two products
            // of the others are in either way, so that no zeros are written for them to add to)
            constexpr std::integral_constant<int, 2> last_part{};
            if (x_more) {
                constexpr int PA[3] = {0, 1, 0}, PB[3] = {2, 1, 1};
                static_for<0, 12>([&](auto i_) __attribute__((always_inline)) {
                    constexpr int p = decltype(i_)::value / 4;
                    product(i_, std::integral_constant<int, PA[p]>{}, std::integral_constant<int, PB[p]>{}, std::bool_constant<(decltype(i_)::value < 2)>{});
                    __builtin_amdgcn_sched_barrier(0);
                });
                static_for<0, 2>([&](auto i_) __attribute__((always_inline)) { product(i_, last_part, std::integral_constant<int, 0>{}, std::false_type{}); });
            } else {
                static_for<0, 2>([&](auto i_) __attribute__((always_inline)) { product(i_, last_part, std::integral_constant<int, 0>{}, std::true_type{}); });
            }
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, 12>([&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value;
                if constexpr (i >= 2) product(i_, std::integral_constant<int, 2 - i / 4>{}, std::integral_constant<int, 0>{}, std::false_type{});
                // beside the products: in the first pass two pairs of the second pair's values per 3; a pair of the next dense rows per 3
                if constexpr (pass == 0) {
                    constexpr int j = 2 * (i / 3), ar = j / 4, aj = j % 4;
                    if constexpr (i % 3 == 0) {
                        af[1][ar][0][aj] = ap.first(v[j][0], v[j][1]);
                        af[1][ar][0][aj + 1] = aq.first(v[j + 1][0], v[j + 1][1]);
                    }
                    if constexpr (i % 3 == 1) {
                        af[1][ar][1][aj] = ap.second(split_const);
                        af[1][ar][1][aj + 1] = aq.second(split_const);
                        if constexpr (j == 2) values_at(std::integral_constant<int, 1>{}, 1, u);
                        if constexpr (j < 6) {
                            values_of(std::integral_constant<int, (j + 2) % 4>{}, v[j + 2]);
                            values_of(std::integral_constant<int, (j + 3) % 4>{}, v[j + 3]);
                        }
                    }
                    if constexpr (i % 3 == 2) {
                        af[1][ar][2][aj] = ap.third(split_const, low);
                        af[1][ar][2][aj + 1] = aq.third(split_const, low);
                    }
                }
                constexpr int xj = i / 3, piece = 2 * pass + xj / 2, xh = xj % 2;
                if constexpr (i % 3 == 0) xq[0][xh] = xp.first(xst[piece][2 * xh], xst[piece][2 * xh + 1]);
                if constexpr (i % 3 == 1) xq[1][xh] = xp.second(split_const);
                if constexpr (i % 3 == 2) xq[2][xh] = xp.third(split_const, low_x);
                if constexpr (i % 3 == 2 && xh == 1) {
                    more_x |= xq[1][0] | xq[1][1];
#pragma unroll
                    for (int s = 0; s < 3; ++s) *reinterpret_cast<u2 *>(x_next + piece * (8 * S::XC * PS_WAVES) + s * S::XSB) = xq[s];
                    request_x(std::integral_constant<int, piece>{});
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (pass == 0) {
                if (split_inexact<2>(low, [&](int i) __attribute__((always_inline)) { return af[1][i][2]; })) exact(std::integral_constant<int, 1>{});
            }
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                acc[pass][n] += t[n];
                asm volatile("" : "+v"(acc[pass][n]));
            }
            if constexpr (pass == 0) {
                asm volatile("" : "+v"(xst[2]), "+v"(xst[3]));       // (come before the values are asked for)
                request_values_of(next);
                barrier();                           // (nobody reads the values any more)
                static_for<0, S::SLOTS>([&](auto i_) __attribute__((always_inline)) { request_values(i_); });
            }
        });
        raise(buf ^ 1, low_x, more_x);
        cur = next;
        next = third;
        third = advance();
        // (the values have come: of the requests at most the dense rows' last 2 are still out)
        asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
        barrier();
        buf ^= 1;
    }
}

template <int LC, int K>
hipError_t ps_launch_one(const PlaneLaunch &L)
{
    const bool fused = L.ep.bias != nullptr || L.ep.act != 0;
    constexpr int XT = 128 / PsShape<LC, K>::XS;
    const long long full = (long long)L.nseg * (L.tp / XT), part = L.nseg;       // units (the kernel's head)
    const unsigned grid = (unsigned)(((full + 7) / 8 * XT + (part + 7) / 8 * (L.tp % XT)) * 8 * L.col_tiles);
    note_kernel("spmm_split_kernel<%d, %d, %s>", LC, K, fused ? "true" : "false");
    auto go = [&](auto kernel) {
        launch_kernel(kernel, dim3(grid), dim3(PS_THREADS), 0, L.stream, L.tab, L.ngroups, L.period, L.s0, L.astep4, L.tp,
                      L.nseg, L.cuts, L.vals, L.B, L.ldb, L.dst, L.ldd, L.n_out, L.n_in, L.batch, L.alpha, L.beta,
                      L.col_tiles, L.a_bytes, L.ep);
    };
    if (fused) go(spmm_split_kernel<LC, K, true>);
    else go(spmm_split_kernel<LC, K, false>);
    return hipGetLastError();
}

}  // namespace

hipError_t spmm_split_launch(const PlaneLaunch &L) { return ps_launch_one<13, 13>(L); }

bool spmm_split_plan(const WalkView &wk, long long n_out, int batch, bool force, bool walks, PlaneLaunch &L)
{
    using S = PsShape<13, 13>;
    if (wk.tab_dev == nullptr || wk.spans == nullptr || wk.k != 13 || wk.lck != 13 || wk.ngroups * 13 > 256 || wk.period < 32) return false;
    const PlaneSpans &spans = *wk.spans;
    if (spans.work == 0) return false;
    L.col_tiles = (batch + S::COLS - 1) / S::COLS;
    L.tp = (wk.period + S::XS - 1) / S::XS;
    // (a segment that has the end of a map in it walks both maps' ends)
    const double walk_ends = 0.9 * (wk.k - 1) * spans.most * (spans.groups.size() > 1 ? 2 : 1);
    const int walk_len = (int)(n_out / wk.period);
    const double shares[] = {0, 2, 2};               // (a workgroup alone on its CU takes as long as two)
    const double over = plane_over(spans, walk_len, 128 / S::XS, 2, shares, walk_ends, L);
    // Taken where the rounds' steps, with the columns and positions that only fill tiles up, come to at most 2.1 times the
    // segments' own where the tile-by-tile kernel would run, 1.65 times where the plane's walk would.  Measured on 210 random
    // products of 13 x 13 windows, 1 to 5 maps, 40 to 640 wide, batch 24 to 640, a third of them with bias and sigmoid: 79 are
    // taken, at 0.90 - 4.7 times the rate of the kernels that served them (one below 0.97; median 1.25, with bias and sigmoid
    // 1.42; samples 0.98 - 1.28).  Forced on 111 others: up to these lines 4 % below 0.97 in place of the tile-by-tile kernel, beyond
    // them more than a third.  The line of 1.65 is a cautious one: the plane's walk keeps 20 of the 210, of which 13 would be
    // up to 1.6 times as fast here and 4 at 0.91 - 0.96.
    const double padded = over * L.col_tiles * S::COLS / batch * L.tp * S::XS / wk.period;
    if (!force && padded > (walks ? 1.65 : 2.1)) return false;
    plane_cut(spans, walk_len, S::PY, L);
    return true;
}

}  // namespace cuvdia
