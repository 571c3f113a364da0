// The dense x dense^T projection of square windows of 13 rows: fp32 products as bfloat16 ones on the matrix cores.
//
//   C_d[i] = beta * C_d[i] + alpha * sum_c A[i, c] * B[i + k_d, c]
//
// A tile is 32 map positions of 8 map rows.  v_mfma_f32_16x16x32_bf16 multiplies a patch of 4 x 4 positions of A with a patch of
// 4 x 4 of B; a patch of A meets 4 x 4 patches of B, and 66 % (13 * 13 of 16 * 16) of what they make are slots of the window.  The
// others are sums of their own that nobody reads, so no value of theirs, infinite or not, reaches a slot.  Every number is split
// into three bfloat16 ones where it is staged (split.hpp), six of their nine products are made: 16 columns of two pairs of parts
// fill an instruction's 32, three instructions are 16 columns.  What the split does not hold exactly (an infinity, a NaN, a
// number below 2^-110) is seen there, and the stage that has it is multiplied in fp32 from memory, behind the other stages of its 1024
// columns: 4.0 ms where every stage has some, 0.99 where one of 16 has (4 maps of 256 x 256 to 4, batch 256; 0.82 without).
//
// Per stage of 16 columns the loads of the next one are on their way to registers; the split, transposed, goes to LDS; a wave
// works two patches of A.  The products of a stage are one stretch of code without a branch, a patch's sums are added while the next
// one's products are made.  (With a branch per patch of B to the fp32 way every sum was waited for, 4800 - 5100 clocks a stage.)
//
// Bound: the loads.  A stage's products take 3300 clocks of a wave that is first on its SIMD, 4500 of the other, the split and its way
// to LDS 2500; with all CUs at work the loads have come 5000 after the products begin, 80 KB in segments of 176 bytes (tiles 16
// positions wide: 112 bytes, and half as long again), a third of them from beyond the L2: 8400 a stage, 9300 before the branches went.
// (The clock falls with every saving, 2.02 -> 1.92 GHz.)  Measured against the kernel with a wave per window row, in brackets with the
// branches: 4 channels of 256 x 256 maps, batch 256 981 -> 815 us (838; 69 TFLOP/s); 416 x 416, batch 357 421 -> 314 (323); 200 x 200, 2
// maps to 2, batch 256 357 -> 211 (228); 272 x 272 to 2, batch 388 413 -> 311 (329); 192 x 192 to 8, batch 160 266 (274).  (With the branches and
// parts cut off instead of rounded: 825, 332, 228 and 331 on the first four.)  Windows of 7 to 11 rows have fewer products for the same
// loads and fewer of them are slots: 0.5 - 0.95 times the kernels that serve them.
//
// Accumulation order: of every 16 columns the six products of all columns, smallest first, rounded as the matrix core does
// (split.hpp); these sums in fp32, within each 1024 columns those of the stages that the split holds, ascending, then the others',
// each a chain of fp32 FMAs, ascending.  Error against 64 bits (2-norm, relative; uniform operands in -1 .. 1) at
// batch 37, 128, 256 and 2048: 0.5, 0.7, 0.9 and 2.2e-7, where a chain of fp32 FMAs has 1.1, 2.0, 2.9 and 8.1e-7.  Sums of 1, 2,
// 4, 8 and 16 products spread over 128 columns: 3.1, 4.1, 5.1, 5.9 and 6.6e-8, the chain 2.5, 3.1, 4.0, 5.4 and 7.4e-8: a sum of
// few is rounded where the others' meet the first parts' products and again where the blocks of 16 columns meet.  (First parts'
// products as a fourth instruction, a sum of their own: 2.5, 3.4, 4.4, 5.4 and 6.2e-8, and 838 -> 918 us on the first case above.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "device.hpp"
#include "kernels.hpp"
#include "split.hpp"

namespace cuvdia {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

constexpr int DS_XT = 32, DS_YT = 8;                 // a tile: map positions, map rows
constexpr int DS_WAVES = 8, DS_THREADS = 64 * DS_WAVES;      // two patches of 4 x 4 each, one below the other
constexpr int DS_COLS = 16;                          // batch columns per stage
constexpr int DS_MAX_GROUPS = 32;

// The tiles that have slots: those of group g's map-row blocks first_block[g] ..., first_tile[g] tiles before them.
struct DsTiles {
    int first_tile[DS_MAX_GROUPS + 1], first_block[DS_MAX_GROUPS];
};

template <int LC, int K>
struct DsShape {
    static constexpr int BX = (LC + 3 + 3) / 4, BY = (K + 3 + 3) / 4;      // patches of B that a patch of A meets
    static constexpr int NBX = DS_XT / 4 + BX - 1, NBY = DS_YT / 4 + BY - 1;       // ... and a tile
    static constexpr int PART = 512, PATCH = 3 * PART + 16;      // bytes: [part][8 columns][position], 16 each; the odd 16 spread the writes over the banks
    static constexpr int A_PATCHES = DS_XT / 4 * DS_YT / 4;      // behind B's
    // Staging: 4 rows x 8 columns a thread (a "task"), from one operand per wave: B's, then A's first 8 columns.  A's second 8 come
    // by way of LDS, a column per wave.
    static constexpr int KQ = DS_COLS / 8, QUADS = 4 * NBY * NBX, A_QUADS = DS_YT * DS_XT / 4, B_WAVES = DS_WAVES - 1;
    static_assert(KQ == 2 && KQ * QUADS <= 64 * B_WAVES && A_QUADS == 64, "B on all waves but one, A's quads on that one");
    static constexpr int LOADS = 9;                  // per stage and wave
    static constexpr int PITCH = DS_XT * DS_YT / 2 + 1;  // of a slot's results for half a tile on their way out, floats
    static constexpr int STAGE = (NBX * NBY + A_PATCHES) * PATCH, OUT = LC * K * PITCH * 4;
    static constexpr int RAW = STAGE;                // A's second 8 columns as they are: [column][quad]
    static constexpr int STAGED = STAGE + 8 * 1024;
    static constexpr int FLAGS = ((STAGED > OUT ? STAGED : OUT) + 15) / 16 * 16;
    static constexpr int TAB = FLAGS + 4 * DS_WAVES;     // of the group's window rows
    static constexpr int LDS = TAB + 4 * K;
    static_assert(LDS <= 160 * 1024, "a workgroup per CU");
};

template <int LC, int K>
__global__ __launch_bounds__(DS_THREADS, 2) void dd2dia_split_kernel(
    const int *__restrict__ tab, int ngroups, int period, int s0, int astep, float *__restrict__ C,
    const float *__restrict__ A, long long lda, const float *__restrict__ B, long long ldb, int h, int w, int batch,
    float alpha, float beta, unsigned a_bytes, unsigned b_bytes, unsigned c_bytes, int txn, DsTiles tiles)
{
    using S = DsShape<LC, K>;
    __shared__ __attribute__((aligned(16))) unsigned char lds[S::LDS];
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);

    // each XCD takes a contiguous stretch of the tiles: neighbours share rows of A and B
    const int ntiles = tiles.first_tile[ngroups], each = ntiles / 8, more = ntiles % 8, xcd = blockIdx.x % 8;
    if ((int)blockIdx.x >= ntiles) return;                       // (5000 of 8192 on the large layer: no difference in time)
    const int tile = xcd * each + min(xcd, more) + blockIdx.x / 8;
    int g = 0;
    while (g + 1 < ngroups && tile >= tiles.first_tile[g + 1]) ++g;
    const int in_group = tile - tiles.first_tile[g], ty = tiles.first_block[g] + in_group / txn, tx = in_group % txn;
    const int i_tile = ty * DS_YT * period + tx * DS_XT;         // the tile's first row of A
    const int s_g = s0 + tab[g];
    const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(A), 0, a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), 0, b_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t cr = __builtin_amdgcn_make_buffer_rsrc(C, 0, c_bytes, 0x00020000);
    const unsigned lda4 = (unsigned)lda * 4u, ldb4 = (unsigned)ldb * 4u;

    // Columns past the batch lie out of the resources' range (0).  Rows outside the operands are not asked for, and are 0 as
    // well: what memory holds there must not decide whether the split holds a stage's numbers.

    // This thread's task of a stage: the first of its 4 rows, its 8 columns, the place of the first row's.
    const int thread = threadIdx.x;
    const bool of_a = wave >= S::B_WAVES;
    const int task = of_a ? thread - 64 * S::B_WAVES : thread, quads = of_a ? S::A_QUADS : S::QUADS, wide = of_a ? DS_XT / 4 : S::NBX;
    const int kq = task / quads, quad_y = (task - kq * quads) / wide, quad_x = (task - kq * quads) % wide;
    const bool have = kq < (of_a ? 1 : S::KQ);
    const __amdgpu_buffer_rsrc_t rsrc = of_a ? ar : br;
    const unsigned ld4 = of_a ? lda4 : ldb4;
    // A piece that reaches over an end of B is fetched from the last place inside and moved when it is split (the hardware would
    // answer it with zeros as a whole): first row wanted - first row fetched.
    const int row_wanted = (of_a ? i_tile : i_tile + s_g) + quad_y * period + 4 * quad_x;
    const int row = of_a ? row_wanted : row_wanted < 0 && row_wanted > -4 ? 0 : row_wanted > w - 4 && row_wanted < w ? w - 4 : row_wanted;
    const int moved = row_wanted - row;
    const bool inside = have && row_wanted > -4 && row_wanted < (of_a ? h : w);
    const unsigned off = (unsigned)row * 4u + (unsigned)(8 * kq) * ld4;
    unsigned char *const to = lds + ((of_a ? S::NBX * S::NBY : 0) + quad_y / 4 * wide + quad_x) * S::PATCH + kq * 256 + quad_y % 4 * 64;
    // ... and of A's second 8 columns: a quad of the wave's column on its way to LDS, half a task from there
    const sp_int4 a_raw = raw_rsrc(A, a_bytes);
    const int raw_row = i_tile + lane / (DS_XT / 4) * period + 4 * (lane % (DS_XT / 4));
    const unsigned raw_off = (unsigned)raw_row * 4u + (unsigned)(8 + wave) * lda4;
    const unsigned raw_to = (unsigned)(unsigned long long)(__attribute__((address_space(3))) unsigned char *)&lds[S::RAW] + 1024u * wave;
    // (a tile whose rows of B cross an end of the operand)
    const int b_first = i_tile + s_g, b_last = b_first + (4 * S::NBY - 1) * period + 4 * S::NBX - 1;
    const bool ends = b_first < 0 || b_last >= w;
    // As the matrix instruction has its operands: lane (m, kg) holds 8 columns of position m of a patch, of one part for kg < 2
    // and of another for the other half.  A wave's two patches of A lie one below the other.
    const int m16 = lane % 16, kg = lane / 16, at = kg % 2 * 256 + m16 * 16;
    const unsigned char *const b21 = lds + wave * S::PATCH + at + (kg < 2 ? S::PART : 0), *const b31 = lds + wave * S::PATCH + at + (kg < 2 ? 2 * S::PART : 0);
    const unsigned char *const a11 = lds + (S::NBX * S::NBY + wave) * S::PATCH + at, *const a13 = a11 + (kg < 2 ? 0 : 2 * S::PART);
    unsigned *const flags = reinterpret_cast<unsigned *>(lds + S::FLAGS);
    int *const row_tab = reinterpret_cast<int *>(lds + S::TAB);
    if (threadIdx.x < K) row_tab[threadIdx.x] = tab[ngroups + g * K + threadIdx.x] / 4;
    const SplitConst split_const;

    f4 st[8];
    auto request = [&](auto first_, auto last_, int c) __attribute__((always_inline)) {
        static_for<decltype(first_)::value, decltype(last_)::value>([&](auto j_) {
            constexpr int j = decltype(j_)::value;
            if constexpr (j == 8) {
                lds_load_b128(a_raw, raw_to, raw_row < h ? raw_off + (unsigned)c * lda4 : OOB_OFFSET, 0);
            } else {
                st[j] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, inside ? off + (unsigned)(c + j) * ld4 : OOB_OFFSET, 0, 0));
            }
        });
    };
    // (where a thread of the first four waves puts a position's second 8 columns of A)
    auto second = [&](int t) __attribute__((always_inline)) {
        const int quad = t / 4;
        return lds + (S::NBX * S::NBY + quad / (DS_XT / 4) / 4 * (DS_XT / 4) + quad % (DS_XT / 4)) * S::PATCH + 256 + quad / (DS_XT / 4) % 4 * 64 + t % 4 * 16;
    };
    auto place = [&]() __attribute__((always_inline)) {
        unsigned low = 0;
        if (ends) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    if (moved < -k) st[j] = f4{0.f, st[j][0], st[j][1], st[j][2]};
                    if (moved > k) st[j] = f4{st[j][1], st[j][2], st[j][3], 0.f};
                }
        }
        if (have) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v[8] = {st[0][e], st[1][e], st[2][e], st[3][e], st[4][e], st[5][e], st[6][e], st[7][e]};
                u4 p[3];
                low |= split8(v, split_const, p);
                asm volatile("" : "+v"(low));
#pragma unroll
                for (int s = 0; s < 3; ++s) *reinterpret_cast<u4 *>(to + s * S::PART + e * 16) = p[s];
            }
        }
        // (A's second columns: a position's 8 a thread, four waves)
        if (wave < 4) {
            const int t = here(thread);
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const float *>(lds + S::RAW + j * 1024 + t * 4);
            unsigned char *const there = second(t);
            u4 p[3];
            low |= split8(v, split_const, p);
#pragma unroll
            for (int s = 0; s < 3; ++s) *reinterpret_cast<u4 *>(there + s * S::PART) = p[s];
        }
        const bool bad = split_inexact<5>(low, [&](int i) __attribute__((always_inline)) {
            if (i < 4 ? !have : wave >= 4) return u4{0u, 0u, 0u, 0u};
            return *reinterpret_cast<const u4 *>((i < 4 ? to + i * 16 : second(here(thread))) + 2 * S::PART);
        });
        if (lane == 0) flags[wave] = bad;
    };
    auto barrier = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    f4 acc[2][S::BY][S::BX];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int y = 0; y < S::BY; ++y)
#pragma unroll
            for (int x = 0; x < S::BX; ++x) acc[i][y][x] = f4{0.f, 0.f, 0.f, 0.f};

    constexpr int TILES = (S::BY + 1) * S::BX;
    f4 sum[2][2];
    auto add = [&](auto t_) __attribute__((always_inline)) {
        constexpr int t = decltype(t_)::value, y = t / S::BX, x = t % S::BX;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (y - i >= 0 && y - i < S::BY) {
                acc[i][y - i][x] += sum[t % 2][i];
                asm volatile("" : "+v"(acc[i][y - i][x]));       // (here, not where it is used next)
            }
    };
    request(std::integral_constant<int, 0>{}, std::integral_constant<int, S::LOADS>{}, 0);
    for (int c0 = 0; c0 < batch; c0 += 64 * DS_COLS) {
        unsigned long long exact = 0;                // stages of these 64 that the split does not hold
        const int c1 = min(c0 + 64 * DS_COLS, batch);
        for (int c = c0; c < c1; c += DS_COLS) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (the loads to LDS are not the compiler's)
            barrier();                                   // nobody reads the last stage any more
            place();
            barrier();
            const unsigned flag = flags[lane % DS_WAVES];
            u4 af[2][3], bf[2][2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                af[i][0] = *reinterpret_cast<const u4 *>(a13 + i * (DS_XT / 4) * S::PATCH);
                af[i][1] = *reinterpret_cast<const u4 *>(a11 + i * (DS_XT / 4) * S::PATCH + S::PART);
                af[i][2] = *reinterpret_cast<const u4 *>(a11 + i * (DS_XT / 4) * S::PATCH);
            }
            auto fetch = [&](auto t_) __attribute__((always_inline)) {
                constexpr int t = decltype(t_)::value, at = (t / S::BX * S::NBX + t % S::BX) * S::PATCH;
                if constexpr (t < TILES) {
                    bf[t % 2][0] = *reinterpret_cast<const u4 *>(b31 + at);
                    bf[t % 2][1] = *reinterpret_cast<const u4 *>(b21 + at);
                }
            };
            fetch(std::integral_constant<int, 0>{});
            if (__builtin_expect(__any(flag), 0)) {
                exact |= 1ull << ((c - c0) / DS_COLS);
                request(std::integral_constant<int, 0>{}, std::integral_constant<int, S::LOADS>{}, c + DS_COLS);
                continue;
            }
            // (the next stage's requests a few at a time, past the last one too, and by two thirds of the products: all at once they
            // wait for each other, the last ones at the end are waited for)
            static_for<0, TILES>([&](auto t_) {
                constexpr int t = decltype(t_)::value, y = t / S::BX;
                constexpr int first = 3 * S::LOADS * t / (2 * TILES), last = 3 * S::LOADS * (t + 1) / (2 * TILES);
                fetch(std::integral_constant<int, t + 1>{});
                request(std::integral_constant<int, (first < S::LOADS ? first : S::LOADS)>{}, std::integral_constant<int, (last < S::LOADS ? last : S::LOADS)>{}, c + DS_COLS);
                // the six products: a1 b3, a3 b1; a2 b2, a2 b1; a1 b2, a1 b1
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        if (y - i >= 0 && y - i < S::BY) sum[t % 2][i] = split_mfma(af[i][p], bf[t % 2][p > 0], p == 0 ? f4{0.f, 0.f, 0.f, 0.f} : sum[t % 2][i]);
                if constexpr (t > 0) add(std::integral_constant<int, t - 1>{});
                __builtin_amdgcn_sched_barrier(0);
            });
            add(std::integral_constant<int, TILES - 1>{});
        }
        // An operand that the split does not hold exactly -- an infinity, a NaN, a number next to the smallest ones --: its stage
        // in fp32, four columns at a time, from memory.  (Behind the loop: a second way through it cost its registers' places.)
        while (exact) {
            const int c = c0 + DS_COLS * __builtin_ctzll(exact);
            exact &= exact - 1;
            static_for<0, TILES>([&](auto t_) {
                constexpr int t = decltype(t_)::value, y = t / S::BX, x = t % S::BX;
                const int l = here(lane), row_a = i_tile + l % 16 / 4 * period + 4 * wave + l % 4, row_b = row_a + s_g + 4 * y * period + 4 * x;
                sum[t % 2][0] = sum[t % 2][1] = f4{0.f, 0.f, 0.f, 0.f};
#pragma nounroll
                for (int k = c; k < min(c + DS_COLS, batch); k += 4) {
                    const int col = k + l / 16;
                    const float b_col = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, col < batch ? (unsigned)row_b * 4u + (unsigned)col * ldb4 : OOB_OFFSET, 0, 0));
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const float a_col = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ar, col < batch ? (unsigned)(row_a + 4 * i * period) * 4u + (unsigned)col * lda4 : OOB_OFFSET, 0, 0));
                        sum[t % 2][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a_col, b_col, sum[t % 2][i], 0, 0, 0);
                    }
                }
                add(t_);
            });
        }
    }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");            // (what was requested past the last stage)
    // Results: acc[u][y][x][i] of lane (n, q) is row q, position i of the wave's patch u of A and row n / 4, position n % 4 of a
    // patch of B: slot (4 y + n / 4 - q, 4 x + n % 4 - i).  Through LDS, 4 map rows at a time, to 4 positions of a slot per lane:
    // lane (slot, place), slots 16 apart from one to the next.  What the slots held is on its way meanwhile.
    float *const out = reinterpret_cast<float *>(lds);
    const int q4 = lane / 16, by = m16 / 4 - q4, bx = m16 % 4;
    float *const there = out + (by * LC + bx) * S::PITCH + q4 * DS_XT + 4 * wave;
    constexpr int PLACES = DS_XT * DS_YT / 2 / 4, SLOTS = DS_THREADS / PLACES, ITS = (LC * K + SLOTS - 1) / SLOTS;
    const int place_y = thread % PLACES / (DS_XT / 4), place_x = 4 * (thread % (DS_XT / 4));
    static_for<0, 2>([&](auto half_) {
        constexpr int half = decltype(half_)::value;
        const int to_row = i_tile + (4 * half + place_y) * period + place_x;
        const bool is_row = tx * DS_XT + place_x < period && to_row < h;
        unsigned to_off[ITS], over = 0;              // (over: a piece that reaches over an end of B, position by position)
        f4 old[ITS];
        barrier();                                   // (the last stage's operands; the first half's results)
#pragma unroll
        for (int k = 0; k < ITS; ++k) {
            const int slot = thread / PLACES + SLOTS * k, dy = slot / LC, dx = slot - dy * LC, in0 = to_row + s_g + dy * period + dx;
            const bool is = is_row && slot < LC * K && in0 > -4 && in0 < w, whole = in0 >= 0 && in0 + 3 < w;
            to_off[k] = is ? (unsigned)(row_tab[min(dy, K - 1)] + to_row + dx * astep) * 4u : OOB_OFFSET;
            old[k] = f4{0.f, 0.f, 0.f, 0.f};
            if (beta != 0.f && whole) old[k] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(cr, to_off[k], 0, 0));
            if (is && !whole) over |= 1u << k;
        }
        static_for<0, S::BY * S::BX * 4>([&](auto e_) {
            constexpr int e = decltype(e_)::value, y = e / (4 * S::BX), x = e / 4 % S::BX, i = e % 4;
            // (checked only where a patch of B reaches over the window's edge)
            const bool in_y = (4 * y >= 3 && 4 * y + 3 < K) || (unsigned)(4 * y + by) < (unsigned)K;
            const bool in_x = (4 * x >= i && 4 * x + 3 - i < LC) || (unsigned)(4 * x - i + bx) < (unsigned)LC;
            if (in_y && in_x) there[(4 * y * LC + 4 * x - i) * S::PITCH + i] = acc[half][y][x][i];
        });
        barrier();
#pragma unroll
        for (int k = 0; k < ITS; ++k) {
            const int slot = thread / PLACES + SLOTS * k;
            const float *const from = out + min(slot, LC * K - 1) * S::PITCH + place_y * DS_XT + place_x;
            f4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = beta == 0.f ? alpha * from[i] : beta * old[k][i] + alpha * from[i];
            if (!((over >> k) & 1u)) {
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), cr, to_off[k], 0, 0);
            } else {
                const int dy = slot / LC, in0 = to_row + s_g + dy * period + slot - dy * LC;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (in0 + i < 0 || in0 + i >= w) continue;
                    float r = alpha * from[i];
                    if (beta != 0.f) r += beta * __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(cr, to_off[k] + 4u * i, 0, 0));
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, r), cr, to_off[k] + 4u * i, 0, 0);
                }
            }
        }
    });
}

template <int LC, int K>
hipError_t ds_launch(const DiaView &C, float *vals, const float *A, long long lda, const float *B, long long ldb, int batch,
                     float alpha, float beta, hipStream_t stream, long long workgroups, int txn, const DsTiles &tiles)
{
    const WalkView &wk = C.walk_n;
    note_kernel("dd2dia_split_kernel<%d, %d>", LC, K);
    launch_kernel((dd2dia_split_kernel<LC, K>), dim3((unsigned)std::max(workgroups, (long long)tiles.first_tile[wk.ngroups])), dim3(DS_THREADS), 0, stream,
                  wk.tab_dev, wk.ngroups, wk.period, wk.s0, wk.astep4 / 4, vals, A, lda, B, ldb, C.h, C.w, batch, alpha, beta,
                  (unsigned)((((long long)batch - 1) * lda + C.h) * 4), (unsigned)((((long long)batch - 1) * ldb + C.w) * 4),
                  (unsigned)((long long)C.nd * C.stride * 4), txn, tiles);
    return hipGetLastError();
}

// Fills in the launch's tiles; false: another table, operands that 16-byte pieces do not fit, or (not force) a launch on
// which the kernel would not be ahead.
bool ds_plan(const DiaView &C, const float *B, long long lda, long long ldb, int batch, bool force, DsTiles &tiles)
{
    const WalkView &wk = C.walk_n;
    if (wk.tab_dev == nullptr || wk.lck != wk.k || wk.k != 13 || wk.ngroups > DS_MAX_GROUPS || batch < 1 ||
        !wk.rows4 || wk.period % 4 != 0 || C.h % 4 != 0 || C.w % 4 != 0 || wk.astep4 % 4 != 0 || lda % 4 != 0 || ldb % 4 != 0 ||
        reinterpret_cast<unsigned long long>(B) % 16 != 0)
        return false;
    const long long block = (long long)DS_YT * wk.period, txn = (wk.period + DS_XT - 1) / DS_XT, tyn = (C.h + block - 1) / block;
    // every byte offset, those of rows past the operands' ends included, on its side of 2^32
    long long far = 0;
    for (int g = 0; g < wk.ngroups; ++g) far = std::max(far, std::abs((long long)wk.s0 + wk.rows_host[g]));
    const long long reach = far + tyn * block + 64 * txn + (wk.k + 16LL) * wk.period;
    if ((((long long)batch + 2 * DS_COLS) * std::max(lda, ldb) + reach) * 4 >= (1LL << 32) || reach >= (1LL << 29) || txn * tyn * wk.ngroups > 0x7fffffffLL)
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
    // three quarters of the rounds' positions are the map's, and from 128 columns on, below which the results' way out (8000
    // clocks and more per tile) is too much of a tile.  Measured on 140 random layers of maps 190 to 545 wide, batch 27 to 720,
    // against the kernel with a wave per window row: 54 are taken, at 0.93 - 1.49 times its rate (median 1.20, two below 1.0);
    // forced on others, 0.74 - 1.25 below 128 columns (median 0.94) and 0.88 - 1.13 where the rounds are emptier.  Not
    // asked where the projection runs chunk by chunk (maps below 256 wide, by that kernel's rule): forced there, 0.89 - 1.38 times
    // the rate from 128 columns on, ahead where the rounds are full.
    const long long rounds = ((n + 7) / 8 + 31) / 32;
    return force || (batch >= 128 && 4 * n * wk.period >= 3 * rounds * 256 * txn * DS_XT);
}

}  // namespace

hipError_t launch_dd2dia_split(const DiaView &C, float *vals, const float *A, long long lda, const float *B, long long ldb,
                               int batch, float alpha, float beta, hipStream_t stream, long long workgroups)
{
    DsTiles tiles;
    if (!ds_plan(C, B, lda, ldb, batch, workgroups == 0, tiles)) return hipErrorNotSupported;
    const int txn = (C.walk_n.period + DS_XT - 1) / DS_XT;
    return ds_launch<13, 13>(C, vals, A, lda, B, ldb, batch, alpha, beta, stream, workgroups, txn, tiles);
}

}  // namespace cuvdia
