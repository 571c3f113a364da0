// Device helpers shared by the translation units that hold kernels.
#pragma once
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace cuvdia {
namespace {

// Every kernel is launched through here.  A caller that is going to wait has an event signalled by the dispatch
// itself, which saves the packet that hipStreamSynchronize would queue behind it: launch and wait of an empty kernel
// take 9.2 us instead of 11.4.
template <class... P, class... A>
void launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, A... args)
{
    if (hipEvent_t e = launch_event()) hipExtLaunchKernelGGL(kernel, grid, block, (unsigned)lds, stream, nullptr, e, 0, static_cast<P>(args)...);
    else hipLaunchKernelGGL(kernel, grid, block, (unsigned)lds, stream, static_cast<P>(args)...);
}

// Results leave through non-temporal stores: they are streamed past the
// caches instead of waiting there, dirty, for the write-back at the kernel's
// end, which every store of a one-round kernel would otherwise meet at once.
template <class V>
__device__ __forceinline__ void stream_store(V *p, V v)
{
    __builtin_nontemporal_store(v, p);
}
// Four consecutive floats as one 16-byte store; 4-byte alignment is all a 16-byte global store needs.
__device__ __forceinline__ void stream_store4(float *p, float a, float b, float c, float d)
{
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
    __builtin_nontemporal_store(f4u{a, b, c, d}, reinterpret_cast<f4u *>(p));
}

// Hardware hands consecutive workgroup ids to the 8 XCDs round-robin, and each
// XCD has its own L2.  Remap so that every XCD works on contiguous spans of
// tiles: neighbouring row tiles share dense-operand rows (the halo and the
// bands +-px apart), which then hit in that XCD's L2.  The tiles are dealt out
// in groups of 8 spans of XCD_SPAN, one span per XCD and group, so that work
// which varies along the rows (chunks falling outside the operand) still
// spreads evenly; the last, partial group is split into 8 near-equal spans.
// The very last span is dealt backwards: the tiles at the high end of the
// rows take the slower body for tiles at the operand's ends, exactly like the
// first tiles of the first span, and dealt in order they would be the last to
// start as well -- a launch of one or two rounds then ends when they do.
constexpr int XCD_SPAN = 64;
__device__ __forceinline__ int xcd_tile(int bid, int nblk)
{
    constexpr int XCDS = 8, GROUP = XCDS * XCD_SPAN;
    const int full = nblk / GROUP * GROUP;           // tiles in whole groups
    if (bid < full) {
        const int g = bid / GROUP, in = bid - g * GROUP;
        const int xcd = in % XCDS;
        int slot = in / XCDS;
        if (xcd == XCDS - 1 && (g + 1) * GROUP == nblk) slot = XCD_SPAN - 1 - slot;
        return g * GROUP + xcd * XCD_SPAN + slot;
    }
    const int rest = nblk - full, b = bid - full;
    const int q = rest / XCDS, r = rest % XCDS;
    const int xcd = b % XCDS;
    int slot = b / XCDS;
    if (xcd == XCDS - 1) slot = q - 1 - slot;        // the last span has q tiles (r < XCDS)
    return full + xcd * q + (xcd < r ? xcd : r) + slot;
}

// Orders this wave's LDS writes before its later LDS reads (and the reverse)
// for data exchanged between lanes of ONE wave.  The LDS unit executes a
// wave's instructions in order, so only the compiler needs restraining.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw: "Parallel random numbers: as easy
// as 1, 2, 3", SC'11): a counter-based generator, 4 x 32 random bits per
// 128-bit counter and 64-bit key, no state.  The result element (row, col)
// draws word col & 3 of the block with counter (row, col >> 2, 0, 0) and key
// (seed_lo, seed_hi), so a sample depends on the seed and the element's
// position only -- not on which kernel, tile or lane produced it.
struct SpRand4 { unsigned w[4]; };
__device__ __forceinline__ SpRand4 sp_philox(unsigned row, unsigned colblock, unsigned k0, unsigned k1)
{
    unsigned c0 = row, c1 = colblock, c2 = 0u, c3 = 0u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const unsigned hi0 = __umulhi(0xD2511F53u, c0), lo0 = 0xD2511F53u * c0;
        const unsigned hi1 = __umulhi(0xCD9E8D57u, c2), lo1 = 0xCD9E8D57u * c2;
        c0 = hi1 ^ c1 ^ k0;
        c1 = lo1;
        c2 = hi0 ^ c3 ^ k1;
        c3 = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return SpRand4{{c0, c1, c2, c3}};
}
// 24 random bits -> a uniform variate in [0, 1), exactly representable
__device__ __forceinline__ float sp_uniform(unsigned word) { return (float)(word >> 8) * 0x1p-24f; }

// Last step of an SpMM result element: optional per-row bias, optional
// logistic sigmoid 1/(1+exp(-v)) (src/cuv/tensor_ops/functors.hpp:122),
// optional Bernoulli sample of that probability, v > u
// (src/cuv/random/random.cu:86-91).
__device__ __forceinline__ float sp_finish(float v, float bias, int act, unsigned word = 0u)
{
    v += bias;
    if (act == 0) return v;
    // v_exp_f32 and v_rcp_f32 (1 ulp each) instead of the library's exp and an
    // IEEE division: p is off by < 1e-7 absolute, inside what the sum's own
    // rounding allows, and the store costs a dozen instructions less per element
    const float p = __builtin_amdgcn_rcpf(1.f + __expf(-v));
    return act == 2 ? (p > sp_uniform(word) ? 1.f : 0.f) : p;
}

// Loads that deliver straight into LDS (no vector register in between): lane i
// of the wave writes its 16 bytes at lds_byte_addr + 16*i; an
// out-of-range lane writes zeros, an inactive lane writes nothing.  They are
// vector-memory operations and complete in order with the wave's other loads
// (s_waitcnt vmcnt).  Written in assembly so that the waits can be
// placed by hand: the loops keep them in flight across
// barriers, which no automatic placement allows.  M0 is written inside the
// statement without appearing among its clobbers: the compiler treats M0 as a
// reserved register (it never keeps a value there across other code, and sets
// it immediately before each instruction of its own that reads it), and it
// rejects reserved registers in a clobber list with a warning.
typedef int sp_int4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ sp_int4 raw_rsrc(const void *base, unsigned bytes)
{
    const unsigned long long b = reinterpret_cast<unsigned long long>(base);
    return sp_int4{(int)(unsigned)b, (int)((unsigned)(b >> 32) & 0xffffu), (int)bytes, 0x00020000};
}
// The wait: five issue slots between a vector instruction that writes a scalar register and a load that reads it -- the compiler
// brings a resource or an offset back from vector registers right in front of a statement, and does not look into it --, one
// behind the write of M0.  (Eight slots more cost the plane's walk 0.6 - 2.6 %, patches 0.5 - 2.8 %, the other kernels less.)
#define CUVDIA_LDS_LOAD "s_mov_b32 m0, %0\n\ts_nop 3\n\t"
// (operands that are in scalar registers as it is)
__device__ __forceinline__ void lds_load_b128_scalar(sp_int4 rsrc, unsigned lds_byte_addr, unsigned voff, unsigned soff)
{
    asm volatile(CUVDIA_LDS_LOAD "buffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_byte_addr), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
__device__ __forceinline__ void lds_load_b128(sp_int4 rsrc, unsigned lds_byte_addr, unsigned voff, unsigned soff)
{
    // all three are wave-uniform by construction; this keeps them in scalar registers whatever the compiler infers
    lds_byte_addr = __builtin_amdgcn_readfirstlane(lds_byte_addr);
    soff = __builtin_amdgcn_readfirstlane(soff);
    rsrc = sp_int4{__builtin_amdgcn_readfirstlane(rsrc.x), __builtin_amdgcn_readfirstlane(rsrc.y),
                   __builtin_amdgcn_readfirstlane(rsrc.z), __builtin_amdgcn_readfirstlane(rsrc.w)};
    lds_load_b128_scalar(rsrc, lds_byte_addr, voff, soff);
}
// the same with 4 bytes per lane: lane i writes at lds_byte_addr + 4*i
__device__ __forceinline__ void lds_load_b32(sp_int4 rsrc, unsigned lds_byte_addr, unsigned voff)
{
    lds_byte_addr = __builtin_amdgcn_readfirstlane(lds_byte_addr);
    rsrc = sp_int4{__builtin_amdgcn_readfirstlane(rsrc.x), __builtin_amdgcn_readfirstlane(rsrc.y),
                   __builtin_amdgcn_readfirstlane(rsrc.z), __builtin_amdgcn_readfirstlane(rsrc.w)};
    asm volatile(CUVDIA_LDS_LOAD "buffer_load_dword %1, %2, 0 offen lds"
                 :: "s"(lds_byte_addr), "v"(voff), "s"(rsrc) : "memory");
}
#undef CUVDIA_LDS_LOAD

// f(integral_constant<I>) ... f(integral_constant<N - 1>)
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// acc[r] += a(lane 16 n + r) * x[r], r = 0..7: the values broadcast inside each row of 16 lanes; fma16_dpp after that
// += a(lane 16 n + 8 + r) * x[1 + r].  A DPP operand must not have been written by a VALU instruction in the two preceding
// issue slots, and the compiler does not look into a statement: hence the wait at its head.
#define CUVDIA_FMA_DPP(r, x, lane) "v_fmac_f32_dpp %" #r ", %8, %" #x " row_newbcast:" #lane " row_mask:0xf bank_mask:0xf\n\t"
#define CUVDIA_FMA8_DPP                                                                                     \
    CUVDIA_FMA_DPP(0, 9, 0) CUVDIA_FMA_DPP(1, 10, 1) CUVDIA_FMA_DPP(2, 11, 2) CUVDIA_FMA_DPP(3, 12, 3)      \
    CUVDIA_FMA_DPP(4, 13, 4) CUVDIA_FMA_DPP(5, 14, 5) CUVDIA_FMA_DPP(6, 15, 6) CUVDIA_FMA_DPP(7, 16, 7)
__device__ __forceinline__ void fma8_dpp(float (&acc)[8], float a, const float *x)
{
    asm("s_nop 1\n\t" CUVDIA_FMA8_DPP
        : "+&v"(acc[0]), "+&v"(acc[1]), "+&v"(acc[2]), "+&v"(acc[3]), "+&v"(acc[4]), "+&v"(acc[5]), "+&v"(acc[6]), "+&v"(acc[7])
        : "v"(a), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]));
}
__device__ __forceinline__ void fma16_dpp(float (&acc)[8], float a, const float *x)
{
    asm("s_nop 1\n\t" CUVDIA_FMA8_DPP
        CUVDIA_FMA_DPP(0, 10, 8) CUVDIA_FMA_DPP(1, 11, 9) CUVDIA_FMA_DPP(2, 12, 10) CUVDIA_FMA_DPP(3, 13, 11)
        CUVDIA_FMA_DPP(4, 14, 12) CUVDIA_FMA_DPP(5, 15, 13) CUVDIA_FMA_DPP(6, 16, 14) CUVDIA_FMA_DPP(7, 17, 15)
        : "+&v"(acc[0]), "+&v"(acc[1]), "+&v"(acc[2]), "+&v"(acc[3]), "+&v"(acc[4]), "+&v"(acc[5]), "+&v"(acc[6]), "+&v"(acc[7])
        : "v"(a), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]), "v"(x[8]));
}
#undef CUVDIA_FMA8_DPP
#undef CUVDIA_FMA_DPP

constexpr unsigned OOB_OFFSET = 0x80000000u;     // >= every resource size used here

// Four floats as one 16-byte buffer store at a vector offset and a scalar one.  Such a store reads its registers up to two issue
// slots late, and the compiler waits for that only where there is no scalar offset: the last lanes once stored the address that the
// next instruction had written there.  The wait names the registers, so they are not written before it.
template <int CPOL>
__device__ __forceinline__ void buffer_store4(float __attribute__((ext_vector_type(4))) v, __amdgpu_buffer_rsrc_t rsrc, unsigned voff, unsigned soff)
{
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), rsrc, voff, soff, CPOL);
    asm volatile("s_nop 1" :: "v"(v));
}

}  // namespace
}  // namespace cuvdia
