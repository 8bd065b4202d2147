// Loads, waits and operand unpacking shared by the decode kernels on prepared operands (abq_gemm_decode_tiled.hip,
// abq_gemm_decode_tiled_grouped.hip).  The loads are issued from inline assembly because the compiler would sink plain
// loads below a barrier, next to their first use; a value loaded that way is consumed through a landed() call behind a
// counted wait.
#pragma once
#include "abq_kernels.h"
#include "abq_lds_dma.h"
#include "abq_bits.h"

namespace abq {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr bool decode_tiled_width(int b) { return b == 2 || b == 4 || b == 8; }
// single-field widths, activations at least as wide as the weights
constexpr bool decode_tiled_built(int q, int p) { return decode_tiled_width(q) && decode_tiled_width(p) && q >= p; }

__device__ __forceinline__ v4u dt_load16(const char *base, uint32_t off)
{
    v4u v;
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(v) : "v"(off), "s"(base) : "memory");
    return v;
}
// the same for weight records.  once: nothing reads the record a second time (the grid has one block of rows), and the
// load is marked non-temporal, so that the lines do not displace what the workgroups share in the L2; with several
// blocks of rows the other blocks' workgroups read the record again and it is loaded like anything else.  (wave-uniform)
// (One statement with a scalar branch inside, not two statements under an if: the destination is then one register
// whichever way the load is issued, and no copy of a register still in flight can come between load and wait.)
__device__ __forceinline__ v4u dt_load16_weights(const char *base, uint32_t off, int once)
{
    v4u v;
    asm volatile("s_cmp_lg_u32 %3, 0\n\t"
                 "s_cbranch_scc1 .Ldt_once_%=\n\t"
                 "global_load_dwordx4 %0, %1, %2\n\t"
                 "s_branch .Ldt_issued_%=\n"
                 ".Ldt_once_%=:\n\t"
                 "global_load_dwordx4 %0, %1, %2 nt\n"
                 ".Ldt_issued_%=:"
                 : "=&v"(v)
                 : "v"(off), "s"(base), "s"(__builtin_amdgcn_readfirstlane(once))
                 : "memory", "scc");
    return v;
}

template <int N> __device__ __forceinline__ void dt_wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// the same with a count that is constant only after unrolling
__device__ __forceinline__ void dt_wait_loads_n(int n)
{
#define ABQ_DT_WAIT_CASE(i) case i: dt_wait_loads<i>(); break;
#define ABQ_DT_WAIT_CASES8(i) ABQ_DT_WAIT_CASE(i) ABQ_DT_WAIT_CASE(i + 1) ABQ_DT_WAIT_CASE(i + 2) ABQ_DT_WAIT_CASE(i + 3) \
    ABQ_DT_WAIT_CASE(i + 4) ABQ_DT_WAIT_CASE(i + 5) ABQ_DT_WAIT_CASE(i + 6) ABQ_DT_WAIT_CASE(i + 7)
    switch (n) {
    ABQ_DT_WAIT_CASES8(0) ABQ_DT_WAIT_CASES8(8) ABQ_DT_WAIT_CASES8(16) ABQ_DT_WAIT_CASES8(24)
    ABQ_DT_WAIT_CASES8(32) ABQ_DT_WAIT_CASES8(40) ABQ_DT_WAIT_CASES8(48) ABQ_DT_WAIT_CASES8(56)
    default: dt_wait_loads<0>(); break;
    }
#undef ABQ_DT_WAIT_CASES8
#undef ABQ_DT_WAIT_CASE
}
// ties a register filled by dt_load16 to the wait in front of it: every use comes after
__device__ __forceinline__ void dt_landed(v4u &v) { asm volatile("" : "+v"(v)); }

// One 16-byte unit of a BITS-wide single-field record -> 8 / BITS MFMA operands of four dwords.
// Signed: value * 2^(8 - BITS) (the field at the top of the byte); unsigned: the value.
template <int BITS, bool SIGNED> __device__ __forceinline__ void dt_unpack(const v4u &u, v4i (&out)[8 / BITS])
{
    if (BITS == 8) {
        out[0] = v4i{ (int)u[0], (int)u[1], (int)u[2], (int)u[3] };
    } else if (BITS == 4) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t a = u[2 * i], b = u[2 * i + 1];
            if (SIGNED)
                out[i] = v4i{ (int)((a << 4) & 0xF0F0F0F0u), (int)(a & 0xF0F0F0F0u), (int)((b << 4) & 0xF0F0F0F0u), (int)(b & 0xF0F0F0F0u) };
            else
                out[i] = v4i{ (int)(a & 0x0F0F0F0Fu), (int)((a >> 4) & 0x0F0F0F0Fu), (int)(b & 0x0F0F0F0Fu), (int)((b >> 4) & 0x0F0F0F0Fu) };
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w = u[i];
            if (SIGNED)
                out[i] = v4i{ (int)((w << 6) & 0xC0C0C0C0u), (int)((w << 4) & 0xC0C0C0C0u), (int)((w << 2) & 0xC0C0C0C0u), (int)(w & 0xC0C0C0C0u) };
            else
                out[i] = v4i{ (int)(w & 0x03030303u), (int)((w >> 2) & 0x03030303u), (int)((w >> 4) & 0x03030303u), (int)((w >> 6) & 0x03030303u) };
        }
    }
}

typedef unsigned v2u __attribute__((ext_vector_type(2)));

// a lane's share of one weight record (32 elements): P dwords
// ONCE: kernels whose grid never has a second block of rows say so, and their loads go out without two branches each
template <int P> struct DtgShare {
    v4u v[P / 4];
    static constexpr int kLoads = P / 4;
    template <bool ONCE = false> __device__ __forceinline__ void issue(const char *base, uint32_t off, int once)
    {
#pragma unroll
        for (int i = 0; i < P / 4; ++i) {
            if constexpr (ONCE)
                asm volatile("global_load_dwordx4 %0, %1, %2 nt" : "=&v"(v[i]) : "v"(off + 16u * i), "s"(base) : "memory");
            else
                v[i] = dt_load16_weights(base, off + 16u * i, once);
        }
    }
    __device__ __forceinline__ void landed()
    {
#pragma unroll
        for (int i = 0; i < P / 4; ++i)
            dt_landed(v[i]);
    }
};
template <> struct DtgShare<2> {
    v2u v;
    static constexpr int kLoads = 1;
    template <bool ONCE = false> __device__ __forceinline__ void issue(const char *base, uint32_t off, int once)
    {
        if constexpr (ONCE)
            asm volatile("global_load_dwordx2 %0, %1, %2 nt" : "=&v"(v) : "v"(off), "s"(base) : "memory");
        else
            asm volatile("s_cmp_lg_u32 %3, 0\n\t"
                     "s_cbranch_scc1 .Ldt_once_%=\n\t"
                     "global_load_dwordx2 %0, %1, %2\n\t"
                     "s_branch .Ldt_issued_%=\n"
                     ".Ldt_once_%=:\n\t"
                     "global_load_dwordx2 %0, %1, %2 nt\n"
                     ".Ldt_issued_%=:"
                     : "=&v"(v)
                     : "v"(off), "s"(base), "s"(__builtin_amdgcn_readfirstlane(once))
                     : "memory", "scc");
    }
    __device__ __forceinline__ void landed() { asm volatile("" : "+v"(v)); }
};

// one dword of a 2-bit record -> one MFMA operand
template <bool SIGNED> __device__ __forceinline__ v4i dtg_unpack2(uint32_t w)
{
    if (SIGNED)
        return v4i{ (int)((w << 6) & 0xC0C0C0C0u), (int)((w << 4) & 0xC0C0C0C0u), (int)((w << 2) & 0xC0C0C0C0u), (int)(w & 0xC0C0C0C0u) };
    return v4i{ (int)(w & 0x03030303u), (int)((w >> 2) & 0x03030303u), (int)((w >> 4) & 0x03030303u), (int)((w >> 6) & 0x03030303u) };
}

template <int P, bool SIGNED> __device__ __forceinline__ void dtg_operands(const DtgShare<P> &w, v4i (&bv)[2])
{
    if constexpr (P == 2) {
        bv[0] = dtg_unpack2<SIGNED>(w.v[0]);
        bv[1] = dtg_unpack2<SIGNED>(w.v[1]);
    } else if constexpr (P == 4) {
        dt_unpack<4, SIGNED>(w.v[0], bv);
    } else {
        bv[0] = v4i{ (int)w.v[0][0], (int)w.v[0][1], (int)w.v[0][2], (int)w.v[0][3] };
        bv[1] = v4i{ (int)w.v[1][0], (int)w.v[1][1], (int)w.v[1][2], (int)w.v[1][3] };
    }
}

} // namespace abq
