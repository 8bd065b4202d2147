// GEMM core for 17 to 64 rows (more in blocks of 64) on prepared operands with group-wise weight scales (groups of 128),
// 8-bit activations, fp16 output, zero points on either side, optionally the fused SiLU gate:
//
// D[m][n] = x_scale[m] * ( sum_g w_scale[n][g] * (acc_g - w_zero[n][g] * Sx[m][g]) - x_zero[m] * T[n] ),
//
// semantics of algorithm/quantize/quantizer.py:111-179 of the reference.  One (x_bits, w_bits) pair per translation unit:
// compile with -DABQ_Q=8 -DABQ_P=<w_bits>.
//
// What bounds it: the weights' one trip from memory (4 to 90 MB) and, on narrow outputs, the activations' trip from L2 into
// every compute unit (M x K bytes each).  Neither of the neighbouring kernels serves that range: the decode kernel walks
// blocks of 16 rows and streams the weights once per block, and the staged prefill tiles take a barrier and a memory
// latency per K tile with 64 to 344 workgroups on the chip (64x64 tile, 0.26 us per K tile).  Here, as in the decode kernel,
//   * a wave owns blocks of four K tiles (block b goes to wave b mod NW) for T tiles of 16 weight rows, and meets the other
//     waves only in the final sum: no barrier in the K loop;
//   * the weights go from memory to the registers of the wave that multiplies them, D steps (K tiles) ahead, and are unpacked
//     once for all MB blocks of 16 rows;
//   * the activations of a step go from L2 into a ring of R buffers of the wave's own LDS (global_load_lds, no registers);
//     a buffer is refilled as soon as its operands are in registers, so R steps are in flight beside the products;
//   * T is chosen so that the workgroups make as few rounds of the 256 compute units as possible (rows_grouped_plan).
// The order of every sum depends on K alone, so all T and MB give the same bits.
//
// W4A8 with zero points on both sides, 43 rows (us, against the 64x64 and 64x128 prefill tiles on the same records): 4096 x
// 4096 7.9 / 13.4, 12288 x 4096 12.9 / 13.7, 22016 x 4096 with the gate 19.8 / 26.6, 4096 x 11008 15.0 / 26.4.  What is left
// above the weights' trip (2 to 9 us): the launch, the first loads, the fold of every tile, and the final sum, in that order
// in every workgroup, since one fills a compute unit.
#include <type_traits>

#include "abq_decode_loads.h"
#include "abq_kernels.h"
#include "abq_rows_grouped.h"

#if !defined(ABQ_Q) || !defined(ABQ_P) || ABQ_Q != 8
#error "compile with -DABQ_Q=8 -DABQ_P=<w_bits>"
#endif

namespace abq {

// ONE: the grid has one block of rows (m_blocks = 1): no division to find the workgroup's place, and the weight loads carry
// the hint without two branches each (W4A8 with zero points, eight decoder layers at 43 tokens: 275.8 -> 271.6 us).
template <int P, int T, int MB, bool ZP, bool ONE> __device__ __forceinline__ void rows_grouped(const GemmArgs &a, int m_blocks)
{
    constexpr int R = rows_ring(P, T, MB), D = rows_ahead(P, T, MB);
    constexpr int LX = 2 * MB;                 // wave loads of a step: activations (into LDS)
    constexpr int LW = T * DtgShare<P>::kLoads; // ... weights
    constexpr int LS = rows_scale_loads(T, MB, ZP); // ... of a block: scales, zero points, group sums (into LDS)
    constexpr int XB = MB * 2048;              // bytes of a step's activations
    static_assert(4 % D == 0 && R <= D && R < 4, "the rings' places follow from the step of the block");
    extern __shared__ __align__(16) unsigned char smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int NW = blockDim.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int M = a.M, N = a.N;
    const int KT = a.K >> 7;
    const int nblocks = (KT + 3) >> 2;
    // The blocks of rows of one set of weight rows run on one XCD (workgroup id modulo 8), one after the other: the second
    // finds the weights in that L2.
    const int slot = blockIdx.x >> 3;
    const int nb = ONE ? (int)blockIdx.x : (slot / m_blocks) * 8 + (blockIdx.x & 7);
    const int m0 = ONE ? 0 : (slot % m_blocks) * (MB * 16);
    const int tile0 = nb * T;
    if (tile0 * 16 >= N)
        return; // uniform over the workgroup, before any barrier
    const int Mb = min(MB * 16, M - m0);
    const int once = m_blocks == 1; // no other workgroup reads this one's weights
    const bool row_zero = a.x_zero != nullptr;

    unsigned char *ring = smem + wid * (R * XB);
    float *sws = reinterpret_cast<float *>(smem + NW * (R * XB) + wid * (LS * 256)); // [T][16 rows][4 groups]
    float *zws = sws + T * 64;                                                       // [T][16 rows][4 groups]
    int *sxs = reinterpret_cast<int *>(zws + T * 64);                                // [MB][4 groups][16 rows]
    float *par = reinterpret_cast<float *>(smem + rows_lds_for_rows(NW, P, T, MB, ZP)); // [2][64]: scales, zero points of the rows
    float *terms = par + 128;                                                        // [128]

    // ---- byte offsets of the lane's share ---------------------------------------------------------------------------
    uint32_t woff[T], soff[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        woff[t] = (uint32_t)min((tile0 + t) * 16 + r, N - 1) * (P * 16u) + (uint32_t)g * (4u * P);
        soff[t] = (uint32_t)min((tile0 + t) * 16 + (lane >> 2), N - 1) * (uint32_t)KT;
    }
    // Place 64 i + lane of a step's activations = row 8 i + lane / 8, place lane % 8 of its eight 16-byte chunks: chunk c of
    // row m sits at place c ^ ((m / 2) % 8), so that sixteen rows' reads of one chunk hit sixteen different bank groups (a
    // row is half the banks wide).  Rows past the last one are copies of it.
    uint32_t xoff[LX], sumoff[MB];
#pragma unroll
    for (int i = 0; i < LX; ++i) {
        const int m = 8 * i + (lane >> 3);
        xoff[i] = (uint32_t)(m0 + min(m, Mb - 1)) * 128u + (uint32_t)((lane & 7) ^ ((m >> 1) & 7)) * 16u;
    }
#pragma unroll
    for (int b = 0; b < MB; ++b)
        sumoff[b] = (uint32_t)(m0 + min(16 * b + r, Mb - 1)) * (uint32_t)KT;
    int a_off[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
        a_off[j] = r * 128 + ((2 * g + j) ^ ((r >> 1) & 7)) * 16;
    const size_t wstep = (size_t)N * (P * 16u), xstep = (size_t)M * 128u;
    const char *Xt = reinterpret_cast<const char *>(a.X);
    const char *Wt = reinterpret_cast<const char *>(a.W);

    // What the final sum needs per row and column: the oldest loads of their waves.
    if (wid == 0) {
        const uint32_t row = (uint32_t)(m0 + min(lane, Mb - 1)) * 4u;
        lds_dma4(a.x_scale, row, (unsigned)(size_t)par);
        if (row_zero)
            lds_dma4(a.x_zero, row, (unsigned)(size_t)(par + 64));
    }
    if (row_zero && wid == NW - 1) {
#pragma unroll
        for (int i = 0; i < (T + 3) / 4; ++i)
            lds_dma4(a.w_zero_term, (uint32_t)min(tile0 * 16 + i * 64 + lane, N - 1) * 4u, (unsigned)(size_t)(terms + i * 64));
    }

    // Step s of the wave: K tile s % 4 of its block s / 4 (steps past the end of K repeat the last tile and count nothing).
    auto k_tile = [&](int blk, int i) { return min(4 * (blk * NW + wid) + i, KT - 1); };
    DtgShare<P> wb[D][T];
    auto request_w = [&](int blk, int i, int at) {
        const char *wp = Wt + (size_t)k_tile(blk, i) * wstep;
#pragma unroll
        for (int t = 0; t < T; ++t)
            wb[at][t].template issue<ONE>(wp, woff[t], once);
    };
    auto request_x = [&](int blk, int i, int buf) {
        const char *xp = Xt + (size_t)k_tile(blk, i) * xstep;
        const unsigned to = (unsigned)(size_t)ring + (unsigned)buf * XB;
#pragma unroll
        for (int c = 0; c < LX; ++c)
            lds_dma16(xp, xoff[c], to + c * 1024u);
    };
    // a block's scales: sixteen rows times four groups per instruction, neighbouring lanes on neighbouring groups
    auto request_scales = [&](int blk) {
        const int first = 4 * (blk * NW + wid);
        const uint32_t grp = (uint32_t)min(first + (lane & 3), KT - 1);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const uint32_t off = (soff[t] + grp) * 4u;
            lds_dma4(a.w_scale, off, (unsigned)(size_t)(sws + t * 64));
            if constexpr (ZP)
                lds_dma4(a.w_zero, off, (unsigned)(size_t)(zws + t * 64));
        }
        if constexpr (ZP) {
#pragma unroll
            for (int b = 0; b < MB; ++b)
                lds_dma4(a.x_group_sums, (sumoff[b] + (uint32_t)min(first + g, KT - 1)) * 4u, (unsigned)(size_t)(sxs + b * 64));
        }
    };

    typedef float v4f __attribute__((ext_vector_type(4)));
    v4f facc[T][MB];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int b = 0; b < MB; ++b)
            facc[t][b] = v4f{ 0.f, 0.f, 0.f, 0.f };
    // signed codes are fed at the top of the byte: acc_g carries a factor 2^(16 - 8 - P), and so do the group sums (exact)
    constexpr float kShift = (float)(1 << (8 - P));

    const int blocks = (nblocks - wid + NW - 1) / NW; // of this wave, at least one
    // The first requests, in the order in which the steps below make them.
#pragma unroll
    for (int v = -D; v < 0; ++v) {
        if (v == -1)
            request_scales(0);
        if (v + R >= 0)
            request_x(0, v + R, v + R);
        request_w(0, v + D, v + D);
    }

    // One block.  Step i waits for its operands, reads those that lie in LDS, requests the scales of the next block (step 3,
    // once they have been read) and the activations of step i + R into the buffer just read, multiplies, and requests the
    // weights of step i + D into the registers just used.  LAST: nothing is requested past the block.
    int buf0 = 0;
    auto block = [&](int blk, auto last) {
        constexpr bool LAST = decltype(last)::value;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // Loads requested after the youngest one that step i needs: its activations (step i - R) or, where the weights
            // are no further ahead, its weights (same step, later); the first step of a block its scales (the step before).
            auto loads_of = [](int j, bool scales, bool x, bool w) { // requested by step j, of the kinds named
                const bool next = !LAST || j < 0;
                return (scales && j == -1 ? LS : scales && next && j == 3 ? LS : 0) + (x && (next || j + R < 4) ? LX : 0) +
                       (w && (next || j + D < 4) ? LW : 0);
            };
            int younger = 0;
            if (i == 0) {
                younger = R > 1 ? loads_of(-1, false, true, D > 1) : 0;
            } else {
                younger = D > R ? loads_of(i - R, false, false, true) : 0;
                for (int j = i - R + 1; j < i; ++j)
                    younger += loads_of(j, true, true, true);
            }
            dt_wait_loads_n(younger);
            auto &w = wb[i % D];
#pragma unroll
            for (int t = 0; t < T; ++t)
                w[t].landed();
            const unsigned char *buf = ring + (unsigned)buf0 * XB;
            v4i av[MB][2], sx[MB];
            float sw[T], zw[T];
            const bool have = 4 * (blk * NW + wid) + i < KT;
#pragma unroll
            for (int b = 0; b < MB; ++b) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    av[b][j] = *reinterpret_cast<const v4i *>(buf + b * 2048 + a_off[j]);
                if constexpr (ZP)
                    sx[b] = *reinterpret_cast<const v4i *>(sxs + b * 64 + i * 16 + 4 * g);
            }
#pragma unroll
            for (int t = 0; t < T; ++t) {
                sw[t] = sws[t * 64 + r * 4 + i];
                if constexpr (ZP)
                    zw[t] = zws[t * 64 + r * 4 + i] * -kShift;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // what was read may be written again
            if (!LAST && i == 3)
                request_scales(blk + 1);
            if (!LAST || i + R < 4)
                request_x(i + R < 4 ? blk : blk + 1, (i + R) & 3, buf0);
            buf0 = buf0 + 1 == R ? 0 : buf0 + 1;
#pragma unroll
            for (int t = 0; t < T; ++t)
                sw[t] = have ? sw[t] : 0.f;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                v4i bv[2];
                dtg_operands<P, true>(w[t], bv);
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[b][0], bv[0], v4i{ 0, 0, 0, 0 }, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[b][1], bv[1], acc, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        facc[t][b][e] = __builtin_fmaf(sw[t], ZP ? __builtin_fmaf(zw[t], (float)sx[b][e], (float)acc[e]) : (float)acc[e], facc[t][b][e]);
                }
            }
            // (nothing of the next step before this one is through: the registers of two steps' operands would spill)
            __builtin_amdgcn_sched_barrier(0);
            if (!LAST || i + D < 4)
                request_w(i + D < 4 ? blk : blk + 1, (i + D) & 3, i % D);
        }
    };
    for (int blk = 0; blk + 1 < blocks; ++blk)
        block(blk, std::false_type{});
    block(blocks - 1, std::true_type{});

    // ---- the waves' partial tiles meet in LDS, added in the order of the waves ----------------------------------------
    // [wave][tile][block of rows][column][16 rows]: a lane's four rows are one 16-byte piece, and a wave's pieces lie one
    // after the other.
    v4f *red = reinterpret_cast<v4f *>(smem);
    _Float16 *out = reinterpret_cast<_Float16 *>(a.D);
    // (All tiles at once: two at a time, a pair of barriers for each, 22016 x 4096 took 21.2 us in a trace instead of 19.9.)
    __syncthreads(); // every wave is through with its ring and its scales
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int b = 0; b < MB; ++b)
            red[((wid * T + t) * MB + b) * 64 + r * 4 + g] = facc[t][b];
    __syncthreads();
    for (int o = tid; o < T * MB * 64; o += (int)blockDim.x) {
        const int t = o / (MB * 64), rem = o % (MB * 64), b = rem >> 6, gg = (rem >> 4) & 3, c = rem & 15;
        const int n = (tile0 + t) * 16 + c, mr = b * 16 + gg * 4;
        if (n >= N || mr >= Mb || (a.act && (t & 1)))
            continue;
        auto total = [&](int tt) {
            v4f v = v4f{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll 8
            for (int w = 0; w < NW; ++w)
                v += red[((w * T + tt) * MB + b) * 64 + c * 4 + gg];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float f = v[e] * (1.0f / kShift);
                if (row_zero)
                    f = __builtin_fmaf(-par[64 + mr + e], terms[tt * 16 + c], f);
                f *= par[mr + e];
                // (rounded to fp32 here in every instance: in some of them the compiler would fuse this product into the conversion
                // to fp16, and they would differ in a last place now and then)
                asm("" : "+v"(f));
                v[e] = f;
            }
            return v;
        };
        const v4f v = total(t);
        if (T > 1 && a.act) { // this tile holds gate rows, the next one their up rows
            const v4f up = total(T > 1 ? t + 1 : t);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (mr + e < Mb)
                    out[(size_t)(m0 + mr + e) * (N / 2) + (n >> 5) * 16 + c] = (_Float16)(silu(v[e]) * up[e]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (mr + e < Mb)
                    out[(size_t)(m0 + mr + e) * N + n] = (_Float16)v[e];
        }
    }
}

template <int P, int T, int MB, bool ZP> __global__ __launch_bounds__(64 * kRowsWaves) void gemm_rows_grouped(const GemmArgs a)
{
    rows_grouped<P, T, MB, ZP, true>(a, 1);
}
template <int P, int T, int MB, bool ZP> __global__ __launch_bounds__(64 * kRowsWaves) void gemm_rows_grouped(const GemmArgs a, int m_blocks)
{
    rows_grouped<P, T, MB, ZP, false>(a, m_blocks);
}

// ---- launch -------------------------------------------------------------------------------------------------------

template <int P, int T, int MB, bool ZP> static hipError_t launch_rows_instance(const GemmArgs &a, const RowsPlan &plan, hipStream_t stream)
{
    if constexpr (!rows_built(P, T, MB)) {
        return hipErrorInvalidValue;
    } else {
        void (*const one)(GemmArgs) = &gemm_rows_grouped<P, T, MB, ZP>;
        void (*const several)(GemmArgs, int) = &gemm_rows_grouped<P, T, MB, ZP>;
        auto may_use_lds = [](const void *kernel) { return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); };
        static const hipError_t attr_one = may_use_lds(reinterpret_cast<const void *>(one)),
                                attr_several = may_use_lds(reinterpret_cast<const void *>(several));
        if (attr_one != hipSuccess || attr_several != hipSuccess)
            return attr_one != hipSuccess ? attr_one : attr_several;
        if (plan.m_blocks == 1)
            hipLaunchKernelGGL(one, dim3(plan.grid), dim3(64 * plan.waves), plan.lds, stream, a);
        else
            hipLaunchKernelGGL(several, dim3(plan.grid), dim3(64 * plan.waves), plan.lds, stream, a, plan.m_blocks);
        return hipGetLastError();
    }
}

#define ABQ_CAT_(a, b, c) a##b##c
#define ABQ_CAT(a, b, c) ABQ_CAT_(a, b, c)

hipError_t ABQ_CAT(launch_rows_grouped_8, _, ABQ_P)(const GemmArgs &a, hipStream_t stream)
{
    if (!rows_grouped_runs(a.M, a.N, a.K, 8, ABQ_P, a.group_size, a.act) || !a.w_scale || !a.x_scale || (a.w_zero && !a.x_group_sums) ||
        (a.x_zero && !a.w_zero_term))
        return hipErrorInvalidValue;
    const RowsPlan plan = rows_grouped_plan(ABQ_P, a.M, a.N, a.K, a.act, a.w_zero != nullptr);
    auto with_t = [&](auto bb, auto zp) -> hipError_t {
        constexpr int MB = decltype(bb)::value;
        constexpr bool ZP = decltype(zp)::value;
        switch (plan.tiles) {
        case 1: return launch_rows_instance<ABQ_P, 1, MB, ZP>(a, plan, stream);
        case 2: return launch_rows_instance<ABQ_P, 2, MB, ZP>(a, plan, stream);
        case 3: return launch_rows_instance<ABQ_P, 3, MB, ZP>(a, plan, stream);
        case 4: return launch_rows_instance<ABQ_P, 4, MB, ZP>(a, plan, stream);
        case 6: return launch_rows_instance<ABQ_P, 6, MB, ZP>(a, plan, stream);
        default: return hipErrorInvalidValue;
        }
    };
    using std::integral_constant;
    auto with_mb = [&](auto zp) -> hipError_t {
        return plan.row_blocks == 2   ? with_t(integral_constant<int, 2>{}, zp)
               : plan.row_blocks == 3 ? with_t(integral_constant<int, 3>{}, zp)
                                      : with_t(integral_constant<int, 4>{}, zp);
    };
    return a.w_zero ? with_mb(std::true_type{}) : with_mb(std::false_type{});
}

} // namespace abq
