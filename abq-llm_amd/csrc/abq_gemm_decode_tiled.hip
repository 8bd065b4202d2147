// GEMM core for decode-sized M on prepared operands: both operands in the K-tiled field-packed layout
// (abq_bits.h), widths of a single field (2, 4 or 8 bits).
//
// Replaces AqBMMAKernel::mainLoop + ::epilogue of the reference
// (engine/mma_any/aq_bmma_kernel.h:109-271, :485-580) for one (x_bits, w_bits) pair per
// translation unit: compile with -DABQ_Q=<x_bits> -DABQ_P=<w_bits>.
//
// A decode GEMM streams 4 to 11 MB of weights once; at 8 TB/s that takes 0.5 to 1.4 us, the same order as
// one memory round trip and as a kernel launch, and every kernel starts with cold caches.  What decides
// the time is therefore the length of the dependent chain from the first instruction to the last store and
// the number of vector instructions on it (with sixteen waves on a compute unit an instruction of every
// wave costs sixteen issue cycles per SIMD quad), not the byte count.  Hence:
//   * prepared operands: a lane's 16-byte weight load is what it feeds the matrix core after a shift and a
//     mask per four elements (no bit-matrix transpose), activations are int8-ready records (nothing to
//     expand, no bytes more than the planes have);
//   * a workgroup is T tiles of 16 weight rows over the whole K; wave w takes K steps w, w + NW, ...
//     (a step = one 16-byte load per lane = 512 / P elements of K over the four lane groups);
//   * the activations of the workgroup's rows go from global memory straight into LDS
//     (global_load_lds_dwordx4: no registers, nothing to wait for before the weight loads are issued);
//     chunk c of a row lands at c ^ (row & (Q - 1)) so that the sixteen rows a lane group reads hit
//     different banks (the permutation is applied to the source address, the destination is linear);
//   * the first D steps' weight loads of every wave are issued right behind them, all before the first
//     wait; one counted wait (the activation loads are older than the weight loads) and one barrier
//     later every wave reads its A operands with ds_read_b128;
//   * the loads are issued from inline assembly: the compiler would sink plain loads below the barrier,
//     next to their first use.  Values loaded that way are consumed through `landed()` after a counted
//     wait, in the loop iteration that issued them (no register of theirs lives across the back edge,
//     where a compiler-inserted copy could read it before it has landed);
//   * per-wave partial tiles meet in LDS and are summed by the threads that store them (integer adds:
//     any order gives the same bits).
// K longer than NW * D steps runs further rounds of the same loop (their latency is exposed).
#include <type_traits>

#include "abq_kernels.h"
#include "abq_bits.h"
#include "abq_decode_loads.h"

#ifndef ABQ_Q
#error "compile with -DABQ_Q=<x_bits> -DABQ_P=<w_bits>"
#endif

namespace abq {

// XF16: the activations arrive as fp16 [M][K] and are quantised here with one static scale, value =
// (int)(half(x) * half(scale)) as pack_half of the reference does (abq_gemm_wrapper.cu:29-54), straight into the
// int8 records in LDS: the pack kernel and its launch in front of every decode GEMM of the FT wrapper fall away.
// Every workgroup converts the rows it multiplies (M x K halves, from L2 after the first).  8-bit activations.
// XF16 is the number of 16-byte units of eight halves a thread holds per pass (0: the activations arrive packed; 1, 2
// or 4, the launcher takes the fewest that cover the rows in one pass, at most 4: eight rows of 4096 with sixteen waves;
// more spills, and with four the instances need 95 - 104 registers against 52 - 67, which costs workgroups per unit).
// FLIP (unsigned pairs): the 8-bit records hold codes up to 255, which the signed matrix cores take as value - 128
// (bit 7 flipped: one xor per dword after the load); the result is put right with 128 x the other operand's row
// sums (GemmArgs::x_row_sums / w_row_sums, abq_row_sums) and, when both operands are 8 bits wide, - 2^14 K.  Without
// FLIP the bytes of an unsigned 8-bit record are fed as they are: padded records of narrower codes (below 128).
template <int Q, int P, bool SIGNED, int NW, int D, int T, int XF16 = 0, bool FLIP = false>
__global__ __launch_bounds__(64 * NW) void gemm_decode_tiled(const GemmArgs a, int mrows)
{
    static_assert(!XF16 || Q == 8, "in-kernel quantisation writes 8-bit records");
    static_assert(!FLIP || (!SIGNED && Q == 8 && !XF16), "flipping is for unsigned 8-bit records");
    constexpr bool FLIP_X = FLIP && Q == 8, FLIP_W = FLIP && P == 8;
    static_assert(XF16 == 0 || XF16 == 1 || XF16 == 2 || XF16 == 4, "units per thread and pass");
    constexpr int XP = XF16 > 0 ? XF16 : 1;
    constexpr int NXL = Q / P;   // activation chunks (16 bytes) per weight unit
    constexpr int NM = 8 / P;    // MFMAs per weight unit
    constexpr int MX = 8 / Q;    // MFMAs per activation chunk
    constexpr int NT = 64 * NW;
    constexpr int QLOG = Q == 8 ? 3 : Q == 4 ? 2 : 1;
    constexpr int XC = 6;        // activation wave loads per wave that are unrolled
    extern __shared__ __align__(16) unsigned char smem[];
    int *red = reinterpret_cast<int *>(smem);   // [NW][T][16][16]
    unsigned char *xs = smem + NW * T * 1024;   // [kt][row][Q chunks], chunks permuted within a row

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int M = a.M, N = a.N;
    const int KT = a.K >> 7;
    const int U = KT * P;            // 16-byte units per weight row
    const int S = (U + 3) >> 2;      // steps
    const int tile0 = blockIdx.x * T;
    const int m0 = blockIdx.y * mrows;
    const int once = gridDim.y == 1; // no other workgroup reads this one's weight records
    const int Mb = min(mrows, M - m0);
    const char *Xt = reinterpret_cast<const char *>(a.X);
    const char *Wt = reinterpret_cast<const char *>(a.W);
    const unsigned xs_addr = (unsigned)(size_t)xs;
    const int xchunks = KT * Mb * Q;

    // The scales that are one number for the whole call, and the row sums of flipped records, are each wave's oldest loads
    // and land in the first KB of its share of red, which is free until the K loop is over.  Loaded next to their uses, the
    // scale the activations are quantised with waited for every weight load in flight as well (a compiler's wait behind
    // loads it does not know of), and what the result needs put a memory latency behind the last barrier: with the
    // activations requested up here as well, W2A8 x 1 row with a static scale 5.2 -> 4.2 us a GEMM over 4096 x 4096,
    // 11008 x 4096 and 4096 x 11008, W8A8 9.9 -> 9.2.
    // (The scale of the result only with fp16 activations: the instances for packed ones feed the int32 results, where the test
    // and its branches cost 0.02 us of 4.04 a launch, and gained nothing on W4A4 with a scale.)
    const bool tensor_scale = XF16 && a.out_kind == 3;
    int *own = red + wid * T * 256;
    const unsigned own_addr = (unsigned)(size_t)own;
    if constexpr (XF16)
        lds_dma4(a.x_pack_scale, 0u, own_addr);
    if (tensor_scale)
        lds_dma4(a.C, 0u, own_addr + 256u);
    if constexpr (FLIP_X)
        lds_dma4(a.w_row_sums, (uint32_t)min(tile0 * 16 + lane, N - 1) * 4u, own_addr + 512u);
    if constexpr (FLIP_W)
        lds_dma4(a.x_row_sums, (uint32_t)min(m0 + lane, M - 1) * 4u, own_addr + 768u);

    // ---- activations: LDS chunk p <- chunk p ^ ((p / Q) & (Q - 1)) of the workgroup's rows -----------
    // (XF16: loaded, quantised and written inside the first round below)
    const int upr = a.K >> 3;     // XF16: units of eight halves per row
    const int nunits = Mb * upr;
    // units -> rows: all of them are below 2^15 (their bytes lie in LDS), half a unit outweighs the reciprocal's error
    const float row_of_unit = XF16 ? __builtin_amdgcn_rcpf((float)upr) : 0.f;
    const char *Xh = Xt + (size_t)m0 * a.K * 2;
    v4u xr[XP];
    if constexpr (XF16) {
        // every pass is loaded, past the rows' end the last unit once more: a load under a condition would leave the
        // compiler a register to merge with an undefined one, and a copy it inserts for that reads before the data lands.
        // (Up here, not with the first weights: the hundred instructions that prepare the K loop issue in their shadow.)
#pragma unroll
        for (int i = 0; i < XP; ++i)
            xr[i] = dt_load16(Xh, (uint32_t)min(tid + i * NT, nunits - 1) * 16u);
    }
    uint32_t sel_pair = 0, sel_half = 0;
    if constexpr (XF16)
        quad_transpose_selectors(tid & 3, sel_pair, sel_half);
    // eight halves of unit p (row p / upr, elements 8 u .. 8 u + 7) -> their bytes of the row's int8 record: the
    // quad's four units are one word-set, whose expanded dword s, byte c is element 7 - s of lane 3 - c
    auto quantise_unit = [&](const v4u &raw, int p, _Float16 hs) {
        union {
            v4u q;
            _Float16 h[8];
        } r;
        r.q = raw;
        int v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c)
            v[c] = (int)(_Float16)(r.h[c] * hs); // fp16 product rounded to nearest even, conversion truncating
        const uint32_t e_even = quad_transpose_bytes(pack_low_bytes(v[7], v[5], v[3], v[1]), sel_pair, sel_half);
        const uint32_t e_odd = quad_transpose_bytes(pack_low_bytes(v[6], v[4], v[2], v[0]), sel_pair, sel_half);
        if (p < nunits) {
            const int row = (int)(((float)p + 0.5f) * row_of_unit), u = p - row * upr;
            const int rowi = (u >> 4) * Mb + row;                        // K tile * rows + row
            const int dw = 8 * ((u >> 2) & 3) + 2 * (u & 3);             // first of the lane's two dwords in the record
            const int chunk = (dw >> 2) ^ (rowi & 7);
            *reinterpret_cast<uint2 *>(xs + ((uint32_t)rowi * 8 + chunk) * 16u + (dw & 3) * 4u) = make_uint2(e_even, e_odd);
        }
    };
    if constexpr (XF16) {
    } else if (Mb == M) { // the rows of all K tiles are one contiguous block
#pragma unroll
        for (int i = 0; i < XC; ++i) {
            const int pb = wid * 64 + i * NT; // wave-uniform
            if (pb < xchunks) {
                const int p = pb + lane;
                const int src = min(p ^ ((p >> QLOG) & (Q - 1)), xchunks - 1);
                lds_dma16(Xt + (uint32_t)src * 16u, xs_addr + (unsigned)pb * 16u);
            }
        }
        for (int pb = wid * 64 + XC * NT; pb < xchunks; pb += NT) {
            const int p = pb + lane;
            const int src = min(p ^ ((p >> QLOG) & (Q - 1)), xchunks - 1);
            lds_dma16(Xt + (uint32_t)src * 16u, xs_addr + (unsigned)pb * 16u);
        }
    } else { // several blocks of rows: a K tile's rows are Mb * Q chunks out of M * Q
        const int per = Mb * Q;
        for (int pb = wid * 64; pb < xchunks; pb += NT) {
            const int p = min(pb + lane, xchunks - 1);
            const int q = p ^ ((p >> QLOG) & (Q - 1));
            const int kt = q / per, rem = q - kt * per;
            lds_dma16(Xt + ((size_t)(kt * M + m0) * Q + rem) * 16u, xs_addr + (unsigned)pb * 16u);
        }
    }

    // ---- weights: byte offset of (lane, step s, tile t) = step_w(s) + woff[t] ------------------------
    uint32_t woff[T], back;
    {
        const int n = min(tile0 * 16 + r, N - 1);
        const uint32_t lane_w = P == 2 ? ((uint32_t)(g >> 1) * N + n) * 32u + (g & 1) * 16u : (uint32_t)n * (P * 16u) + g * 16u;
        back = lane_w - (uint32_t)n * (P * 16u); // distance to the first unit of the step in the same row
#pragma unroll
        for (int t = 0; t < T; ++t)
            woff[t] = lane_w + ((T > 1 && (tile0 + t) * 16 + r < N) ? t * (16u * P * 16u) : 0u);
    }
    const uint32_t step_bytes = (uint32_t)N * 64u; // a step covers 4 units of every row: 64 bytes times N rows
    auto step_w = [&](int s) -> uint32_t {
        return P == 8 ? (uint32_t)(s >> 1) * (2u * step_bytes) + (s & 1) * 64u : (uint32_t)s * step_bytes;
    };
    const bool ragged = (U & 3) != 0; // the last step has fewer than four units

    v4i acc[T][2];
#pragma unroll
    for (int t = 0; t < T; ++t)
        acc[t][0] = acc[t][1] = v4i{ 0, 0, 0, 0 };
    const int ml = min(r, Mb - 1);

    int round = 0;
    do {
        // this round's steps of the wave: wid + (round * D + d) * NW.  Every wave issues D * T loads (steps past
        // the end repeat the last one), so that the waits below can count.
        v4u wb[D][T];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int s = min(wid + (round * D + d) * NW, S - 1);
            const char *wp = Wt + step_w(s);
            // lanes past the end of K (last step only) read the step's first unit of their row instead
            const uint32_t bk = (ragged && s == S - 1 && 4 * s + g >= U) ? back : 0u;
#pragma unroll
            for (int t = 0; t < T; ++t)
                wb[d][t] = dt_load16_weights(wp, woff[t] - bk, once);
        }
        if (round == 0) {
            dt_wait_loads<D * T>(); // the loads of the scales and the activations are older than these
            if constexpr (XF16) {
                const _Float16 hs = (_Float16)__builtin_bit_cast(float, own[0]);
#pragma unroll
                for (int i = 0; i < XP; ++i)
                    dt_landed(xr[i]);
#pragma unroll
                for (int i = 0; i < XP; ++i) {
                    if (i * NT < nunits) // the quads of a wave are whole
                        quantise_unit(xr[i], tid + i * NT, hs);
                }
                // rows too long for one pass: further passes, their latency exposed
                for (int base = XP * NT; base < nunits; base += XP * NT) {
                    v4u more[XP];
#pragma unroll
                    for (int i = 0; i < XP; ++i)
                        more[i] = dt_load16(Xh, (uint32_t)min(base + tid + i * NT, nunits - 1) * 16u);
                    dt_wait_loads<0>(); // these are the youngest loads
#pragma unroll
                    for (int i = 0; i < XP; ++i) {
                        dt_landed(more[i]);
                        if (base + i * NT < nunits)
                            quantise_unit(more[i], base + tid + i * NT, hs);
                    }
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int cs = wid + (round * D + d) * NW;
            const bool have = cs < S; // wave-uniform
            v4i av[NM];
            if (have) {
                const int u0 = (4 * cs + g) * NXL;           // first activation chunk of lane group and step along K
                const int rowi = (u0 >> QLOG) * Mb + ml;      // row index in LDS: K tile * rows + row
#pragma unroll
                for (int i = 0; i < NXL; ++i) {
                    const int part = ((u0 + i) & (Q - 1)) ^ (rowi & (Q - 1));
                    const v4u xv = *reinterpret_cast<const v4u *>(xs + ((uint32_t)rowi * Q + part) * 16u);
                    v4i tt[MX];
                    dt_unpack<Q, SIGNED>(xv, tt);
                    if constexpr (FLIP_X)
                        tt[0] = v4i{ tt[0][0] ^ (int)0x80808080u, tt[0][1] ^ (int)0x80808080u, tt[0][2] ^ (int)0x80808080u,
                                     tt[0][3] ^ (int)0x80808080u };
#pragma unroll
                    for (int k = 0; k < MX; ++k)
                        av[i * MX + k] = tt[k];
                }
            }
            // Waited for and marked as landed on every path: a register with a load still in flight must not
            // look free to the compiler (it would reuse it, and the late data would land on the new value).
            dt_wait_loads_n((D - 1 - d) * T);
#pragma unroll
            for (int t = 0; t < T; ++t)
                dt_landed(wb[d][t]);
            if (have) {
                const bool ok = 4 * cs + g < U;
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    // (lanes past the end of K feed zeros, also where the weights are flipped)
                    constexpr unsigned kFlipW = FLIP_W ? 0x80808080u : 0u;
                    const v4u wv = ok ? v4u{ wb[d][t][0] ^ kFlipW, wb[d][t][1] ^ kFlipW, wb[d][t][2] ^ kFlipW, wb[d][t][3] ^ kFlipW }
                                      : v4u{ 0u, 0u, 0u, 0u };
                    v4i bv[NM];
                    dt_unpack<P, SIGNED>(wv, bv);
#pragma unroll
                    for (int i = 0; i < NM; ++i)
                        acc[t][i & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[i], bv[i], acc[t][i & 1], 0, 0, 0);
                }
            }
        }
        ++round;
    } while (wid + round * D * NW < S);

    // ---- the waves' partial tiles meet in LDS ----------------------------------------------------------
    // (scale and row sums are read in front of what takes their place: held through the K loop they would be registers
    // more, and some instances a workgroup per CU less.  A thread has at most one element of the result.)
    static_assert(T * 256 <= NT, "one element per thread");
    const int out_scale = tensor_scale ? own[64] : 0;
    const int w_sum = FLIP_X ? own[128 + (tid >> 8) * 16 + (tid & 15)] : 0, x_sum = FLIP_W ? own[192 + ((tid >> 4) & 15)] : 0;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (4 * g + e < Mb)
                red[((wid * T + t) * 16 + 4 * g + e) * 16 + r] = acc[t][0][e] + acc[t][1][e];
    __syncthreads();
    if (tid < T * 256) {
        const int t = tid >> 8, rem = tid & 255;
        const int n = (tile0 + t) * 16 + (rem & 15);
        if ((rem >> 4) < Mb && n < N) {
            int part[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w)
                part[w] = red[(w * T + t) * 256 + rem];
            int v = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w)
                v += part[w];
            if (SIGNED)
                v >>= 16 - Q - P; // both operands were fed at the top of the byte
            if constexpr (FLIP_X)
                v = (int)((unsigned)v + 128u * (unsigned)w_sum);
            if constexpr (FLIP_W)
                v = (int)((unsigned)v + 128u * (unsigned)x_sum);
            if constexpr (FLIP_X && FLIP_W)
                v = (int)((unsigned)v - 16384u * (unsigned)a.K);
            if (tensor_scale)
                store_scaled(a, m0 + (rem >> 4), n, v, (_Float16)__builtin_bit_cast(float, out_scale));
            else
                store_result(a, m0 + (rem >> 4), n, v);
        }
    }
}

// ---- weights of several fields ------------------------------------------------------------------
//
// Widths of 3, 5, 6 and 7 bits are records of a 4-bit, a 2-bit and a 1-bit field (abq_bits.h: a row's K tile is
// P * 16 bytes, the field of width F the F units of 16 bytes at byte 16 * (P & ~(2F - 1))).  Inside its region a
// field is laid out exactly as a single-field record of that width, so the plan above carries over field by field:
// a step of field F is one 16-byte load per lane, lane group g taking unit 4 cs + g of the field's units along K
// (K tile (4 cs + g) / F, unit (4 cs + g) % F of it), 8 / F MFMAs against the 128 / F activations the unit covers.
// A field is fed at the place its bits have in the code (signed: in the code moved to the top of the byte, so that
// the widest field carries the sign and the others are non-negative), all fields into one accumulator: the sum is
// the dot product times 2^(16 - QP - P) as for a single field.  The steps of all fields form one list (4-bit
// field first), wave w takes steps w, w + NW, ...; which field a step belongs to is the same for the whole wave.
// The weights are the records the prefill kernels read (abq_relayout_planes): one copy serves both.  The
// activations are records of a single field of QP bits: their own width, or for 3, 5, 6 and 7 bits the next such
// width with the codes extended (abq_relayout_planes_padded); activation bytes are small at decode.
template <int F, int POS, bool TOP> __device__ __forceinline__ void dt_unpack_field(const v4u &u, v4i (&out)[8 / F])
{
    // word j of the unit carries in byte c, at bits [F s, F s + F), the field of expanded dword (8 / F) j + s;
    // operand i = expanded dwords 4 i .. 4 i + 3.  The field goes to bits [POS, POS + F) of the byte.
    constexpr uint32_t mask = field_mask(F) << POS;
    constexpr int per = 8 / F; // expanded dwords per word
#pragma unroll
    for (int i = 0; i < 8 / F; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int d = 4 * i + c, j = d / per, sft = POS - F * (d % per);
            const uint32_t w = u[j];
            out[i][c] = (int)((sft >= 0 ? w << (sft >= 0 ? sft : 0) : w >> (sft < 0 ? -sft : 0)) & mask);
        }
    (void)TOP;
}

constexpr int dt_field_steps(int kt, int p, int f) { return (p & f) ? (kt * f + 3) / 4 : 0; }

template <int QP, int P, bool SIGNED, int NW, int D, bool FLIP_X = false>
__global__ __launch_bounds__(64 * NW) void gemm_decode_fields(const GemmArgs a, int mrows)
{
    static_assert(QP == 4 || QP == 8, "activations as records of one field");
    static_assert(P == 3 || P == 5 || P == 6 || P == 7, "weights of several fields");
    static_assert(!FLIP_X || (!SIGNED && QP == 8), "flipping is for unsigned 8-bit records");
    constexpr int MX = 8 / QP; // MFMAs per activation chunk
    constexpr int NT = 64 * NW;
    constexpr int QLOG = QP == 8 ? 3 : 2;
    constexpr int XC = 6;
    constexpr int WPOS = SIGNED ? 8 - P : 0; // place of the code's lowest bit in the byte
    extern __shared__ __align__(16) unsigned char smem[];
    int *red = reinterpret_cast<int *>(smem); // [NW][16][16]
    unsigned char *xs = smem + NW * 1024;     // [kt][row][QP chunks], chunks permuted within a row

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int M = a.M, N = a.N;
    const int KT = a.K >> 7;
    const int S4 = dt_field_steps(KT, P, 4), S2 = dt_field_steps(KT, P, 2), S1 = dt_field_steps(KT, P, 1);
    const int S = S4 + S2 + S1;
    const int tile0 = blockIdx.x;
    const int m0 = blockIdx.y * mrows;
    const int once = gridDim.y == 1;
    const int Mb = min(mrows, M - m0);
    const char *Xt = reinterpret_cast<const char *>(a.X);
    const char *Wt = reinterpret_cast<const char *>(a.W);
    const unsigned xs_addr = (unsigned)(size_t)xs;
    const int xchunks = KT * Mb * QP;

    // the weights' row sums: as in gemm_decode_tiled
    int *own = red + wid * 256;
    if constexpr (FLIP_X)
        lds_dma4(a.w_row_sums, (uint32_t)min(tile0 * 16 + lane, N - 1) * 4u, (unsigned)(size_t)own + 256u);

    // ---- activations: as in gemm_decode_tiled ---------------------------------------------------------
    if (Mb == M) {
#pragma unroll
        for (int i = 0; i < XC; ++i) {
            const int pb = wid * 64 + i * NT;
            if (pb < xchunks) {
                const int p = pb + lane;
                const int src = min(p ^ ((p >> QLOG) & (QP - 1)), xchunks - 1);
                lds_dma16(Xt + (uint32_t)src * 16u, xs_addr + (unsigned)pb * 16u);
            }
        }
        for (int pb = wid * 64 + XC * NT; pb < xchunks; pb += NT) {
            const int p = pb + lane;
            const int src = min(p ^ ((p >> QLOG) & (QP - 1)), xchunks - 1);
            lds_dma16(Xt + (uint32_t)src * 16u, xs_addr + (unsigned)pb * 16u);
        }
    } else {
        const int per = Mb * QP;
        for (int pb = wid * 64; pb < xchunks; pb += NT) {
            const int p = min(pb + lane, xchunks - 1);
            const int q = p ^ ((p >> QLOG) & (QP - 1));
            const int kt = q / per, rem = q - kt * per;
            lds_dma16(Xt + ((size_t)(kt * M + m0) * QP + rem) * 16u, xs_addr + (unsigned)pb * 16u);
        }
    }

    // ---- weights: byte offset of (lane, field F, step cs) = K tile * tile_bytes + row_off + field_off[F] ----
    const uint32_t tile_bytes = (uint32_t)N * (P * 16u);
    const uint32_t row_off = (uint32_t)min(tile0 * 16 + r, N - 1) * (P * 16u);
    // flat step t -> field (4: t < S4; 2: t < S4 + S2; else 1) and the field's own step; wave-uniform
    auto weight_offset = [&](int t) -> uint32_t {
        int kt;
        uint32_t fo;
        if (t < S4) {
            kt = t;
            fo = 16u * field_list_index(P, 4) + 16u * g;
        } else if (t < S4 + S2) {
            kt = 2 * (t - S4) + (g >> 1);
            fo = 16u * field_list_index(P, 2) + 16u * (g & 1);
        } else {
            kt = 4 * (t - S4 - S2) + g;
            fo = 16u * field_list_index(P, 1);
        }
        return (uint32_t)min(kt, KT - 1) * tile_bytes + row_off + fo; // lanes past the end of K repeat the last K tile
    };

    v4i acc[2];
    acc[0] = acc[1] = v4i{ 0, 0, 0, 0 };
    const int ml = min(r, Mb - 1);

    // the activations of the unit (field F, step cs) of this lane group -> 8 / F MFMA operands
    auto read_x = [&](auto fc, int cs, v4i(&av)[8]) {
        constexpr int F = decltype(fc)::value;
        constexpr int NXL = QP >= F ? QP / F : 1; // activation chunks per weight unit
        const int uu = min(4 * cs + g, KT * F - 1);
        const int u0 = uu * NXL;
        const int rowi = (u0 >> QLOG) * Mb + ml;
#pragma unroll
        for (int i = 0; i < NXL; ++i) {
            const int part = ((u0 + i) & (QP - 1)) ^ (rowi & (QP - 1));
            const v4u xv = *reinterpret_cast<const v4u *>(xs + ((uint32_t)rowi * QP + part) * 16u);
            v4i tt[MX];
            dt_unpack<QP, SIGNED>(xv, tt);
            if constexpr (FLIP_X)
                tt[0] = v4i{ tt[0][0] ^ (int)0x80808080u, tt[0][1] ^ (int)0x80808080u, tt[0][2] ^ (int)0x80808080u,
                             tt[0][3] ^ (int)0x80808080u };
#pragma unroll
            for (int k = 0; k < MX; ++k)
                av[i * MX + k] = tt[k];
        }
    };
    auto multiply = [&](auto fc, int cs, const v4u &wraw, const v4i(&av)[8]) {
        constexpr int F = decltype(fc)::value;
        const bool ok = 4 * cs + g < KT * F;
        const v4u wv = ok ? wraw : v4u{ 0u, 0u, 0u, 0u };
        v4i bv[8 / F];
        dt_unpack_field<F, WPOS + field_base(P, F), SIGNED>(wv, bv);
#pragma unroll
        for (int i = 0; i < 8 / F; ++i)
            acc[i & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[i], bv[i], acc[i & 1], 0, 0, 0);
    };

    int round = 0;
    do {
        v4u wb[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int t = min(wid + (round * D + d) * NW, S - 1);
            wb[d] = dt_load16_weights(Wt, weight_offset(t), once);
        }
        if (round == 0) {
            dt_wait_loads<D>(); // the loads of the sums and the activations are older than these
            __syncthreads();
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int t = wid + (round * D + d) * NW;
            const bool have = t < S; // wave-uniform
            v4i av[8];
            if (have) {
                if ((P & 4) && t < S4)
                    read_x(std::integral_constant<int, 4>{}, t, av);
                else if ((P & 2) && t < S4 + S2)
                    read_x(std::integral_constant<int, 2>{}, t - S4, av);
                else if (P & 1)
                    read_x(std::integral_constant<int, 1>{}, t - S4 - S2, av);
            }
            dt_wait_loads_n(D - 1 - d);
            dt_landed(wb[d]);
            if (have) {
                if ((P & 4) && t < S4)
                    multiply(std::integral_constant<int, 4>{}, t, wb[d], av);
                else if ((P & 2) && t < S4 + S2)
                    multiply(std::integral_constant<int, 2>{}, t - S4, wb[d], av);
                else if (P & 1)
                    multiply(std::integral_constant<int, 1>{}, t - S4 - S2, wb[d], av);
            }
        }
        ++round;
    } while (wid + round * D * NW < S);

    // ---- the waves' partial tiles meet in LDS ----------------------------------------------------------
    static_assert(256 <= NT, "one element per thread");
    const int w_sum = FLIP_X ? own[64 + (tid & 15)] : 0;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (4 * g + e < Mb)
            red[(wid * 16 + 4 * g + e) * 16 + r] = acc[0][e] + acc[1][e];
    __syncthreads();
    if (tid < 256) {
        const int n = tile0 * 16 + (tid & 15);
        if ((tid >> 4) < Mb && n < N) {
            int part[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w)
                part[w] = red[w * 256 + tid];
            int v = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w)
                v += part[w];
            if (SIGNED)
                v >>= 16 - QP - P;
            if constexpr (FLIP_X)
                v = (int)((unsigned)v + 128u * (unsigned)w_sum);
            store_result(a, m0 + (tid >> 4), n, v);
        }
    }
}

template <int QP, int P, bool SIGNED, int NW, int D, bool MAY_FLIP>
static hipError_t launch_decode_fields(const GemmArgs &a, hipStream_t stream)
{
    const int mrows = decode_tiled_rows(NW, 1, a.M, a.K, QP);
    if (mrows == 0 || (size_t)a.N * a.K * P / 8 >= (1ull << 32) || (size_t)a.M * a.K * QP / 8 >= (1ull << 32))
        return hipErrorInvalidValue;
    const size_t lds = decode_tiled_lds(NW, 1, mrows, a.K, QP);
    const int tiles = (a.N + 15) / 16;
    const dim3 grid(tiles, (a.M + mrows - 1) / mrows);
    auto go = [&](auto kernel) -> hipError_t {
        const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (attr != hipSuccess)
            return attr;
        hipLaunchKernelGGL(kernel, grid, dim3(64 * NW), lds, stream, a, mrows);
        return hipGetLastError();
    };
    if constexpr (!SIGNED && QP == 8 && MAY_FLIP) {
        if (a.flip_x) { // true 8-bit codes (fed as value - 128); padded narrower codes go as they are
            if (!a.w_row_sums)
                return hipErrorInvalidValue;
            return go(&gemm_decode_fields<QP, P, SIGNED, NW, D, true>);
        }
    }
    return go(&gemm_decode_fields<QP, P, SIGNED, NW, D, false>);
}

template <int Q, int P, bool SIGNED, int NW, int D, int T, int XU, bool FLIP = false>
static hipError_t launch_decode_tiled_instance(const GemmArgs &a, int mrows, hipStream_t stream)
{
    const size_t lds = decode_tiled_lds(NW, T, mrows, a.K, Q);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_decode_tiled<Q, P, SIGNED, NW, D, T, XU, FLIP>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (attr != hipSuccess)
        return attr;
    const int tiles = (a.N + 15) / 16;
    const dim3 grid((tiles + T - 1) / T, (a.M + mrows - 1) / mrows);
    hipLaunchKernelGGL((gemm_decode_tiled<Q, P, SIGNED, NW, D, T, XU, FLIP>), grid, dim3(64 * NW), lds, stream, a, mrows);
    return hipGetLastError();
}

template <int Q, int P, bool SIGNED, int NW, int D, int T, bool XF16 = false>
static hipError_t launch_decode_tiled(const GemmArgs &a, hipStream_t stream)
{
    const int mrows = decode_tiled_rows(NW, T, a.M, a.K, Q);
    if (mrows == 0 || (size_t)a.N * a.K * P / 8 >= (1ull << 32) || (size_t)a.M * a.K * (XF16 ? 16 : Q) / 8 >= (1ull << 32))
        return hipErrorInvalidValue;
    if (XF16 && !a.x_pack_scale)
        return hipErrorInvalidValue;
    if constexpr (XF16) {
        const int need = (int)(((size_t)mrows * a.K / 8 + 64 * NW - 1) / (64 * NW)); // units per thread for one pass
        if (need <= 1)
            return launch_decode_tiled_instance<Q, P, SIGNED, NW, D, T, 1>(a, mrows, stream);
        if (need <= 2)
            return launch_decode_tiled_instance<Q, P, SIGNED, NW, D, T, 2>(a, mrows, stream);
        return launch_decode_tiled_instance<Q, P, SIGNED, NW, D, T, 4>(a, mrows, stream);
    } else if constexpr (!SIGNED && Q == 8) {
        // unsigned 8-bit records: codes up to 255 in every 8-bit operand (flipped, row sums needed), or padded
        // narrower codes in every one (fed as they are); a mix of the two has no instance
        const bool flip_x = a.flip_x != 0, flip_w = P == 8 && a.flip_w != 0;
        if (!flip_x && !flip_w)
            return launch_decode_tiled_instance<Q, P, SIGNED, NW, D, T, 0>(a, mrows, stream);
        if (!flip_x || (P == 8 && !flip_w) || !a.w_row_sums || (P == 8 && !a.x_row_sums))
            return hipErrorInvalidValue;
        return launch_decode_tiled_instance<Q, P, SIGNED, NW, D, T, 0, true>(a, mrows, stream);
    } else {
        return launch_decode_tiled_instance<Q, P, SIGNED, NW, D, T, 0>(a, mrows, stream);
    }
}

// Native tile space of this kernel: (waves, weight loads in flight per wave, tiles per workgroup).  Entries name
// MFMA 16x16x64 with NSTAGE = 6; wk = waves, tn = tiles, kb = K elements a wave has in flight (D steps).
#define ABQ_DT_VARIANTS(V) V(16, 1, 1) V(16, 3, 1) V(8, 2, 1) V(16, 1, 3) V(8, 1, 2) V(8, 2, 2) V(16, 1, 2)

#define ABQ_DT_ENTRY_T(NW, D, T) { 16, 1, T, 1, 1, NW, 6, &launch_decode_tiled<ABQ_Q, ABQ_P, true, NW, D, T>, (512 / ABQ_P) * D },
#define ABQ_DT_ENTRY_F(NW, D, T) { 16, 1, T, 1, 1, NW, 6, &launch_decode_tiled<ABQ_Q, ABQ_P, false, NW, D, T>, (512 / ABQ_P) * D },

// activations of 3, 5, 6 or 7 bits reach these kernels as records of the next single-field width
#define ABQ_QP (ABQ_Q == 3 ? 4 : (ABQ_Q >= 5 && ABQ_Q <= 7) ? 8 : ABQ_Q)
#define ABQ_P_ONE_FIELD (ABQ_P == 2 || ABQ_P == 4 || ABQ_P == 8)
#define ABQ_Q_ONE_FIELD (ABQ_Q == 2 || ABQ_Q == 4 || ABQ_Q == 8)

#if ABQ_Q_ONE_FIELD && ABQ_P_ONE_FIELD
static const KernelEntry kSigned[] = { ABQ_DT_VARIANTS(ABQ_DT_ENTRY_T) };
// the single-tile instances with in-kernel quantisation of fp16 activations (8-bit activations, signed), same order
#if ABQ_Q == 8
#define ABQ_DT_ENTRY_X(NW, D, T) { 16, 1, T, 1, 1, NW, 6, &launch_decode_tiled<ABQ_Q, ABQ_P, true, NW, D, T, true>, (512 / ABQ_P) * D },
static const KernelEntry kSignedF16[] = { ABQ_DT_ENTRY_X(16, 1, 1) ABQ_DT_ENTRY_X(16, 3, 1) ABQ_DT_ENTRY_X(8, 2, 1) };
#define ABQ_DT_NF16 3
#else
static const KernelEntry *const kSignedF16 = nullptr;
#define ABQ_DT_NF16 0
#endif
static const KernelEntry kUnsigned[] = { ABQ_DT_VARIANTS(ABQ_DT_ENTRY_F) };
#define ABQ_DT_NUNSIGNED ((int)(sizeof(kUnsigned) / sizeof(kUnsigned[0])))
#define ABQ_DT_NSIGNED ((int)(sizeof(kSigned) / sizeof(kSigned[0])))
#else
static const KernelEntry *const kSignedF16 = nullptr;
#define ABQ_DT_NF16 0
#if ABQ_P_ONE_FIELD
// activations of several fields over weights of one (W2A6): the kernel above on activation records padded to ABQ_QP bits
#define ABQ_DT_ENTRY_PT(NW, D, T) { 16, 1, T, 1, 1, NW, 6, &launch_decode_tiled<ABQ_QP, ABQ_P, true, NW, D, T>, (512 / ABQ_P) * D },
#define ABQ_DT_ENTRY_PF(NW, D, T) { 16, 1, T, 1, 1, NW, 6, &launch_decode_tiled<ABQ_QP, ABQ_P, false, NW, D, T>, (512 / ABQ_P) * D },
static const KernelEntry kSigned[] = { ABQ_DT_VARIANTS(ABQ_DT_ENTRY_PT) };
static const KernelEntry kUnsigned[] = { ABQ_DT_VARIANTS(ABQ_DT_ENTRY_PF) };
#else
// weights of several fields: (waves, weight loads in flight per wave); warp K in the tile's name = 128 D
#define ABQ_DF_VARIANTS(V) V(16, 2) V(16, 4) V(8, 4)
#define ABQ_DF_ENTRY_T(NW, D) { 16, 1, 1, 1, 1, NW, 6, &launch_decode_fields<ABQ_QP, ABQ_P, true, NW, D, false>, 128 * D },
#define ABQ_DF_ENTRY_F(NW, D) { 16, 1, 1, 1, 1, NW, 6, &launch_decode_fields<ABQ_QP, ABQ_P, false, NW, D, ABQ_Q == 8>, 128 * D },
static const KernelEntry kSigned[] = { ABQ_DF_VARIANTS(ABQ_DF_ENTRY_T) };
static const KernelEntry kUnsigned[] = { ABQ_DF_VARIANTS(ABQ_DF_ENTRY_F) };
#endif
#define ABQ_DT_NUNSIGNED ((int)(sizeof(kUnsigned) / sizeof(kUnsigned[0])))
#define ABQ_DT_NSIGNED ((int)(sizeof(kSigned) / sizeof(kSigned[0])))
#endif

#define ABQ_CAT_(a, b, c, d) a##b##c##d
#define ABQ_CAT(a, b, c, d) ABQ_CAT_(a, b, c, d)

void ABQ_CAT(abq_decode_tiled_register_, ABQ_Q, _, ABQ_P)(KernelTable *out)
{
    out[0] = KernelTable{ ABQ_Q, ABQ_P, 1, kSigned, ABQ_DT_NSIGNED };
    out[1] = KernelTable{ ABQ_Q, ABQ_P, 0, kUnsigned, ABQ_DT_NUNSIGNED };
}

void ABQ_CAT(abq_decode_tiled_f16_register_, ABQ_Q, _, ABQ_P)(KernelTable *out)
{
    out[0] = KernelTable{ ABQ_Q, ABQ_P, 1, kSignedF16, ABQ_DT_NF16 };
    out[1] = KernelTable{ ABQ_Q, ABQ_P, 0, nullptr, 0 };
}

} // namespace abq
