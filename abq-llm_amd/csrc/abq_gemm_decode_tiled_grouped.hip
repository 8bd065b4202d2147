// GEMM core for decode-sized M on prepared operands with group-wise weight scales (groups of 128 or 64), fp16 output,
// zero points on either side, optionally the fused SiLU gate (tile pairs: 16 gate rows, their 16 up rows):
//
// D[m][n] = x_scale[m] * ( sum_g w_scale[n][g] * (acc_g - w_zero[n][g] * Sx[m][g]) - x_zero[m] * T[n] ),
//
// acc_g the integer dot product over scale group g, Sx the sums of the activation codes; semantics of
// algorithm/quantize/quantizer.py:111-179 of the reference.  One (x_bits, w_bits) pair per translation unit: compile
// with -DABQ_Q=<x_bits> -DABQ_P=<w_bits>.
//
// A matrix-core instruction sums over its four lane groups, so all four must hold elements of the same scale group: a
// step is ONE K tile (one group of 128), lane group g holds 32 of its elements (4 P bytes of the weight record, 4 Q
// bytes of the activation record), and the step's two instructions leave acc_g, which is folded into fp32 right away.
//
// What bounds it: launch, one cold memory round trip and the stream of weights, scales and zero points (4 to 34 MB), so
// everything of a wave is requested before its first wait, and no wave waits for another before the final sum:
//   * a wave owns blocks of S = four K tiles (block b of K goes to wave b mod NW) for T tiles of 16 weight rows.  Every
//     record of the activations, every scale and zero point is then used by exactly one wave of the workgroup, which
//     brings it in for itself.  (Staging the rows in LDS for the whole workgroup kept 16 rows x 4096 to one workgroup per
//     compute unit, split 16 rows x 11008 over two workgroups that each streamed the weights, and put a barrier in front
//     of the first product.)
//   * the four steps of a block times sixteen rows are the 64 dwords of one DMA instruction: a tile's scales cost one
//     instruction per block.
//   * below K = 4096 the blocks are of one to three K tiles, so that there are still up to eight waves (blocks of four throughout
//     left one or two: W2A8 16 x 8192 x 512 5.3 -> 3.3 us, 1 x 1024 x 512 2.5 -> 2.1, 16 x 8192 x 3072 5.4 -> 4.8).
//   * T is chosen so that the workgroups make one round of the compute units where the rows are worth it
//     (dtg_pick_tiles): sixteen rows of activations cost a workgroup more L2 traffic than one tile's weights.
//   * B = 2: the steps of two blocks in one unrolled round (long K); a wave's odd last block is a round of its own (as the first
//     half of a round of two, its other half repeating the last loads, W8A8 8192 x 11008 took 25.6 us instead of 20.1).
//   * the waves' partial tiles meet in LDS and are added in the order of the waves: which blocks a wave owns depends on
//     K alone, so every variant below gives the same bits.
#include <type_traits>

#include "abq_kernels.h"
#include "abq_decode_loads.h"
#include "abq_quant.h"

#ifndef ABQ_Q
#error "compile with -DABQ_Q=<x_bits> -DABQ_P=<w_bits>"
#endif

namespace abq {

// Threads an instance is compiled for: those that need more than 128 registers run with at most eight waves.
constexpr int dtg_threads(int p, int t, int b, int xm, bool g64)
{
    return g64 || p == 8 || xm == 4 || t >= 3 || (t * b >= 4 && xm != 1) || (p == 4 && b == 2 && xm == 0) ? 512 : 1024;
}

// Steps whose loads a wave has in flight beside the step it multiplies: about 6 KB of weights.  More would not be in
// flight: a compute unit's loads are served in order, and a wave that issues everything first stands at its last loads
// until the stream has come that far, with the quantisation and the products waiting behind (22016 x 4096 at one token,
// six tiles: half the kernel).
// x: bytes of activations a lane loads per step, 0 where they are quantised here.  steps: of a round; all of them where that many
// may be in flight, so that no request waits for the first loads to land, but one fewer where the quantisation stands in
// between (one token through eight layers 222 us with all of them, 208 with one fewer).
constexpr int dtg_ahead(int p, int t, int steps, int x)
{
    const int d = (x ? 44 : 24) / (t * p + x), most = (x && steps < 4) || steps == 1 ? steps : steps - 1;
    return d < 1 ? 1 : d > most ? most : d;
}

// XM: how the activations arrive.
//   0      packed records
//   1, 4   fp16 [M][K] of at most XM rows, quantised here per token, symmetric or with a zero point (a.x_dynamic = 1 or
//          2), with the formulas of the quantise-and-pack kernel (abq_quant.h): every wave loads the halves of its own
//          blocks, the row's extrema meet in LDS (one barrier), and the wave writes the int8 records of its own blocks
//          into LDS of its own.  The quantising launch in front of the GEMM and the memory round trip between the two
//          fall away.  The group sums come from the matrix core (the records times ones).
//   8      the same for any number of rows: the halves are loaded a second time for the codes instead of being held.
// XL: packed activations (XM = 0): 16-byte loads per lane and step, 1 for up to 1 KB of records, 2 for up to 2 KB.  They
// are loaded as they lie in memory, lane after lane, and brought into the operand layout through LDS of the wave's own.
// (Loaded in the operand layout neighbouring lanes would sit in different cache lines, 64 look-ups per instruction
// instead of 8, and the requests themselves became the bound: 16 x 4096 x 4096 5.3 against 4.5 us.)
// FE: rows of the result a lane folds: 1 if there is only one, else 4.
// G64: groups of 64, two to a K tile: lane groups 0, 1 hold the elements of the first, 2, 3 those of the second, and the
// matrix core sums over all four, so a step runs its two instructions twice: once on all lanes and once with the
// activations of lane groups 2, 3 zeroed; the difference is the second group's dot product.
// ONCE: requests as short as they get: weight loads without the test for a second block of rows, offsets of K tiles in 32 bits
// (dtg_once).
template <int Q, int P, bool SIGNED, int T, int B, int S, int XM, int XL, int FE, bool G64, bool ONCE>
__global__ __launch_bounds__(dtg_threads(P, T, B, XM, G64)) void gemm_decode_tiled_grouped(const GemmArgs a)
{
    static_assert(!XM || (Q == 8 && SIGNED && !G64), "in-kernel quantisation writes signed 8-bit records, groups of 128");
    constexpr int GPT = G64 ? 2 : 1;               // scale groups per K tile
    constexpr int LPS = DtgShare<P>::kLoads;       // weight loads per step and tile
    constexpr bool XS = XM == 0;
    constexpr int LPX = XS ? XL : 0;               // activation loads per step
    constexpr int SL = (S * GPT + 3) / 4;          // scale loads per block and tile
    constexpr int SC = 64 * SL;                    // floats of a tile's scales per block: [SL][16 rows][4 groups]
    constexpr int XB = XS ? Q * 256 : 0;           // XS: bytes of sixteen rows' records of a step
    extern __shared__ __align__(16) unsigned char smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int NW = blockDim.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int M = a.M, N = a.N;
    const int KT = a.K >> 7; // K tiles = steps
    const int NG = KT * GPT; // scale groups along K
    const int nblocks = (KT + S - 1) / S;
    const int tile0 = blockIdx.x * T;
    const int rows = min(M, 16);
    const int m0 = blockIdx.y * 16;
    const int Mb = min(16, M - m0);
    const int once = gridDim.y == 1; // no other workgroup reads this one's weight records (XM: always so, its rows are at most sixteen)
    const bool zp = a.w_zero != nullptr;

    // LDS: [wave][tile][row][16] partial results | per wave: scales, zero points, group sums of its blocks in flight
    // (and its int8 records) | the rows' scales and zero points, the tiles' zero-point terms | extrema of rows quantised here
    const int blocks_of_wave = XM ? (nblocks + NW - 1) / NW : 0;
    const unsigned own_bytes = B * (2 * T + 1) * SC * 4 + 2 * XB + (XM ? (unsigned)(blocks_of_wave * S * rows) * 128u : 0u);
    float *red = reinterpret_cast<float *>(smem);
    unsigned char *own = smem + (unsigned)(NW * T * rows) * 64u + (unsigned)wid * own_bytes;
    float *sws = reinterpret_cast<float *>(own);           // [B][T][SC]
    float *zws = sws + B * T * SC;                         // [B][T][SC]
    int *sxs = reinterpret_cast<int *>(zws + B * T * SC);  // [B][4 * SL groups][16 rows]
    unsigned char *xq = own + B * (2 * T + 1) * SC * 4;    // XM: [block of the wave][S][row][8 chunks], XS: [2][row][Q chunks]
    float *par = reinterpret_cast<float *>(smem + (unsigned)(NW * T * rows) * 64u + (unsigned)NW * own_bytes); // [2][64]: scales, zero points
    float *terms = par + 128;                              // [128]
    float *row_ext = terms + 128;                          // XM: [row][2][16 waves]

    // ---- byte offsets of the lane's share: weight tile t, activation row, scales --------------------------------
    uint32_t woff[T], soff[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint32_t n = (uint32_t)min((tile0 + t) * 16 + r, N - 1);
        woff[t] = n * (P * 16u) + (uint32_t)g * (4u * P);
        soff[t] = (uint32_t)min((tile0 + t) * 16 + (lane >> 2), N - 1) * (uint32_t)NG;
    }
    using Step = typename std::conditional<ONCE, uint32_t, size_t>::type; // (records lie within 4 GiB)
    const Step wstep = (Step)N * (P * 16u), xstep = (Step)M * (Q * 16u);
    // activations: chunk `lane` (and 64 + lane) of the rows' records, past the last row's end the last chunk once more
    const uint32_t xoff = (uint32_t)m0 * (Q * 16u) + (uint32_t)min(lane, Mb * Q - 1) * 16u;
    const uint32_t xoff2 = (uint32_t)m0 * (Q * 16u) + (uint32_t)min(64 + lane, Mb * Q - 1) * 16u;
    const uint32_t sumoff = (uint32_t)(m0 + min(r, Mb - 1)) * (uint32_t)NG;
    const char *Xt = reinterpret_cast<const char *>(a.X);
    const char *Wt = reinterpret_cast<const char *>(a.W);
    const bool row_zero = XM ? a.x_dynamic == 2 : a.x_zero != nullptr;
    uint32_t zp_mask = zp ? ~0u : 0u;
    if constexpr (XM != 0)
        asm volatile("" : "+v"(zp_mask));

    float facc[T][FE];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < FE; ++e)
            facc[t][e] = 0.f;
    // signed codes are fed at the top of the byte, so acc_g carries a factor 2^(16 - Q - P): the group sums get the same
    // factor (exact) and the finished sum is divided by it
    constexpr float kShift = SIGNED ? (float)(1 << (16 - Q - P)) : 1.0f;

    // what the final sum needs per row and column goes to LDS now (the oldest loads of their waves): fetched behind the K
    // loop it would put one more memory latency at the end
    if (XM == 0 && wid == 0) {
        lds_dma4(a.x_scale, (uint32_t)(m0 + min(r, Mb - 1)) * 4u, (unsigned)(size_t)par); // (lanes 0 .. 15 are read)
        if (row_zero)
            lds_dma4(a.x_zero, (uint32_t)(m0 + min(r, Mb - 1)) * 4u, (unsigned)(size_t)(par + 64));
    }
    if (row_zero && wid == NW - 1) {
#pragma unroll
        for (int i = 0; i < (T + 3) / 4; ++i)
            lds_dma4(a.w_zero_term, (uint32_t)min(tile0 * 16 + i * 64 + lane, N - 1) * 4u, (unsigned)(size_t)(terms + i * 64));
    }

    const int upr = a.K >> 3; // XM: units of eight halves per row
    // One round: the next NB of the wave's blocks, `done` of them being behind it.
    auto round = [&](int done, auto blocks_of_round) {
        constexpr int NB = decltype(blocks_of_round)::value;
        if (done) // the scales of the last round have been read before new ones land on them
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        constexpr int NS = S * NB;                         // steps of a round
        constexpr int D = dtg_ahead(P, T, NS, 4 * LPX);    // steps whose weights are requested ahead of the one multiplied
        // A step's request is its weights and, in front of them, the next step's activations, so that those have landed
        // when the step's weights have.
        auto loads_of = [](int i) { return T * LPS + (i + 1 < NS ? LPX : 0); };
        auto loads_of_steps = [&](int from, int to) { // constant after unrolling
            int n = 0;
            for (int i = from; i < to; ++i)
                n += loads_of(i);
            return n;
        };
        constexpr int WB = D + 1 < NS ? D + 1 : NS, XR = D + 2 < NS ? D + 2 : NS; // ring sizes
        DtgShare<P> wb[WB][T];
        v4u xs[XS ? XR : 1][XS ? XL : 1];
        constexpr int XH = XM == 1 || XM == 4 ? XM : 1;
        v4u xr[XH][NB];
        auto block_of = [&](int b) { return (done + b) * NW + wid; };
        // XM: the lane's unit of a block (S < 4: the further lanes repeat the last one and write nothing)
        auto unit_of = [&](int blk) { return min(blk * (16 * S) + (S == 4 ? lane : min(lane, 16 * S - 1)), upr - 1); };

        if constexpr (XM == 1 || XM == 4) {
            // the wave's own units of the rows (past the rows' end the last one once more)
#pragma unroll
            for (int m = 0; m < XH; ++m)
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    xr[m][b] = dt_load16(Xt, (uint32_t)(min(m, Mb - 1) * upr + unit_of(block_of(b))) * 16u);
        }
        // ---- scales, zero points and group sums of the blocks ----------------------------------------------------
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < SL; ++i) {
                // sixteen rows times four groups, neighbouring lanes on neighbouring groups: sixteen cache lines per instruction
                const int first = S * GPT * block_of(b) + 4 * i;
                const uint32_t grp = (uint32_t)min(first + (lane & 3), NG - 1);
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const uint32_t off = (soff[t] + grp) * 4u;
                    lds_dma4(a.w_scale, off, (unsigned)(size_t)(sws + (b * T + t) * SC + i * 64));
                    if (zp)
                        lds_dma4(a.w_zero, off, (unsigned)(size_t)(zws + (b * T + t) * SC + i * 64));
                }
                if (XM == 0 && zp)
                    lds_dma4(a.x_group_sums, (sumoff + (uint32_t)min(first + g, NG - 1)) * 4u, (unsigned)(size_t)(sxs + b * SC + i * 64));
            }
        // ---- a step's weights and the next one's activations (steps past the end of K repeat the last one) ---------------
        auto k_tile = [&](int i) { return min(S * block_of(i / S) + i % S, KT - 1); };
        auto request_acts = [&](int i) {
            const char *xp = Xt + (Step)k_tile(i) * xstep;
            if constexpr (XS) {
                xs[i % XR][0] = dt_load16(xp, xoff);
                if constexpr (XL > 1)
                    xs[i % XR][1] = dt_load16(xp, xoff2);
            }
        };
        auto request = [&](int i) {
            if (i + 1 < NS)
                request_acts(i + 1);
            const char *wp = Wt + (Step)k_tile(i) * wstep;
#pragma unroll
            for (int t = 0; t < T; ++t)
                wb[i % WB][t].template issue<ONCE>(wp, woff[t], once);
        };
        request_acts(0);
#pragma unroll
        for (int i = 0; i < D; ++i)
            request(i);

        if constexpr (XM != 0) {
            if (XM == 8 ? done == 0 : true) {
                typedef _Float16 h2 __attribute__((ext_vector_type(2)));
                auto dpp = [](float v, auto ctrl, auto row_mask) {
                    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v),
                                                                                 decltype(ctrl)::value, decltype(row_mask)::value, 0xF, false));
                };
                using std::integral_constant;
                // extremum over the sixteen lanes of a row: quads, halves of the row, the row
                auto row_max = [&](float v) {
                    v = fmaxf(v, dpp(v, integral_constant<int, 0xB1>{}, integral_constant<int, 0xF>{}));  // quad_perm [1,0,3,2]
                    v = fmaxf(v, dpp(v, integral_constant<int, 0x4E>{}, integral_constant<int, 0xF>{}));  // quad_perm [2,3,0,1]
                    v = fmaxf(v, dpp(v, integral_constant<int, 0x141>{}, integral_constant<int, 0xF>{})); // row_half_mirror
                    v = fmaxf(v, dpp(v, integral_constant<int, 0x140>{}, integral_constant<int, 0xF>{})); // row_mirror
                    return v;
                };
                // ... and over the wave, in lane 63
                auto wave_max = [&](float v) {
                    v = row_max(v);
                    v = fmaxf(v, dpp(v, integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{})); // row_bcast 15 into rows 1, 3
                    v = fmaxf(v, dpp(v, integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{})); // row_bcast 31 into rows 2, 3
                    return v;
                };
                auto unit_max = [](const v4u &u) {
                    union {
                        v4u q;
                        h2 h[4];
                    } raw;
                    raw.q = u;
                    const h2 m = __builtin_elementwise_max(__builtin_elementwise_max(raw.h[0], raw.h[1]), __builtin_elementwise_max(raw.h[2], raw.h[3]));
                    return fmaxf((float)m.x, (float)m.y);
                };
                auto reload = [&](int m, int blk) {
                    return *reinterpret_cast<const v4u *>(Xt + ((size_t)m * upr + unit_of(blk)) * 16u);
                };
                const bool symmetric = a.x_dynamic == 1;
                // symmetric: the maximum of |x| stands for both extrema; else the maxima of x and of -x
                const uint32_t keep = symmetric ? 0x7FFF7FFFu : 0xFFFFFFFFu;
                if constexpr (XM != 8) {
                    if (zp) // the halves are the oldest loads
                        dt_wait_loads_n(loads_of_steps(0, D) + 2 * NB * SL * T);
                    else
                        dt_wait_loads_n(loads_of_steps(0, D) + NB * SL * T);
#pragma unroll
                    for (int m = 0; m < XH; ++m)
#pragma unroll
                        for (int b = 0; b < NB; ++b)
                            dt_landed(xr[m][b]);
                }
                auto extrema = [&](int m, auto unit, int count) {
                    float hi = -INFINITY, lo = -INFINITY;
                    for (int b = 0; b < count; ++b) {
                        const v4u u = unit(b);
                        hi = fmaxf(hi, unit_max(v4u{ u[0] & keep, u[1] & keep, u[2] & keep, u[3] & keep }));
                        if (!symmetric)
                            lo = fmaxf(lo, unit_max(v4u{ u[0] ^ 0x80008000u, u[1] ^ 0x80008000u, u[2] ^ 0x80008000u, u[3] ^ 0x80008000u }));
                    }
                    hi = wave_max(hi);
                    if (!symmetric)
                        lo = wave_max(lo);
                    if (lane == 63) {
                        row_ext[(m * 2) * 16 + wid] = hi;
                        row_ext[(m * 2 + 1) * 16 + wid] = lo;
                    }
                };
                if constexpr (XM == 8) {
                    for (int m = 0; m < Mb; ++m)
                        extrema(m, [&](int b) { return reload(m, b * NW + wid); }, blocks_of_wave);
                } else {
#pragma unroll
                    for (int m = 0; m < XH; ++m)
                        if (m < Mb)
                            extrema(m, [&](int b) { return xr[m][b]; }, NB);
                }
                __syncthreads();
                uint32_t sel_pair, sel_half;
                quad_transpose_selectors(tid & 3, sel_pair, sel_half);
                auto params = [&](int m) {
                    const int slot = min(r, NW - 1);
                    const float hi = row_max(row_ext[(m * 2) * 16 + slot]);
                    const float lo = symmetric ? hi : row_max(row_ext[(m * 2 + 1) * 16 + slot]);
                    const QuantRow qr = quant_row_params(hi, -lo, 8, symmetric);
                    if (tid == 0) {
                        par[m] = qr.scale;
                        par[64 + m] = qr.zero_out;
                    }
                    return qr;
                };
                // eight halves of a lane -> their bytes of the row's record: the quad's four units are one word-set, whose
                // expanded dword s, byte c is element 7 - s of lane 3 - c; sixteen lanes hold a K tile
                auto quantise = [&](int m, int b, const v4u &u, const QuantRow &qr) {
                    union {
                        v4u q;
                        _Float16 h[8];
                    } raw;
                    raw.q = u;
                    int v[8];
                    if (symmetric && qr.finite) {
#pragma unroll
                        for (int c = 0; c < 8; ++c)
                            v[c] = quant_code_bits_symmetric((float)raw.h[c], qr);
                    } else {
#pragma unroll
                        for (int c = 0; c < 8; ++c)
                            v[c] = quant_code_bits((float)raw.h[c], qr);
                    }
                    uint32_t e_even = quad_transpose_bytes(pack_low_bytes(v[7], v[5], v[3], v[1]), sel_pair, sel_half);
                    uint32_t e_odd = quad_transpose_bytes(pack_low_bytes(v[6], v[4], v[2], v[0]), sel_pair, sel_half);
                    if ((b * NW + wid) * (16 * S) + lane >= upr) // past the end of K
                        e_even = e_odd = 0u;
                    const int rowi = (b * S + g) * rows + m;
                    const int dw = 8 * ((lane >> 2) & 3) + 2 * (lane & 3); // first of the lane's two dwords in the record
                    const int chunk = (dw >> 2) ^ (rowi & 7);
                    if (S == 4 || g < S)
                        *reinterpret_cast<uint2 *>(xq + ((uint32_t)rowi * 8 + chunk) * 16u + (dw & 3) * 4u) = make_uint2(e_even, e_odd);
                };
                if constexpr (XM == 8) {
                    for (int m = 0; m < Mb; ++m) {
                        const QuantRow qr = params(m);
                        for (int b = 0; b < blocks_of_wave; ++b)
                            quantise(m, b, reload(m, b * NW + wid), qr);
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < XH; ++m)
                        if (m < Mb) {
                            const QuantRow qr = params(m);
#pragma unroll
                            for (int b = 0; b < NB; ++b)
                                quantise(m, b, xr[m][b], qr);
                        }
                }
                // (the records are read by the lanes of this wave only, whose LDS operations keep their order)
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
        }

        // ---- the steps: LDS reads one step ahead of the products, the fold one step behind them -----------------------
        dt_wait_loads_n(loads_of_steps(0, D)); // older than these: the DMA loads and the first step's activations
        struct Operands {
            float sw[GPT][T], zw[GPT][T];
            int sx[GPT][FE];
            v4i av[2]; // XM, XS
        };
        struct Products {
            int lo[T][FE], hi[T][FE]; // hi: the second group of a K tile (G64)
            int sum[FE];              // XM
        };
        auto read_lds = [&](int i, Operands &s) {
            const int b = i / S, d = i % S;
            // (wave-uniform) steps past the end of K count nothing; rows quantised here have zero records there
            const bool have = !XS || S * block_of(b) + d < KT;
#pragma unroll
            for (int j = 0; j < GPT; ++j) {
                const int at = (GPT * d + j) * 16, place = ((GPT * d + j) >> 2) * 64 + r * 4 + ((GPT * d + j) & 3);
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const float sw = sws[(b * T + t) * SC + place], zw = zws[(b * T + t) * SC + place];
                    s.sw[j][t] = have ? sw : 0.f;
                    // (XM: by a mask; a select the compiler turns into a branch around the read, with a wait in it, which made one
                    // token through eight layers 218 us instead of 209)
                    s.zw[j][t] = XS ? (have && zp ? zw : 0.f) : __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, zw) & zp_mask);
                }
                if constexpr (XM == 0) {
                    if constexpr (FE == 1) {
                        s.sx[j][0] = zp ? sxs[b * SC + at] : 0;
                    } else {
                        const v4i sx = *reinterpret_cast<const v4i *>(sxs + b * SC + at + 4 * g);
#pragma unroll
                        for (int e = 0; e < FE; ++e)
                            s.sx[j][e] = zp ? sx[e] : 0;
                    }
                }
            }
            if constexpr (XS) {
                // the records as they were loaded -> the wave's LDS, chunks of a row permuted -> the operand
                auto &x = xs[i % XR];
                unsigned char *buf = xq + (i & 1) * XB;
#pragma unroll
                for (int j = 0; j < XL; ++j) {
                    dt_landed(x[j]);
                    const int c = j * 64 + lane, row = c / Q;
                    if (XL * 64 <= Q * 16 || c < Q * 16)
                        *reinterpret_cast<v4u *>(buf + (row * Q + ((c & (Q - 1)) ^ (row & (Q - 1)))) * 16) = x[j];
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const int row = min(r, Mb - 1);
                const unsigned char *xrow = buf + row * (Q * 16);
                if constexpr (Q == 8) {
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        s.av[j] = *reinterpret_cast<const v4i *>(xrow + (((2 * g + j) ^ (row & 7)) * 16));
                } else if constexpr (Q == 4) {
                    dt_unpack<4, SIGNED>(*reinterpret_cast<const v4u *>(xrow + ((g ^ (row & 3)) * 16)), s.av);
                } else {
                    const v2u xv = *reinterpret_cast<const v2u *>(xrow + (((g >> 1) ^ (row & 1)) * 16) + (g & 1) * 8);
                    s.av[0] = dtg_unpack2<SIGNED>(xv[0]);
                    s.av[1] = dtg_unpack2<SIGNED>(xv[1]);
                }
            }
            if constexpr (XM != 0) {
                const int rowi = ((XM == 8 ? done + b : b) * S + d) * rows + min(r, Mb - 1);
                const unsigned char *xrow = xq + (uint32_t)rowi * 128u;
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    s.av[j] = *reinterpret_cast<const v4i *>(xrow + (((2 * g + j) ^ (rowi & 7)) * 16u));
            }
        };
        auto multiply = [&](int i, const Operands &s, Products &p) {
            const v4i zero = v4i{ 0, 0, 0, 0 };
            v4i av[2];
            av[0] = s.av[0];
            av[1] = s.av[1];
            if constexpr (XM != 0) {
                constexpr int one = 0x01010101 << (8 - P);
                const v4i ones = v4i{ one, one, one, one };
                v4i sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[0], ones, zero, 0, 0, 0);
                sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[1], ones, sum, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < FE; ++e)
                    p.sum[e] = sum[e];
            }
            const v4i a0 = g < 2 ? av[0] : zero, a1 = g < 2 ? av[1] : zero; // G64: the first group's lanes alone
#pragma unroll
            for (int t = 0; t < T; ++t) {
                v4i bv[2];
                dtg_operands<P, SIGNED>(wb[i % WB][t], bv);
                v4i acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[0], bv[0], zero, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[1], bv[1], acc, 0, 0, 0);
                if constexpr (G64) {
                    v4i lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, bv[0], zero, 0, 0, 0);
                    lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, bv[1], lo, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < FE; ++e) {
                        p.lo[t][e] = lo[e];
                        p.hi[t][e] = acc[e] - lo[e];
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < FE; ++e)
                        p.lo[t][e] = acc[e];
                }
            }
        };
        auto fold = [&](const Operands &s, const Products &p) {
#pragma unroll
            for (int e = 0; e < FE; ++e) {
                float sx[GPT];
#pragma unroll
                for (int j = 0; j < GPT; ++j)
                    sx[j] = XM ? (float)p.sum[e] : (float)s.sx[j][e] * kShift;
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    facc[t][e] = __builtin_fmaf(s.sw[0][t], __builtin_fmaf(-s.zw[0][t], sx[0], (float)p.lo[t][e]), facc[t][e]);
                    if constexpr (G64)
                        facc[t][e] = __builtin_fmaf(s.sw[GPT - 1][t], __builtin_fmaf(-s.zw[GPT - 1][t], sx[GPT - 1], (float)p.hi[t][e]), facc[t][e]);
                }
            }
        };
        Operands ops[3];
        Products prod[2];
        read_lds(0, ops[0]);
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            if (i + D < NS)
                request(i + D);
            // (marked as landed on every path: a register with a load still in flight must not look free to the compiler)
            dt_wait_loads_n(loads_of_steps(i + 1, i + D < NS ? i + D + 1 : NS));
#pragma unroll
            for (int t = 0; t < T; ++t)
                wb[i % WB][t].landed();
            if (i + 1 < NS)
                read_lds(i + 1, ops[(i + 1) % 3]);
            multiply(i, ops[i % 3], prod[i & 1]);
            if (i)
                fold(ops[(i - 1) % 3], prod[(i - 1) & 1]);
        }
        fold(ops[(NS - 1) % 3], prod[(NS - 1) & 1]);
    };
    if constexpr (XM == 1 || XM == 4) {
        round(0, std::integral_constant<int, B>{}); // (rows held in registers: all blocks are in flight)
    } else {
        // (block b of K is the wave's if b mod NW = wid; every wave has at least one)
        int done = 0;
        for (; (done + B - 1) * NW + wid < nblocks; done += B)
            round(done, std::integral_constant<int, B>{});
        if constexpr (B > 1) // the odd one (padded to a round of two, its repeated loads made W8A8 at K = 11008 a quarter slower)
            if (done * NW + wid < nblocks)
                round(done, std::integral_constant<int, 1>{});
    }

    // ---- the waves' partial tiles meet in LDS, added in the order of the waves ---------------------------------------
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < FE; ++e)
            if (FE == 1 ? g == 0 : 4 * g + e < rows)
                red[((wid * T + t) * rows + (FE == 1 ? 0 : 4 * g + e)) * 16 + r] = facc[t][e];
    __syncthreads();
    constexpr int TS = FE == 1 ? 16 : 256; // threads a tile's results are dealt to
    for (int o = tid; o < T * TS; o += (int)blockDim.x) {
        const int t = o / TS, rem = o % TS, i = rem >> 4, c = rem & 15;
        const int n = (tile0 + t) * 16 + c;
        if (i < Mb && n < N && !(a.act && (t & 1))) {
            const float xz = row_zero ? par[64 + i] : 0.f, xsc = par[i];
            auto total = [&](int tt) {
                float v = 0.f;
#pragma unroll 4
                for (int w = 0; w < NW; ++w)
                    v += red[(w * T + tt) * rows * 16 + rem];
                v *= 1.0f / kShift;
                if (row_zero)
                    v -= xz * terms[tt * 16 + c];
                v *= xsc;
                // (rounded to fp32 here in every variant: left to itself the compiler fuses this product into the
                // conversion to fp16 in some of them, and the variants would differ in a last place now and then)
                asm("" : "+v"(v));
                return v;
            };
            const float v = total(t);
            if (T > 1 && a.act) // this tile holds gate rows, the next one their up rows
                reinterpret_cast<_Float16 *>(a.D)[(size_t)(m0 + i) * (N / 2) + (n >> 5) * 16 + c] = (_Float16)(silu(v) * total(T > 1 ? t + 1 : t));
            else
                reinterpret_cast<_Float16 *>(a.D)[(size_t)(m0 + i) * N + n] = (_Float16)v;
        }
    }
}

// ---- launch -------------------------------------------------------------------------------------------------------

// LDS of a workgroup without what the quantising variants add
static size_t dtg_lds(int nw, int t, int b, int s, int rows, bool g64)
{
    return (size_t)nw * t * rows * 64 + (size_t)nw * b * (2 * t + 1) * 256 * (g64 && s >= 3 ? 2 : 1) + 1024;
}

// instances that are built: what the registers hold
constexpr bool dtg_built(int p, int t, int b, bool g64) { return t * b * p <= (g64 && p < 8 ? 8 : 16) && t * b <= 6 && !(g64 && b == 2 && t > 1); }

// Rows quantised here, whose grid never has a second block of rows: where the short requests (ONCE) are ahead.  They bring a wave's
// weights forward against the activations every wave of the workgroup waits for, which pays where a wave requests one tile's or
// where most of the time is the stream; where two to four tiles go out in front of one block's quantisation the activations of the
// workgroup's last waves stand behind the weights of its first.  One row, us without / with: W2A8 3072 x 1792 3.80 / 3.69, 8192 x 2944
// 4.35 / 4.82, 8192 x 5504 5.6 / 5.4, 12288 x 2432 4.7 / 5.1, 22016 x 4096 8.2 / 8.1; W4A8 7424 x 2944 4.40 / 5.14.  The same one tile at
// more than eight waves (4096 x 11008 on 11: 0.95 to 0.98 of the speed), 4-bit weights on two tiles and more than a round of
// workgroups (9216 x 4608 0.94), 4-bit blocks of four K tiles (4096 x 4096 0.97 to 0.98).  Two to four rows: 2-bit weights level
// or ahead up to K = 4096, 4-bit ones to 2048, behind beyond (2 x 4096 x 6144 W4A8 0.93); 8-bit weights behind but for one row of K up
// to 2048 (4096 x 2432 0.95).
constexpr bool dtg_once(int p, int t, int s, int b, int xm, bool crowded)
{
    if (xm == 1)
        return p == 2   ? t == 1 ? !(b == 2 && crowded) : b == 2 || t == 6 || (t == 4 && s % 2 == 0)
               : p == 4 ? t == 1 ? (b == 2 ? !crowded : s < 4) : (t == 2 && b == 2 && !crowded) || (t == 4 && s < 3)
                        : t == 1 && s < 3;
    if (xm == 4)
        return b == 1 && (p == 2 || (p == 4 && s < 3));
    return xm == 8;
}

template <int Q, int P, bool SIGNED, int T, int B, int S, int XM, int XL, int FE, bool G64, bool ONCE>
static hipError_t launch_dtg_instance(const GemmArgs &a, hipStream_t stream)
{
    if constexpr (!dtg_built(P, T, B, G64)) {
        return hipErrorInvalidValue;
    } else {
        const int nw = decode_grouped_tiled_waves(a.K, P, a.group_size), rows = a.M < 16 ? a.M : 16;
        const int nblocks = (a.K / 128 + S - 1) / S;
        size_t lds = dtg_lds(nw, T, B, S, rows, G64) + (!XM && XL ? (size_t)nw * 2 * Q * 256 : 0);
        if (XM)
            lds += (size_t)nw * ((nblocks + nw - 1) / nw) * S * rows * 128 + (size_t)rows * 128;
        static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_decode_tiled_grouped<Q, P, SIGNED, T, B, S, XM, XL, FE, G64, ONCE>),
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (attr != hipSuccess)
            return attr;
        if (lds > 160 * 1024)
            return hipErrorInvalidValue;
        const int tiles = (a.N + 15) / 16;
        const dim3 grid((tiles + T - 1) / T, (a.M + 15) / 16);
        hipLaunchKernelGGL((gemm_decode_tiled_grouped<Q, P, SIGNED, T, B, S, XM, XL, FE, G64, ONCE>), grid, dim3(64 * nw), lds, stream, a);
        return hipGetLastError();
    }
}

// Tiles per workgroup, or 0 if the shape has no instance with b blocks in flight.  Up to eight packed rows the fewest:
// several workgroups on a compute unit overlap each other's phases (W2A8 12288 x 4096 at four rows 5.9 us on one tile, 6.3
// on two; gate + up at eight rows 9.4 on two, 10.0 on six).  Rows that every workgroup quantises for itself: the fewest that
// make one round of the 256 compute units (12288 x 4096 at one fp16 row 7.2 us on one, 5.8 on three; gate + up 9.3 on two, 8.2
// on six).  More than eight packed rows: by what the rounds move (12288 x 4096 at sixteen rows 8.1 us on one tile, 6.9 on three).  Workgroups of a few
// waves share a compute unit whatever their rows are (K < 1024: 16 x 8192 x 512 3.5 us on two tiles, 3.1 on one), those of
// nine waves and more (long K, more than 256 tiles) have one to themselves and take two tiles at any number of rows.
template <int P> static int dtg_pick_tiles(const GemmArgs &a, int q, int xm, bool g64, int b)
{
    const int tiles = (a.N + 15) / 16, nw = decode_grouped_tiled_waves(a.K, P, a.group_size), rows = a.M < 16 ? a.M : 16;
    const int one_round = !xm && decode_grouped_tiled_steps(a.K) == 1 && nw < 8 ? (nw > 2 ? 512 : 1024) : 256;
    const int choices[5] = { 1, 2, 3, 4, 6 };
    int best = 0;
    long best_cost = 0;
    for (int c : choices) {
        // (a single row and the variants that hold several rows have instances of one and two tiles, unless they quantise)
        if (!dtg_built(P, c, b, g64) || (a.act && (c & 1)) || dtg_lds(nw, c, b, 4, rows, g64) > 120 * 1024 || 64 * nw > dtg_threads(P, c, b, xm, g64) ||
            (xm >= 4 && c > 2) || (xm == 8 && b > 1))
            continue;
        const int rounds = ((tiles + c - 1) / c + one_round - 1) / one_round;
        if (!xm && a.M > 8) {
            // weights from memory, activations from L2, which is about three times as fast
            const long cost = (long)rounds * (3 * c * P * 256 + rows * q * 16);
            if (best == 0 || cost <= best_cost) {
                best = c;
                best_cost = cost;
            }
            continue;
        }
        best = c;
        if ((!xm && !(nw > 8 && b == 1 && c == 1)) || rounds == 1)
            break;
    }
    return best;
}

template <int Q, int P, bool SIGNED, bool XDYN, bool G64> static hipError_t launch_dtg(const GemmArgs &a, hipStream_t stream)
{
    const int steps = decode_grouped_tiled_steps(a.K);
    const int nblocks = (a.K / 128 + steps - 1) / steps, nw = decode_grouped_tiled_waves(a.K, P, a.group_size);
    const int per_wave = (nblocks + nw - 1) / nw;
    // two blocks of a wave in flight where it has two and there is an instance, else one after the other; rows held in
    // registers need all of a wave's blocks in flight
    int b = per_wave >= 2 ? 2 : 1;
    int xm = !XDYN ? 0 : per_wave > 2 || a.M > 4 ? 8 : a.M > 1 ? 4 : 1;
    if (xm == 8)
        b = 1;
    // Nor on more than two workgroups per compute unit, or more than one where the registers of two blocks (groups of 64) or
    // their waves (more than eight) leave no room for a second workgroup beside the first: W2A8 at one row 5120 x 13824 9.9 ->
    // 8.3 us on two tiles of one block, 8192 x 11008 9.4 -> 7.2, groups of 64 12288 x 5120 9.2 -> 7.0; at five rows 27648 x 5120
    // 17.4 -> 13.7; at 16 rows of groups of 64 8192 x 11008 17.6 -> 12.8.
    const int tiles = (a.N + 15) / 16;
    if (!xm && (tiles > 512 || (tiles > 256 && (nw > 8 || G64))))
        b = 1;
    int t = dtg_pick_tiles<P>(a, Q, xm, G64, b);
    if (t == 0 && b == 2) {
        b = 1;
        if (XDYN)
            xm = 8;
        t = dtg_pick_tiles<P>(a, Q, xm, G64, b);
    }
    auto go = [&](auto tt, auto bb, auto ss) -> hipError_t {
        constexpr int TT = decltype(tt)::value, BB = decltype(bb)::value, SS = decltype(ss)::value;
        if constexpr (XDYN) {
            if (xm == 1) {
                constexpr bool sparse_once = dtg_once(P, TT, SS, BB, 1, false), crowded_once = dtg_once(P, TT, SS, BB, 1, true);
                if (sparse_once != crowded_once && (TT == 1 ? nw > 8 : (tiles + TT - 1) / TT > 256))
                    return launch_dtg_instance<Q, P, SIGNED, TT, BB, SS, 1, 0, 1, false, crowded_once>(a, stream);
                return launch_dtg_instance<Q, P, SIGNED, TT, BB, SS, 1, 0, 1, false, sparse_once>(a, stream);
            }
            if constexpr (TT <= 2) {
                if (xm == 4)
                    return launch_dtg_instance<Q, P, SIGNED, TT, BB, SS, 4, 0, 4, false, dtg_once(P, TT, SS, BB, 4, false)>(a, stream);
                if constexpr (BB == 1)
                    return launch_dtg_instance<Q, P, SIGNED, TT, 1, SS, 8, 0, 4, false, dtg_once(P, TT, SS, 1, 8, false)>(a, stream);
            }
            return hipErrorInvalidValue;
        } else {
            if (a.M == 1) {
                if constexpr (TT <= 2)
                    return launch_dtg_instance<Q, P, SIGNED, TT, BB, SS, 0, 1, 1, G64, false>(a, stream);
                return hipErrorInvalidValue;
            }
            if constexpr (Q == 8) {
                if (a.M > 8)
                    return launch_dtg_instance<Q, P, SIGNED, TT, BB, SS, 0, 2, 4, G64, false>(a, stream);
            }
            return launch_dtg_instance<Q, P, SIGNED, TT, BB, SS, 0, 1, 4, G64, false>(a, stream);
        }
    };
    using std::integral_constant;
    auto with_b = [&](auto tt) -> hipError_t {
        constexpr integral_constant<int, 1> one{};
        if (steps < 4) // (a wave then has one block)
            return steps == 1 ? go(tt, one, one) : steps == 2 ? go(tt, one, integral_constant<int, 2>{}) : go(tt, one, integral_constant<int, 3>{});
        return b == 2 ? go(tt, integral_constant<int, 2>{}, integral_constant<int, 4>{}) : go(tt, one, integral_constant<int, 4>{});
    };
    switch (t) {
    case 1: return with_b(integral_constant<int, 1>{});
    case 2: return with_b(integral_constant<int, 2>{});
    case 3: return with_b(integral_constant<int, 3>{});
    case 4: return with_b(integral_constant<int, 4>{});
    case 6: return with_b(integral_constant<int, 6>{});
    default: return hipErrorInvalidValue;
    }
}

template <int Q, int P, bool SIGNED, bool XDYN = false> static hipError_t launch_decode_tiled_grouped(const GemmArgs &a, hipStream_t stream)
{
    if ((a.group_size != 128 && !(a.group_size == 64 && !XDYN)) || !a.w_scale || (!XDYN && !a.x_scale) || (size_t)a.N * a.K * P / 8 >= (1ull << 32) ||
        (size_t)a.M * a.K * Q / 8 >= (1ull << 32) || (XDYN && (a.x_dynamic < 1 || a.x_dynamic > 2 || (a.x_dynamic == 2 && !a.w_zero_term))))
        return hipErrorInvalidValue;
    if (XDYN && ((size_t)a.M * a.K > 16384 || a.M > 16))
        return hipErrorInvalidValue;
    if (a.act && a.N % 32 != 0)
        return hipErrorInvalidValue;
    if constexpr (!XDYN) {
        if (a.group_size == 64)
            return launch_dtg<Q, P, SIGNED, false, true>(a, stream);
    }
    return launch_dtg<Q, P, SIGNED, XDYN, false>(a, stream);
}

#define ABQ_ONE_FIELD(b) (b == 2 || b == 4 || b == 8)
#if ABQ_ONE_FIELD(ABQ_Q) && ABQ_ONE_FIELD(ABQ_P)
// one entry: the launcher picks waves, loads in flight and tiles by shape
static const KernelEntry kSigned[] = { { 16, 1, 1, 1, 1, 16, 6, &launch_decode_tiled_grouped<ABQ_Q, ABQ_P, true>, 128 } };
#define ABQ_DTG_NSIGNED 1
#else
static const KernelEntry *const kSigned = nullptr;
#define ABQ_DTG_NSIGNED 0
#endif
#if ABQ_Q < 8 && ABQ_DTG_NSIGNED
static const KernelEntry kUnsigned[] = { { 16, 1, 1, 1, 1, 16, 6, &launch_decode_tiled_grouped<ABQ_Q, ABQ_P, false>, 128 } };
#define ABQ_DTG_NUNSIGNED 1
#else
static const KernelEntry *const kUnsigned = nullptr;
#define ABQ_DTG_NUNSIGNED 0
#endif
// ... and the same quantising fp16 activations per token itself (8-bit activations)
#if ABQ_Q == 8 && ABQ_DTG_NSIGNED
static const KernelEntry kDyn[] = { { 16, 1, 1, 1, 1, 16, 6, &launch_decode_tiled_grouped<ABQ_Q, ABQ_P, true, true>, 128 } };
#define ABQ_DTG_NDYN 1
#else
static const KernelEntry *const kDyn = nullptr;
#define ABQ_DTG_NDYN 0
#endif

#define ABQ_CAT_(a, b, c, d) a##b##c##d
#define ABQ_CAT(a, b, c, d) ABQ_CAT_(a, b, c, d)

void ABQ_CAT(abq_decode_tiled_grouped_register_, ABQ_Q, _, ABQ_P)(KernelTable *out)
{
    out[0] = KernelTable{ ABQ_Q, ABQ_P, 1, kSigned, ABQ_DTG_NSIGNED };
    out[1] = KernelTable{ ABQ_Q, ABQ_P, 0, kUnsigned, ABQ_DTG_NUNSIGNED };
}

void ABQ_CAT(abq_decode_tiled_grouped_dyn_register_, ABQ_Q, _, ABQ_P)(KernelTable *out)
{
    out[0] = KernelTable{ ABQ_Q, ABQ_P, 1, kDyn, ABQ_DTG_NDYN };
    out[1] = KernelTable{ ABQ_Q, ABQ_P, 0, nullptr, 0 };
}

} // namespace abq
