// Numbering of the output tiles of the prefill kernels: which tile a workgroup takes, and how many workgroups a launch has.  Needs
// nothing of the GPU but the two functions marked for it, so that a test compiles it for the host.
#pragma once
#include <stdint.h>

namespace abq {

// Workgroup id -> output tile.  XCD x = id % 8 owns n blocks [x * npx, (x + 1) * npx); inside an XCD the
// workgroups run through groups of four m blocks, M fastest inside a group, then N, then the next group:
// the 32 or 64 workgroups an XCD runs at a time then cover a patch of 4 x 8 (or 4 x 16) tiles, so every
// activation and weight block they load is shared in that XCD's L2, whatever M is (with M fastest over
// all m blocks, 16384 rows ran 25-35 % slower; groups of 2, 4 and 8 measured within 2 %, 4 ahead by up
// to 4 % at 2048 rows).
// Where whole columns of tiles would give some XCDs a good deal more than their share (tiles_spread), an XCD owns n_blocks / 8 of
// them, and the tiles of the n_blocks % 8 that are left are dealt out evenly: behind every eight m blocks of its own an XCD takes an
// eighth of theirs, in runs of consecutive m blocks, whose activations it has just read.
constexpr int kSpreadM = 8;
// Where the XCD with the most columns has at least a round of its 32 compute units, and an eighth, more than its share: 9 columns
// are 2 for four of the XCDs and none for three (decoder-layer linears, W2A8 groups of 128: hidden 1152 8192 rows 615 -> 581 us, W4A4
// 535 -> 505; hidden 2176 1476 -> 1392; 12000 rows of 1536 1173 -> 1134).  Below that the tiles dealt out cost what they save: 2048
// rows of 1408 253 -> 259; W4A4 with one scale, 4096 rows of 1152, 145 -> 150; 86 columns of 16 tiles of the FP6 kernel 68.0 -> 70.5.
inline bool tiles_spread(int m_blocks, int n_blocks)
{
    const long most = (n_blocks + 7) / 8;
    return (8 * most - n_blocks) * m_blocks >= 256 && 8 * 8 * most > 9l * n_blocks;
}

// What the kernels are told of the columns of tiles: columns of an XCD, or minus all columns where they are spread.
inline int tile_columns(int m_blocks, int n_blocks) { return tiles_spread(m_blocks, n_blocks) ? -n_blocks : (n_blocks + 7) / 8; }

// n / d for n below 2^31 and d in 1 .. 4, without a branch
__device__ __forceinline__ int div_small(int n, int d)
{
    const uint32_t m = d == 2 ? 0x80000000u : d == 3 ? 0x55555556u : 0x40000000u; // 2^32 / d, rounded up
    const int q = (int)(((uint64_t)(uint32_t)n * m) >> 32);
    return d == 1 ? n : q;
}

// Returns false for workgroups of a grid (tile_grid) that are left without a tile; a column past the last one (N) has none either.
// (A division by a number the compiler does not know is some 40 instructions in front of a workgroup's first load; grids of up to four
// m blocks have none.)
__device__ __forceinline__ bool tile_of_workgroup(int id, int m_blocks, int columns, int *mb, int *nb)
{
    constexpr int GM = 4;
    const int xcd = id & 7, slot = id >> 3;
    if (__builtin_expect(columns >= 0, 1)) {
        const int per_group = GM * columns;
        const int grp = __builtin_expect(m_blocks > GM, 0) ? slot / per_group : 0, in = slot - grp * per_group;
        const int gm = min(GM, m_blocks - grp * GM); // the last group may be short
        const int col = div_small(in, gm);
        *mb = grp * GM + in - col * gm;
        *nb = xcd * columns + col;
        return true;
    }
    const int npx = -columns >> 3, left = -columns & 7;
    const int per_super = kSpreadM * npx + left; // an XCD's tiles of eight m blocks
    const int sup = slot / per_super, in = slot - sup * per_super;
    const int sm = min(kSpreadM, m_blocks - sup * kSpreadM); // the last ones may be fewer
    if (in < sm * npx) {
        const int per_group = GM * npx;
        const int grp = in >= per_group ? 1 : 0, pos = in - grp * per_group;
        const int gm = min(GM, sm - grp * GM), col = div_small(pos, gm);
        *mb = sup * kSpreadM + grp * GM + pos - col * gm;
        *nb = xcd * npx + col;
        return true;
    }
    const int rest = left * sm, u = xcd * ((rest + 7) >> 3) + in - sm * npx;
    if (u >= rest)
        return false;
    *mb = sup * kSpreadM + u % sm;
    *nb = 8 * npx + u / sm;
    return true;
}

// Workgroups of a launch over m_blocks x n_blocks tiles numbered like that.
inline unsigned tile_grid(int m_blocks, int n_blocks)
{
    if (!tiles_spread(m_blocks, n_blocks))
        return 8u * (((unsigned)n_blocks + 7) / 8) * (unsigned)m_blocks;
    const unsigned npx = (unsigned)n_blocks / 8, left = (unsigned)n_blocks % 8, last = (unsigned)m_blocks % kSpreadM;
    return 8u * ((unsigned)(m_blocks / kSpreadM) * (kSpreadM * npx + left) + last * npx + (last * left + 7u) / 8u);
}

} // namespace abq
