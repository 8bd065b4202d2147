"""CPU tests of what a call launches (kernel, grid, workgroup, LDS) and of what its state says it will, with launches written
down instead of made."""
import re

import pytest

from launch_probe import launches


def staged64(kernel):
    """bits, signedness and K groups of the 64x64 tile's kernel on records without group scales (its LDS stages left out)"""
    m = re.fullmatch(r"gemm_mfma_staged<(\d), (\d), (true|false), false, 1, 1, 2, 2, \d, false, (\d)>", kernel)
    return m and (int(m[1]), int(m[2]), m[3] == "true", int(m[4]))


def tile64(q, p, signed, groups):
    return "AqBMMA_%dx%dx%s_64x64x%d_32x32x128_32x32x32_4" % (q, p, "true" if signed else "false", 128 * groups)


def runs_what_it_says(r):
    (made,) = r["launches"]
    return r["status"] == 0 and (made["grid"], made["block"], made["lds"]) == (r["grid"], r["block"], r["lds"])


@pytest.mark.parametrize("q,p", [(8, 2), (8, 4), (4, 4), (2, 2)])
def test_a_64x64_tile_runs_with_the_k_groups_it_names(tmp_path, q, p):
    for signed in (1, 0):
        groups = (1, 2, 4) if signed or q < 8 else (1, 4)  # (unsigned 8-bit operands have no tile of two groups)
        sums = {} if signed or q < 8 else {"row_sums": (0, 0xB00000)}
        # one shape on which four groups are the library's choice, one on which they are not
        calls = [dict(q=q, p=p, signed=signed, M=128, N=5120, K=k, tile=tile64(q, p, signed, g), **sums) for g in groups for k in (13824, 2048)]
        for c, r in zip(calls, launches(tmp_path, calls)):
            g = int(c["tile"].split("x64x")[1].split("_")[0]) // 128
            assert runs_what_it_says(r), (c, r)
            assert r["tile"] == c["tile"] and r["block"] == [256 * g, 1, 1]
            assert staged64(r["launches"][0]["kernel"]) == (q, p, bool(signed), g), r


def test_four_k_groups_are_picked_on_long_k_while_compute_units_are_free(tmp_path):
    at = lambda groups, q, p, signed, N, K, **c: (groups, dict(q=q, p=p, signed=signed, M=128, N=N, K=K, **c))  # noqa: E731
    sums = {"row_sums": (0, 0xB00000)}
    cases = [at(4, 8, 4, 1, 6144, 8192), at(2, 8, 4, 1, 6208, 8192), at(2, 8, 4, 1, 6144, 8064), at(4, 4, 2, 0, 4096, 11008),
             at(4, 8, 2, 1, 3584, 8192), at(2, 8, 2, 1, 3648, 8192), at(4, 8, 2, 0, 6144, 4096, **sums),
             at(4, 8, 4, 0, 6144, 4096, **sums), at(1, 8, 4, 0, 6144, 3968, **sums), at(1, 8, 4, 0, 6208, 4096, **sums)]
    for (groups, c), r in zip(cases, launches(tmp_path, [c for _, c in cases])):
        assert runs_what_it_says(r) and r["tile"] == tile64(c["q"], c["p"], c["signed"], groups), (c, r)


def test_unsigned_8_bit_operands_take_four_k_groups_once_their_row_sums_are_there(tmp_path):
    c = dict(q=8, p=4, signed=0, M=128, N=5120, K=5120)
    planes = dict(c, layouts=(0, 0))
    calls = [c, dict(c, row_sums=(0, 0xB00000)), dict(c, row_sums=(0, 0xB00000), order=["row_sums", "layouts"]),
             dict(c, tile=tile64(8, 4, 0, 4)), dict(planes, workspace=1 << 30), dict(planes, layouts=(0, 1), row_sums=(0, 0xB00000), workspace=1 << 30)]
    none, after, before, asked, from_planes, mixed = launches(tmp_path, calls)
    plain = "gemm_mfma_tiled<8, 4, false, 1, 1, false, 128, 2, 2>"
    assert none["launches"][0]["kernel"] == plain and none["tile"] == tile64(8, 4, 0, 1) and none["block"] == [256, 1, 1]
    for r in (after, before):
        assert runs_what_it_says(r) and r["tile"] == tile64(8, 4, 0, 4)
    assert asked["launches"][0]["kernel"] == plain  # (the same integers without the sums)
    for r in (from_planes, mixed):
        assert r["status"] == 0 and staged64(r["launches"][-1]["kernel"]) == (8, 4, False, 4) and r["tile"] == tile64(8, 4, 0, 4), r
