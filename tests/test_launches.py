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


ROWS = "AqBMMA_8x%dxtrue_64x16x4096_64x16x512_16x16x64_7"


def rows_kernel(r):
    return r["launches"][-1]["kernel"].startswith("gemm_rows_grouped<")


@pytest.mark.parametrize("order", [["layouts", "scales", "zeros", "act"], ["scales", "layouts", "act", "zeros"], ["scales", "zeros", "act", "layouts"]])
def test_states_of_17_rows_and_more_describe_the_kernel_that_runs(tmp_path, order):
    shapes = [(8, 4, 43, 4096, 4096), (8, 4, 43, 12288, 4096), (8, 4, 43, 22016, 4096), (8, 2, 128, 4096, 4096), (8, 2, 32, 4096, 11008),
              (8, 8, 96, 4096, 4096), (8, 2, 17, 4096, 1024)]
    calls = [dict(q=q, p=p, signed=1, M=m, N=n, K=k, group=128, zeros=z, act=act, order=order)
             for q, p, m, n, k in shapes for z in (0, 1) for act in (0, 1)]
    for c, r in zip(calls, launches(tmp_path, calls)):
        assert rows_kernel(r) and runs_what_it_says(r), (c, r)


@pytest.mark.parametrize("p,m,n", [(2, 128, 4096), (4, 43, 4096), (8, 64, 4096), (4, 64, 12288)])
def test_a_measured_tile_replaces_the_kernel_for_17_rows_only_where_that_was_measured_too(tmp_path, p, m, n):
    k = 4096
    tile = "AqBMMA_8x%dxtrue_128x64x128_64x32x128_32x32x32_4" % p
    entry = lambda name, tops, group=128: "%s %d %d %d %d %s" % (name, m, n, k, group, tops)  # noqa: E731
    rows = ROWS % p
    by_rule, tile_only, tile_ahead, rows_ahead, no_group = launches(tmp_path, [
        dict(q=8, p=p, signed=1, M=m, N=n, K=k, group=128, tuning=t)
        for t in ([], [entry(tile, 500)], [entry(tile, 500), entry(rows, 400)], [entry(rows, 500), entry(tile, 400)])] +
        [dict(q=8, p=p, signed=1, M=m, N=n, K=k, tuning=[entry(rows, 900, 0)])])
    assert rows_kernel(by_rule) == (n == 4096)
    assert rows_kernel(tile_only) == rows_kernel(by_rule)
    assert rows_kernel(rows_ahead) and runs_what_it_says(rows_ahead)
    assert not rows_kernel(tile_ahead) and tile_ahead["tile"] == tile and runs_what_it_says(tile_ahead)
    assert no_group["status"] == 0 and not rows_kernel(no_group)  # (the entry names a kernel that needs group scales)


def test_the_kernel_for_17_rows_runs_by_its_name(tmp_path):
    ask = lambda p=4, **c: dict(dict(q=8, p=p, signed=1, M=300, N=4096, K=512, tile=ROWS % p, group=128), **c)  # noqa: E731
    calls = [ask(p, M=m, zeros=z) for p in (2, 4, 8) for m in (17, 300) for z in (0, 1)]
    for c, r in zip(calls, launches(tmp_path, calls)):
        assert rows_kernel(r) and runs_what_it_says(r) and r["tile"] == c["tile"], (c, r)
    # refused: 16 rows, groups of 64, no group scales, other pairs, another tuple
    few, g64, bare, pair, other = launches(tmp_path, [ask(M=16), ask(group=64), ask(group=0), ask(tile="AqBMMA_4x4xtrue" + ROWS[len("AqBMMA_8x%dxtrue"):], q=4),
                                                      ask(tile=(ROWS % 4).replace("64x16x4096", "64x32x4096").replace("64x16x512", "64x32x512"))])
    assert [r["status"] for r in (few, g64, pair, other)] == [3, 3, 3, 3] and bare["status"] == 4 and not bare["launches"]


@pytest.mark.parametrize("p,group", [(2, 128), (8, 128), (4, 64)])
def test_group_scale_decode_keeps_eight_waves_down_to_1024(tmp_path, p, group):
    """Blocks of four K tiles throughout left one or two waves there.  Above, waves of two blocks; odd counts where no more waves fit."""
    waves = {256: 2, 512: 4, 640: 5, 1024: 8, 1152: 5, 2048: 8, 2944: 8, 4096: 8, 5120: 5, 11008: 11 if p < 8 and group == 128 else 8}
    calls = [dict(q=8, p=p, signed=1, M=m, N=4096, K=k, group=group, zeros=z) for k in waves for m in (1, 8, 16) for z in (0, 1)]
    for c, r in zip(calls, launches(tmp_path, calls)):
        (made,) = r["launches"]
        assert made["kernel"].startswith("gemm_decode_tiled_grouped<") and made["block"] == [64 * waves[c["K"]], 1, 1], (c, made)


def test_the_plan_for_17_rows_counts_rounds_per_xcd(tmp_path):
    """22 sets of three tiles by eleven blocks of rows are 242 workgroups, but six of the eight XCDs would run 33 on 32 compute units."""
    (r,) = launches(tmp_path, [dict(q=8, p=4, signed=1, M=700, N=1024, K=4096, tile=ROWS % 4, group=128, zeros=1)])
    assert r["launches"][0]["kernel"] == "gemm_rows_grouped<4, 4, 4, true>"


def test_the_kernel_for_17_rows_is_bounded_in_rows(tmp_path):
    shape = lambda m, n, k, p=4: dict(q=8, p=p, signed=1, M=m, N=n, K=k, group=128, zeros=1)  # noqa: E731
    on = [shape(43, 4096, 4096), shape(128, 4096, 4096), shape(512, 1024, 4096), shape(32, 12288, 1024), shape(512, 1024, 1024), shape(1024, 256, 4096),
          shape(2048, 128, 1024)]
    off = [shape(700, 1024, 4096), shape(1400, 512, 4096), shape(5000, 128, 4096), shape(192, 3072, 1024), shape(43, 12288, 1024), shape(513, 1024, 4096)]
    for c, r in zip(on + off, launches(tmp_path, on + off)):
        assert rows_kernel(r) == (c in on) and runs_what_it_says(r), (c, r)


def test_no_decode_records_above_128_rows(abq):
    for p in (2, 4, 8):
        for n, k in ((128, 4096), (512, 4096), (1024, 4096), (4096, 4096), (4096, 11008)):
            for m in (129, 200, 700, 1400, 5000):
                assert not abq.prepared_decode_pays(8, p, True, m, n, k, 128)
    assert abq.prepared_decode_pays(8, 4, True, 128, 4096, 4096, 128)


@pytest.mark.parametrize("q,p", [(8, 8), (8, 4)])
def test_k_is_split_over_workgroups_only_where_the_row_sums_are_there(tmp_path, q, p):
    """Unsigned 8-bit operands without the weights' row sums run the kernel that gathers them, which does not split K: on the tile the
    library's rules give it."""
    c = dict(q=q, p=p, signed=0, M=128, N=5120, K=13824, layouts=(0, 1), workspace=1 << 30)
    without, with_sums = launches(tmp_path, [c, dict(c, row_sums=(0, 0xB00000))])
    made = without["launches"][-1]
    assert made["kernel"] == "gemm_mfma_tiled<%d, %d, false, 1, 1, false, 128, 2, 2>" % (q, p), without
    assert without["tile"] == tile64(q, p, 0, 1) and made["grid"] == without["grid"]
    assert with_sums["launches"][-1]["kernel"].startswith("gemm_mfma_staged_parts<%d, %d, false, " % (q, p)), with_sums


def parts_tile(q, p, signed):
    return "AqBMMA_%dx%dx%s_128x64x%d_64x32x128_32x32x32_8" % (q, p, "true" if signed else "false", 256 if q + p <= 8 else 128)


def split(r):
    """workgroups per output tile of the call's GEMM, None if one that the state does not describe ran"""
    convert, made = r["launches"]
    if r["status"] or (made["grid"], made["block"], made["lds"]) != (r["grid"], r["block"], r["lds"]) or not convert["kernel"].startswith("relayout_planes"):
        return None
    parts = made["kernel"].startswith("gemm_mfma_staged_parts<")
    return made["grid"][0] // (8 * -(-r["N"] // 512) * -(-r["M"] // 128)) if parts else 1


# (rows, columns, K) -> parts per pair, on either side of the rule's lines: three quarters of the blocks of rows, four of them, 85 tiles, K tiles
# per part, eight parts
SPLITS = [((192, 200, 13824), {(8, 8): 6, (8, 4): 3, (4, 4): 3, (4, 2): 3, (2, 2): 3, (8, 2): 1}), ((191, 200, 13824), {(8, 8): 1, (8, 4): 1, (4, 4): 1, (2, 2): 1}),
          ((512, 640, 8320), {(8, 8): 4, (8, 4): 1}), ((513, 640, 8320), {(8, 8): 1}), ((128, 5440, 7168), {(8, 8): 3, (8, 4): 1}), ((128, 5504, 7168), {(8, 8): 1}),
          ((200, 200, 10752), {(8, 8): 5, (8, 4): 3, (4, 4): 3, (2, 2): 3}), ((200, 200, 10624), {(8, 8): 5, (8, 4): 1, (4, 4): 1, (2, 2): 1}),
          ((256, 64, 16512), {(8, 8): 8, (8, 4): 4, (4, 4): 4}), ((97, 2600, 10880), {(8, 8): 5, (8, 4): 3})]


@pytest.mark.parametrize("signed", [1, 0])
def test_states_on_parts_of_k_describe_the_kernel_that_runs(tmp_path, signed):
    cases = [(parts, dict(q=q, p=p, signed=signed, M=m, N=n, K=k, layouts=(0, 1), workspace=1 << 30, **({} if signed or 8 not in (q, p) else {"row_sums": (0, 0xB00000)})))
             for (m, n, k), pairs in SPLITS for (q, p), parts in pairs.items()]
    orders = [["layouts", "row_sums", "workspace"], ["row_sums", "workspace", "layouts"], ["workspace", "layouts", "row_sums"]]
    cases = [(parts, dict(c, order=o)) for parts, c in cases for o in orders]
    for (parts, c), r in zip(cases, launches(tmp_path, [c for _, c in cases])):
        assert split(dict(r, **c)) == parts, (c, r)
        assert (r["tile"] == parts_tile(c["q"], c["p"], signed)) == (parts > 1), (c, r)


def test_parts_of_k_are_left_again(tmp_path):
    """A state on that tile moves back when a later declaration takes away what it needs."""
    c = dict(q=8, p=8, signed=0, M=128, N=5120, K=13824, layouts=(0, 1), workspace=1 << 30, row_sums=(0, 0xB00000))
    sums_gone, both_tiled = launches(tmp_path, [dict(c, then=[["row_sums", [0, 0]]]), dict(c, signed=1, then=[["layouts", [1, 1]]])])
    assert sums_gone["tile"] == tile64(8, 8, 0, 1) and sums_gone["launches"][-1]["kernel"].startswith("gemm_mfma_tiled<8, 8, false, 1, 1, ")
    assert runs_what_it_says(both_tiled) and both_tiled["tile"] == tile64(8, 8, 1, 1)


def test_parts_of_k_run_by_name(tmp_path):
    ask = lambda q, p, signed, **c: dict(dict(q=q, p=p, signed=signed, M=128, N=5120, K=13824, tile=parts_tile(q, p, signed), layouts=(0, 1),  # noqa: E731
                                              workspace=1 << 30), **c)
    sums = {"row_sums": (0, 0xB00000)}
    cases = [(3, ask(8, 8, 1)), (3, ask(8, 2, 1)), (3, ask(4, 2, 0)), (3, ask(8, 4, 0, **sums)), (2, ask(8, 8, 1, M=256, N=4096, K=4096)), (8, ask(4, 4, 1, M=3, N=64, K=28672))]
    for (parts, c), r in zip(cases, launches(tmp_path, [c for _, c in cases])):
        assert split(dict(r, **c)) == parts and r["tile"] == c["tile"], (c, r)
    plain, narrow, short, wide, odd, records, scaled, fp16 = launches(tmp_path, [
        ask(8, 8, 0), ask(8, 8, 1, tile=parts_tile(8, 8, 1).replace("128x64x128", "128x64x256")), ask(8, 8, 1, K=3968), ask(8, 8, 1, M=2048), ask(6, 6, 1),
        ask(8, 8, 1, layouts=(1, 1)), ask(8, 8, 1, group=128), ask(8, 8, 1, out_kind=3)])
    assert plain["status"] == 0 and plain["launches"][-1]["kernel"] == "gemm_mfma_tiled<8, 8, false, 2, 1, false, 128, 2, 2>"  # (no sums: the same tile, one part)
    assert [r["status"] for r in (narrow, short, wide, odd, records, scaled, fp16)] == [3] * 7


@pytest.mark.parametrize("out_kind", [1, 2, 3])
def test_halves_are_never_added_in_parts(tmp_path, out_kind):
    (r,) = launches(tmp_path, [dict(q=8, p=8, signed=1, M=128, N=5120, K=13824, layouts=(0, 1), workspace=1 << 30, out_kind=out_kind)])
    assert r["tile"] == tile64(8, 8, 1, 1) and r["launches"][-1]["kernel"].startswith("gemm_mfma_staged<") and r["grid"] == [160, 1, 1]


def test_a_measured_tile_comes_before_parts_of_k(tmp_path):
    c = dict(q=8, p=8, signed=1, M=128, N=4096, K=8192, layouts=(0, 1), workspace=1 << 30)
    entry = lambda name, tops: "%s 128 4096 8192 0 %s" % (name, tops)  # noqa: E731
    tile, parts = "AqBMMA_8x8xtrue_128x64x256_64x32x128_32x32x32_4", parts_tile(8, 8, 1)
    decode = "AqBMMA_8x8xtrue_16x32x512_16x32x64_16x16x64_6"
    by_rule, by_tile, behind, ahead, elsewhere, other_m, decoding = launches(tmp_path, [dict(c, tuning=t) for t in (
        [], [entry(tile, 500)], [entry(parts, 400), entry(tile, 500)], [entry(parts, 500), entry(tile, 400)], [entry(tile, 500).replace("4096", "4224")])] +
        [dict(c, M=90, tuning=[entry(parts, 500)]), dict(c, tuning=[entry(decode, 500)])])
    for r in (by_rule, ahead, elsewhere):
        assert split(dict(r, **c)) == 4 and r["tile"] == parts, r
    for r in (by_tile, behind):
        assert split(dict(r, **c)) == 1 and r["tile"] == tile, r
    assert split(dict(other_m, **dict(c, M=90))) == 4  # (an entry serves the rows of its bucket, where the rule would not split)
    assert decoding["tile"] == decode and decoding["launches"][-1]["kernel"].startswith("gemm_decode_tiled<")
    # an entry of the split tile says nothing of calls it does not run: activations as records, halves, row sums that are not there
    rest = [dict(c, layouts=(1, 1)), dict(c, out_kind=3), dict(c, signed=0)]
    entries = [entry(parts, 500), entry(parts_tile(8, 8, 0), 500)]
    for c_, with_entry, without in zip(rest, launches(tmp_path, [dict(r, tuning=entries) for r in rest]), launches(tmp_path, rest)):
        assert with_entry["status"] == 0 and with_entry["tile"] == without["tile"] and with_entry["launches"] == without["launches"], c_


def test_the_compiled_in_table_holds_parts_of_k_where_they_were_measured(tmp_path):
    calls = [dict(q=q, p=p, signed=s, M=128, N=5120, K=13824, layouts=(0, 1), workspace=1 << 30, builtin=True, **({} if s or q < 8 else {"row_sums": (0, 0xB00000)}))
             for q, p in ((2, 2), (4, 4), (4, 2), (8, 8), (8, 4), (8, 2)) for s in (1, 0)]
    for c, r in zip(calls, launches(tmp_path, calls)):
        assert split(dict(r, **c)) == 3 and r["tile"] == parts_tile(c["q"], c["p"], c["signed"]), (c, r)


def test_unsigned_w2a6_states_describe_the_padded_kernel_that_runs(tmp_path):
    """From a workspace that holds 8-bit activation records on, whatever the order of the declarations, until it is taken away; a measured
    tile of the pair itself comes first unless the padded pair's was measured ahead."""
    c = dict(q=6, p=2, signed=0, M=128, N=4096, K=5120, layouts=(0, 1), workspace=128 * 5120)
    own, padded = "AqBMMA_6x2xfalse_64x64x128_32x32x128_32x32x32_4", "AqBMMA_8x2xfalse_64x64x512_32x32x128_32x32x32_4"
    entry = lambda name, tops: "%s 128 4096 5120 0 %s" % (name, tops)  # noqa: E731
    wide = [c, dict(c, order=["workspace", "layouts"]), dict(c, out_kind=3), dict(c, M=17, N=64, K=512), dict(c, M=2048, workspace=1 << 30),
            dict(c, tuning=[entry(own, 300), entry(padded, 400)]), dict(c, tuning=[entry(padded, 400)]), dict(c, workspace=1024, then=[["workspace", 1 << 30]])]
    narrow = [dict(c, workspace=128 * 5120 - 1), dict(c, tuning=[entry(own, 300)]), dict(c, tuning=[entry(own, 500), entry(padded, 400)]),
              dict(c, then=[["workspace", 128 * 5120 * 6 // 8]])]
    for r in launches(tmp_path, wide):
        convert, made = r["launches"]
        assert r["status"] == 0 and r["tile"].startswith("AqBMMA_8x2xfalse_") and re.match(r"relayout_planes(_ws)?_kernel<8>$", convert["kernel"]), r
        assert made["kernel"].startswith("gemm_mfma_staged<8, 2, false") and (made["grid"], made["block"]) == (r["grid"], r["block"]), r
    for r in launches(tmp_path, narrow):
        assert r["status"] == 0 and r["tile"].startswith("AqBMMA_6x2xfalse_") and r["launches"][-1]["kernel"].startswith("gemm_mfma_tiled<6, 2, false"), r
    # planes against planes, and pairs that are not built, are what they were
    both, records, unbuilt = launches(tmp_path, [dict(c, layouts=(0, 0), workspace=1 << 30), dict(c, layouts=(1, 1)), dict(c, q=5)])
    assert both["tile"].startswith("AqBMMA_6x2xfalse_") and records["tile"].startswith("AqBMMA_6x2xfalse_") and unbuilt["status"] == 3


# prefills of many rows on outputs of few columns of tiles: (call, blocks of rows, columns of tiles, kernel)
SPREAD = [(dict(q=8, p=2, signed=1, M=9500, N=1100, K=256, group=128), 75, 9, "gemm_mfma_staged<8, 2, true, false, 2, 2, 2, 2, 3, true, 1>"),
          (dict(q=8, p=2, signed=1, M=9500, N=600, K=384), 149, 5, "gemm_mfma_staged<8, 2, true, false, 1, 2, 2, 2, 4, false, 1>"),
          (dict(q=4, p=4, signed=1, M=9500, N=130, K=256, group=128, layouts=(2, 2)), 75, 3, "gemm_mfma_staged<6, 6, true, true, 2, 1, 2, 2, 4, true, 1>"),
          (dict(q=4, p=4, signed=1, M=9500, N=1290, K=128, layouts=(2, 2)), 75, 11, "gemm_mfma_staged<6, 6, true, true, 2, 2, 2, 2, 3, false, 1>"),
          (dict(q=3, p=3, signed=1, M=9500, N=130, K=128), 149, 3, "gemm_mfma_tiled<3, 3, true, 1, 1, false, 128, 2, 2>"),
          (dict(q=3, p=3, signed=1, M=9500, N=1100, K=256), 38, 9, "gemm_mfma_tiled<3, 3, true, 2, 2, false, 128, 4, 2>"),
          (dict(q=6, p=6, signed=0, M=9473, N=260, K=128), 75, 3, "gemm_mfma_tiled<6, 6, false, 2, 2, false, 128, 2, 2>"),
          (dict(q=8, p=8, signed=0, M=9600, N=1160, K=256), 75, 10, "gemm_mfma_tiled<8, 8, false, 2, 2, false, 128, 2, 2>"),
          (dict(q=8, p=4, signed=1, M=9500, N=2200, K=256, group=64), 75, 18, "gemm_mfma_tiled<8, 4, true, 2, 2, true, 128, 2, 2>")]


def spread_grid(m_blocks, n_blocks):
    """Workgroups where the columns left over from whole eighths are dealt out by tiles, eight blocks of rows at a time."""
    own, left, last = n_blocks // 8, n_blocks % 8, m_blocks % 8
    return 8 * (m_blocks // 8 * (8 * own + left) + last * own + -(-last * left // 8))


def test_large_prefills_on_few_columns_of_tiles_launch_the_spread_grid(tmp_path):
    for (c, m_blocks, n_blocks, kernel), r in zip(SPREAD, launches(tmp_path, [c for c, *_ in SPREAD])):
        (made,) = r["launches"]
        assert r["status"] == 0 and made["kernel"] == kernel and made["grid"] == r["grid"], (c, r)
        assert r["grid"] == [spread_grid(m_blocks, n_blocks), 1, 1] and r["grid"][0] < 8 * -(-n_blocks // 8) * m_blocks, (c, r)


def test_rows_quantised_in_the_group_scale_decode_kernel_take_short_requests_where_those_were_ahead(tmp_path):
    """(weight bits, rows, N, K) -> whether the weight loads go out without the test for a second block of rows"""
    ahead = {(2, 1, 3072, 1792): True, (2, 1, 4096, 4096): True, (2, 1, 4096, 8192): True, (2, 1, 4096, 11008): False, (2, 1, 4112, 2944): False,
             (2, 1, 8192, 4096): False, (2, 1, 8192, 5504): True, (2, 1, 12288, 4096): False, (2, 1, 12288, 5504): True, (2, 1, 16384, 4096): True,
             (2, 1, 22016, 4096): True, (4, 1, 4096, 2944): True, (4, 1, 4096, 4096): False, (4, 1, 4096, 8192): True, (4, 1, 4096, 8448): False,
             (4, 1, 7424, 2944): False, (4, 1, 8192, 4608): True, (4, 1, 9216, 4608): False, (8, 1, 4096, 2048): True, (8, 1, 4096, 2432): False,
             (8, 1, 8192, 1280): False, (2, 4, 4096, 4096): True, (4, 2, 4096, 2048): True, (4, 2, 4096, 6144): False, (8, 3, 4096, 2432): False}
    calls = [dict(q=8, p=p, signed=1, M=m, N=n, K=k, group=128, dynamic=True) for p, m, n, k in ahead]
    for c, r, want in zip(calls, launches(tmp_path, calls), ahead.values()):
        (made,) = r["launches"]
        assert r["status"] == 0 and re.fullmatch(r"gemm_decode_tiled_grouped<8, %d, true, \d, \d, \d, [148], 0, [14], false, %s>" % (
            c["p"], "true" if want else "false"), made["kernel"]), (c, r)


def test_only_weight_sized_codes_are_packed_past_the_caches(tmp_path):
    lines = {(4096, 4096, 2): True, (22016, 4096, 4): True, (4095, 4096, 2): False, (4095, 4096, 3): False, (2048, 4096, 4): True, (2047, 4096, 4): False, (1966, 4480, 2): False, (12288, 4096, 5): False, (1, 128, 1): False}
    for (rows, k, bits), r in zip(lines, launches(tmp_path, [dict(pack=list(c)) for c in lines])):
        (made,) = r["launches"]
        assert r["status"] == 0 and made["kernel"].startswith("pack_i32_lines_kernel<%d>" % bits if lines[rows, k, bits] else "pack_i32_quads_kernel"), (rows, k, bits, r)
