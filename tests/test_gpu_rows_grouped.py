"""GPU tests of the group-scale kernel for 17 rows and more on prepared operands (weights streamed once for up to 64 rows),
asked for by its name: every instance (bits of the weights, tiles per workgroup, blocks of 16 rows, with and without zero points),
several blocks of 64 rows, the last workgroup ragged, blocks of four K tiles that are not full, one and several blocks per wave.
Expected values are fp64 matmuls of the dequantised operands; the bounds are those of test_gpu_quant_epilogue.py."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_decode_grouped import operands  # noqa: E402
from test_gpu_quant_epilogue import assert_close_rel  # noqa: E402

pytestmark = pytest.mark.gpu

RUNS = 16  # the bit of reserved[4] that says this kernel runs


def rows_tile(abq, p):
    return abq.parse_kernel_name("AqBMMA_8x%dxtrue_64x16x4096_64x16x512_16x16x64_7" % p)[0]


def plan_of(g):
    """tiles of 16 weight rows per workgroup and blocks of 16 rows, from the launch the state describes"""
    assert g.state.reserved[4] & RUNS
    M, tiles = g.state.M, (g.state.N + 15) // 16
    m64 = (M + 63) // 64
    mb = max(2, ((M + m64 - 1) // m64 + 15) // 16)
    sets = g.state.grid_dim.x // ((M + mb * 16 - 1) // (mb * 16))
    return [t for t in (1, 2, 3, 4, 6) if ((tiles + t - 1) // t + 7) // 8 * 8 == sets], mb


@pytest.mark.parametrize("p", [2, 4, 8])
@pytest.mark.parametrize("M,N,K,act", [(17, 40, 1024, False), (32, 4128, 1152, True), (33, 8216, 1152, False), (43, 16416, 1280, True),
                                       (48, 12312, 1024, False), (49, 4104, 4224, False), (64, 12320, 1024, True), (65, 72, 8320, False),
                                       (96, 4112, 1024, False), (110, 96, 1664, True), (128, 24, 1152, False),
                                       # (the fewest workgroups that take the kernel, in two blocks of rows; K of one to five tiles: one
                                       # and two waves, blocks of one and three tiles)
                                       (65, 2056, 8320, False), (128, 1544, 1152, False), (32, 4096, 128, False), (20, 4128, 384, True),
                                       (64, 4100, 640, False)])
def test_rows_blocks_and_tiles(abq, oracle, p, M, N, K, act):
    rng = np.random.default_rng(M + N + K + p)
    xt, wt, kw, want = operands(abq, oracle, rng, M, N, K, 8, p, 128, act)
    tile = rows_tile(abq, p)
    g = abq.Gemm(xt, wt, True, cfg=tile, out_kind=abq.OUT_F16_SCALED, **kw)
    assert g.state.reserved[4] & RUNS
    print(p, M, N, K, act, flush=True)
    got = g.run()
    torch.cuda.synchronize()
    assert_close_rel(got.cpu().numpy(), want)
    # without zero points
    for name in ("w_zero", "x_zero", "x_group_sums", "w_zero_term"):
        del kw[name]
    plain = abq.Gemm(xt, wt, True, cfg=tile, out_kind=abq.OUT_F16_SCALED, **kw)
    assert plain.state.reserved[4] & RUNS
    first = plain.run().clone()
    assert torch.equal(plain.run().view(torch.int16), first.view(torch.int16))
    if not act:
        # rows do not depend on how many others there are: the decode kernel's results for sixteen of them
        lo = abq.Gemm(xt[:, :16].contiguous(), wt, True, out_kind=abq.OUT_F16_SCALED, **{**kw, "x_scale": kw["x_scale"][:16].contiguous()}).run()
        assert_close_rel(first[:16].cpu().numpy(), lo.double().cpu().numpy())


WIDTH = {1: 4072, 2: 8168, 3: 12264, 4: 16360, 6: 24552}  # widest outputs of one round, one tile short of it and ragged
INSTANCES = [(p, t, mb) for p in (2, 4, 8) for mb in (2, 3, 4) for t in (1, 2, 3, 4, 6) if t * p <= 24 and t * mb <= 18]


@pytest.mark.parametrize("p,t,mb", INSTANCES)
def test_every_instance(abq, oracle, p, t, mb):
    rng = np.random.default_rng(100 * p + 10 * t + mb)
    M, N, K = 16 * mb - 5, WIDTH[t], 640
    xt, wt, kw, want = operands(abq, oracle, rng, M, N, K, 8, p, 128, False)
    for zeros in (True, False):
        if not zeros:
            for name in ("w_zero", "x_zero", "x_group_sums", "w_zero_term"):
                del kw[name]
        g = abq.Gemm(xt, wt, True, cfg=rows_tile(abq, p), out_kind=abq.OUT_F16_SCALED, **kw)
        took, blocks = plan_of(g)
        assert t in took and blocks == mb, (took, blocks)
        print(p, t, mb, zeros, flush=True)
        got = g.run()
        torch.cuda.synchronize()
        if zeros:
            assert_close_rel(got.cpu().numpy(), want)
            continue
        # the same without zero points: the terms left out of the operands
        x = abq.Gemm(xt[:, :16].contiguous(), wt, True, out_kind=abq.OUT_F16_SCALED, **{**kw, "x_scale": kw["x_scale"][:16].contiguous()}).run()
        assert_close_rel(got[:16].cpu().numpy(), x.double().cpu().numpy())


@pytest.mark.parametrize("p", [2, 4, 8])
@pytest.mark.parametrize("K", [1152, 4224])
def test_rows_do_not_depend_on_the_plan(abq, oracle, p, K):
    """Bit for bit the same outputs of the same rows and columns, however many others there are of either."""
    rng = np.random.default_rng(K + p)
    M, N = 130, 12312
    xt, wt, kw, _ = operands(abq, oracle, rng, M, N, K, 8, p, 128, False)
    seen, first = set(), None
    for m in (20, 40, 60, 130):
        for n in (1032, 8168, 12312):
            part = dict(kw, x_scale=kw["x_scale"][:m].contiguous(), x_zero=kw["x_zero"][:m].contiguous(), x_group_sums=kw["x_group_sums"][:m].contiguous(),
                        w_scale=kw["w_scale"][:n].contiguous(), w_zero=kw["w_zero"][:n].contiguous(), w_zero_term=kw["w_zero_term"][:n].contiguous())
            g = abq.Gemm(xt[:, :m].contiguous(), wt[:, :n].contiguous(), True, cfg=rows_tile(abq, p), out_kind=abq.OUT_F16_SCALED, **part)
            took, blocks = plan_of(g)
            seen.add((tuple(took), blocks))
            got = g.run()[:20, :1032].clone().view(torch.int16)
            torch.cuda.synchronize()
            first = got if first is None else first
            assert torch.equal(got, first), (m, n, took, blocks)
    assert len(seen) >= 4, seen
