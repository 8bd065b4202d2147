"""Decode on prepared operands with scales that are one number for the whole call: the kernels bring the number the activations are
quantised with, and the one of the result, into LDS ahead of the weights, and find a unit's row by a reciprocal."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def planes_dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int32)).cuda()


# one and several rows, blocks of rows, one K tile, steps left over, several rounds of the K loop, several passes over the activations
@pytest.mark.parametrize("M,N,K", [(1, 40, 128), (3, 16, 384), (7, 130, 1152), (16, 100, 4096), (40, 33, 2176), (1, 24, 19968), (5, 17, 24704), (2, 48, 66048)])
@pytest.mark.parametrize("q,p", [(8, 2), (8, 4), (8, 8), (4, 2), (8, 3)])
def test_scales_of_the_whole_call(abq, oracle, M, N, K, q, p):
    rng = np.random.default_rng(M + N + K + p)
    w = rng.integers(-(1 << p - 1), 1 << p - 1, (N, K), dtype=np.int32)
    codes = rng.integers(-3 if q == 8 else -2, 3, (M, K), dtype=np.int32)
    codes[:, :: max(K // 96, 1)] = rng.integers(-(1 << q - 1), 1 << q - 1, codes[:, :: max(K // 96, 1)].shape, dtype=np.int32)
    x = torch.from_numpy(codes.astype(np.float16) / np.float16(8)).cuda()  # times 8: the codes, without rounding
    want = oracle.np_gemm(codes, w)
    wt = abq.relayout_planes(planes_dev(oracle.pack_i32(w, p)))
    step, out_scale = torch.full((1,), 8.0, device="cuda"), torch.full((1,), 2.0 ** -6 * 1.3, device="cuda")

    def halves(sums):
        with np.errstate(over="ignore"):  # sums beyond fp16 are infinite, as in the reference's epilogue
            return sums.astype(np.float32).astype(np.float16) * out_scale.cpu().numpy().astype(np.float16)

    packed = abq.pack_f16(x, step, q, tiled=True)
    for kw, expect in ((dict(), lambda sums: sums), (dict(out_kind=abq.OUT_F16_TENSOR_F32SCALE, c_scale=out_scale), halves)):
        g = abq.Gemm(packed, wt, True, x_tiled=True, w_tiled=True, **kw)
        assert np.array_equal(g.run().cpu().numpy(), expect(want)), (q, p, M, N, K, kw)
        if q != 8 or p == 3 or M > 16:
            continue
        try:
            g.set_f16_activations(x, step)
        except abq.AbqError:
            assert M * K > 32768  # rows that do not fit
            continue
        for stepped in (1.0, 0.5):  # the scale is read by each call
            step.fill_(8.0 * stepped)
            sums = oracle.np_gemm(np.trunc(codes * stepped).astype(np.int32), w)
            assert np.array_equal(g.run().cpu().numpy(), expect(sums)), (p, M, N, K, kw, stepped)
        step.fill_(8.0)


# unsigned 8-bit codes go into the matrix cores as code - 128 and the row sums make up for it in the result
@pytest.mark.parametrize("M,N,K", [(1, 40, 128), (7, 130, 1152), (16, 100, 4096), (40, 33, 2176), (5, 17, 24704)])
@pytest.mark.parametrize("q,p", [(8, 2), (8, 8), (8, 3)])
def test_row_sums_of_the_result(abq, oracle, M, N, K, q, p):
    rng = np.random.default_rng(M + N + K + p)
    x, w = rng.integers(0, 1 << q, (M, K), dtype=np.int32), rng.integers(0, 1 << p, (N, K), dtype=np.int32)
    planes, wp = planes_dev(oracle.pack_i32(x, q)), planes_dev(oracle.pack_i32(w, p))
    x_tiled, w_tiled, w_sums, x_sums = abq.relayout_planes(planes), abq.relayout_planes(wp), abq.row_sums(wp), abq.row_sums(planes)
    want = oracle.np_gemm(x, w)
    g = abq.Gemm(x_tiled, w_tiled, False, x_tiled=True, w_tiled=True, w_row_sums=w_sums, x_row_sums=x_sums)
    assert np.array_equal(g.run().cpu().numpy(), want), (q, p, M, N, K)
    tiles = [c for c in abq.native_configs(q, p, False) if c.nstage == 6 and c.mma_m == 16]  # the instances it can be tuned to
    for cfg in tiles if M <= 16 else []:
        g = abq.Gemm(x_tiled, w_tiled, False, x_tiled=True, w_tiled=True, w_row_sums=w_sums, x_row_sums=x_sums, cfg=cfg)
        assert np.array_equal(g.run().cpu().numpy(), want), (q, p, M, N, K, cfg)
