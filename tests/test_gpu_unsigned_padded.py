"""Unsigned W2A6 above 16 rows with the activations as planes: as records of the padded width on the LDS-staged kernel where the
workspace holds them, on the pair's own kernel where it does not; unsigned 8-bit records declared to hold narrower codes need no
row sums."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def planes_dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int32)).cuda()


@pytest.mark.parametrize("M,N,K", [(17, 64, 512), (40, 200, 1408), (128, 5120, 640), (128, 328, 5120), (300, 130, 1152), (700, 1088, 256)])
def test_unsigned_activations_of_several_fields(abq, oracle, M, N, K):
    rng = np.random.default_rng(M + N)
    x = rng.integers(0, 64, (M, K), dtype=np.int32)
    w = rng.integers(0, 4, (N, K), dtype=np.int32)
    x[0], x[1], w[0], w[N - 1] = 63, 0, 3, 3
    xd, wt = planes_dev(oracle.pack_i32(x, 6)), abq.relayout_planes(planes_dev(oracle.pack_i32(w, 2)))
    want = oracle.np_gemm(x, w)
    g = abq.Gemm(xd, wt, False, w_tiled=True)
    assert g.state.cfg.x_bits == 6 and g.workspace_bytes >= M * K
    for size in (g.workspace_bytes, M * K - 1, M * K * 6 // 8):  # the wider records, and two workspaces that hold the pair's own only
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        g = abq.Gemm(xd, wt, False, w_tiled=True, workspace=ws)
        assert g.state.cfg.x_bits == (8 if size >= M * K else 6)
        assert np.array_equal(g.run().cpu().numpy(), want), (size, M, N, K)
        assert np.array_equal(g.run_static().cpu().numpy(), want), (size, M, N, K)
    scale = torch.full((1,), 0.125, device="cuda")  # another epilogue: half(sum) * half(scale)
    g = abq.Gemm(xd, wt, False, w_tiled=True, workspace=torch.empty(M * K, dtype=torch.uint8, device="cuda"),
                 out_kind=abq.OUT_F16_TENSOR_F32SCALE, c_scale=scale)
    assert np.array_equal(g.run().cpu().numpy(), want.astype(np.float32).astype(np.float16) * np.float16(0.125))


@pytest.mark.parametrize("q,p", [(6, 2), (6, 6), (7, 7)])
def test_row_sums_of_rows_of_any_length(abq, oracle, q, p):
    rng = np.random.default_rng(q)
    for rows, K in [(1, 128), (5, 8192), (3, 8320), (4, 16512)]:
        v = rng.integers(0, 1 << q, (rows, K), dtype=np.int32)
        assert np.array_equal(abq.row_sums(planes_dev(oracle.pack_i32(v, q))).cpu().numpy(), v.sum(1))


@pytest.mark.parametrize("bits", [(8, 8), (8, 7), (7, 8), (6, 6)])
@pytest.mark.parametrize("M,N,K", [(40, 100, 1152), (300, 130, 384), (517, 1030, 256)])
def test_w8a8_records_of_narrower_codes(abq, oracle, bits, M, N, K):
    """Either operand, both or none fed as code - 128: the result is corrected by the sums of the one or two that are."""
    rng = np.random.default_rng(M + bits[0])
    x, w = (rng.integers(0, 1 << b, (r, K), dtype=np.int32) for b, r in zip(bits, (M, N)))
    xp, wp = planes_dev(oracle.pack_i32(x, 8)), planes_dev(oracle.pack_i32(w, 8))
    g = abq.Gemm(abq.relayout_planes(xp), abq.relayout_planes(wp), False, x_tiled=True, w_tiled=True, value_bits=bits,
                 x_row_sums=abq.row_sums(xp), w_row_sums=abq.row_sums(wp))
    assert np.array_equal(g.run().cpu().numpy(), oracle.np_gemm(x, w)), g.config_name
