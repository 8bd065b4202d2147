"""GPU test of the 64x64 prefill tile whose four groups of waves split K: the pairs it is built for, signed and unsigned, asked for
by name and picked, grids at the limit up to which it is and past it, numbers of K tiles that leave one to
three groups without a tile in the last trip."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q,p,signed", [(8, 2, True), (8, 4, True), (4, 4, True), (4, 2, False), (2, 2, False), (8, 2, False), (8, 4, False)])
@pytest.mark.parametrize("M,N,K", [(130, 72, 8192), (192, 100, 8320), (129, 4096, 8448), (193, 3136, 8576), (200, 64, 4224)])
def test_four_groups(abq, oracle, q, p, signed, M, N, K):
    rng = np.random.default_rng(M + N + K + 10 * q + p)
    lo = (lambda b: -(1 << (b - 1))) if signed else (lambda b: 0)
    hi = (lambda b: 1 << (b - 1)) if signed else (lambda b: 1 << b)
    x, w = rng.integers(lo(q), hi(q), (M, K)).astype(np.int32), rng.integers(lo(p), hi(p), (N, K)).astype(np.int32)
    dev = lambda a, b: torch.from_numpy(oracle.pack_i32(a, b).view(np.int32)).cuda()  # noqa: E731
    xp, wp = dev(x, q), dev(w, p)
    kw = dict(x_tiled=True, w_tiled=True, out_kind=abq.OUT_I32)
    if not signed and 8 in (q, p):
        kw.update(w_row_sums=abq.row_sums(wp))
    g = abq.Gemm(abq.relayout_planes(xp), abq.relayout_planes(wp), signed, **kw)
    flip = not signed and 8 in (q, p)
    four = (M + 63) // 64 * ((N + 63) // 64) <= (112 if (q, p, signed) == (8, 2, True) else 192) and K >= (4096 if flip else 8192)
    groups = 4 if four else 1 if flip else 2
    name = "AqBMMA_%dx%dx%s_64x64x%%d_32x32x128_32x32x32_4" % (q, p, "true" if signed else "false")
    assert g.config_name == name % (128 * groups) and g.state.block_dim.x == 256 * groups
    asked = abq.Gemm(abq.relayout_planes(xp), abq.relayout_planes(wp), signed, cfg=abq.parse_kernel_name(name % 512)[0], **kw)
    assert asked.config_name == name % 512
    print(q, p, signed, M, N, K, flush=True)
    want = torch.from_numpy(x).cuda().double() @ torch.from_numpy(w).cuda().double().t()
    for h in (g, asked):
        out = h.run()
        torch.cuda.synchronize()
        assert torch.equal(out.double(), want)
