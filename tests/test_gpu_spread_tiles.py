"""Prefills of many rows whose columns of tiles do not divide by the eight XCDs: the columns left over are dealt out tile by tile, some
workgroups have none, and every output tile is written."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from test_launches import SPREAD, spread_grid


def codes(gen, rows, k, bits, signed):
    low = -(1 << bits - 1) if signed else 0
    return torch.randint(low, low + (1 << bits), (rows, k), dtype=torch.int32, device="cuda", generator=gen)


@pytest.mark.parametrize("call,m_blocks,n_blocks,kernel", SPREAD)
def test_every_tile_is_written(abq, call, m_blocks, n_blocks, kernel):
    q, p, signed, M, N, K, group = (call.get(n, 0) for n in ("q", "p", "signed", "M", "N", "K", "group"))
    gen = torch.Generator(device="cuda").manual_seed(M + N + q)
    x, w = codes(gen, M, K, q, signed), codes(gen, N, K, p, signed)
    xp, wp = abq.pack_i32(x, q), abq.pack_i32(w, p)
    if call.get("layouts") == (2, 2):
        operands = (abq.relayout_planes_fp6(xp, signed), abq.relayout_planes_fp6(wp, signed), signed)
        kw = dict(x_fp6=q, w_fp6=p)
    else:
        operands, kw = (abq.relayout_planes(xp), abq.relayout_planes(wp), signed), dict(x_tiled=True, w_tiled=True)
    if group:
        # scales that are powers of two: every product and sum is exact in fp32, and the result is rounded once, to fp16
        xs = torch.exp2(torch.randint(-4, -1, (M,), device="cuda", generator=gen).float())
        ws = torch.exp2(torch.randint(-6, -3, (N, K // group), device="cuda", generator=gen).float())
        want = sum((x[:, g * group:][:, :group].double() @ w[:, g * group:][:, :group].double().T) * ws[:, g].double() for g in range(K // group))
        want = (want * xs.double()[:, None]).half()
        kw.update(out_kind=abq.OUT_F16_SCALED, x_scale=xs, w_scale=ws, group_size=group)
        out = torch.full((M, N), 12345.0, dtype=torch.float16, device="cuda")
    else:
        want = (x.double() @ w.double().T).int()
        out = torch.full((M, N), 0x5A5A5A5A, dtype=torch.int32, device="cuda")
    g = abq.Gemm(*operands, out=out, **kw)
    assert g.state.grid_dim.x == spread_grid(m_blocks, n_blocks)
    assert torch.equal(g.run(), want)
    if not signed and 8 in (q, p):  # the kernel that is handed the row sums, on its own tile
        out.fill_(0x5A5A5A5A)
        g = abq.Gemm(*operands, out=out, x_row_sums=abq.row_sums(xp), w_row_sums=abq.row_sums(wp), **kw)
        assert torch.equal(g.run(), want)
