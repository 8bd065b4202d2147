"""int32 GEMMs whose K is split over several workgroups per output tile (activations as planes, long K, few tiles): on either side
of the rule's lines, ragged rows and columns, K tiles that do not divide by the parts, results that held something before."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from test_launches import SPLITS


def operands(abq, q, p, signed, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    codes = []
    for rows, bits in ((M, q), (N, p)):
        lo, hi = (-(1 << (bits - 1)), (1 << (bits - 1)) - 1) if signed else (0, (1 << bits) - 1)
        c = torch.randint(lo, hi + 1, (rows, K), generator=g, device="cuda", dtype=torch.int32)
        c[0], c[-1] = lo, hi
        codes.append(c)
    return codes


def parts(g):
    """workgroups per output tile of the kernel that runs"""
    n = g.state.reserved[4] >> 8 & 15
    assert (n > 1) == (g.state.cfg.nstage == 8)
    return max(n, 1)


def product(x, w):
    return (x.double() @ w.double().T).long()  # exact: sums below 2^31


@pytest.mark.parametrize("q,p,signed", [(8, 8, True), (8, 8, False), (8, 4, True), (8, 4, False), (4, 4, True), (4, 2, False), (2, 2, True)])
@pytest.mark.parametrize("shape,pairs", SPLITS)
def test_parts_add_up(abq, q, p, signed, shape, pairs):
    M, N, K = shape
    x, w = operands(abq, q, p, signed, M, N, K)
    xd, wd = abq.pack_i32(x, q), abq.pack_i32(w, p)
    want = product(x, w)
    kw = {} if signed or 8 not in (q, p) else {"w_row_sums": abq.row_sums(wd)}
    ws = torch.empty(M * K + 4 * M + 1024, dtype=torch.uint8, device="cuda")
    weights = [(abq.relayout_planes(wd), kw)]
    if (q, p, signed) == (8, 8, False):
        weights.append((abq.relayout_planes_biased(wd), dict(kw, biased=(False, True))))
    for wt, k in weights:
        for off in (0, 1):  # a result off 16-byte boundaries as well
            out = torch.full((M * N + 1,), 7, dtype=torch.int32, device="cuda")[off:off + M * N].view(M, N)
            g = abq.Gemm(xd, wt, signed, out=out, w_tiled=True, workspace=ws, **k)
            assert parts(g) == pairs.get((q, p), parts(g)), g.config_name
            for _ in range(2):  # (the second run finds the first one's result)
                assert torch.equal(g.run().long(), want), (g.config_name, off)


@pytest.mark.parametrize("q,p,signed", [(8, 8, True), (8, 4, False), (8, 2, True), (4, 4, False)])
def test_parts_by_name(abq, q, p, signed):
    """Two parts, which the library does not choose by itself, few rows, weights in planes too; without the row sums one part."""
    for M, N, K in ((256, 4096, 7296), (3, 70, 28672)):
        x, w = operands(abq, q, p, signed, M, N, K)
        xd, wd = abq.pack_i32(x, q), abq.pack_i32(w, p)
        name = "AqBMMA_%dx%dx%s_128x64x%d_64x32x128_32x32x32_8" % (q, p, "true" if signed else "false", 256 if q + p <= 8 else 128)
        for sums in ([{}] if signed or q < 8 else [{}, {"w_row_sums": abq.row_sums(wd)}]):
            for tiled in (True, False):
                g = abq.Gemm(xd, abq.relayout_planes(wd) if tiled else wd, signed, w_tiled=tiled, cfg=abq.parse_kernel_name(name)[0], **sums)
                assert parts(g) == (2 if M > 3 else 8) and g.config_name == name
                ws = torch.empty(g.workspace_bytes + 4 * M + 1024, dtype=torch.uint8, device="cuda")
                g = abq.Gemm(xd, abq.relayout_planes(wd) if tiled else wd, signed, w_tiled=tiled, cfg=abq.parse_kernel_name(name)[0], workspace=ws, **sums)
                assert torch.equal(g.run().long(), product(x, w)), (M, sums, tiled)


def test_parts_under_capture(abq):
    M, N, K = 128, 1024, 8192
    x, w = operands(abq, 8, 8, True, M, N, K)
    xd, wt = abq.pack_i32(x, 8), abq.relayout_planes(abq.pack_i32(w, 8))
    g = abq.Gemm(xd, wt, True, w_tiled=True, workspace=torch.empty(M * K, dtype=torch.uint8, device="cuda"))
    assert parts(g) == 4
    g.run()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g.run()
    for i in range(4):
        x = x.roll(1, 0)
        xd.copy_(abq.pack_i32(x, 8))
        g.out.fill_(i)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(g.out.long(), product(x, w)), i
        assert torch.equal(g.run().long(), product(x, w))


@pytest.mark.parametrize("kind", ["scaled", "tensor"])
def test_other_epilogues_keep_one_workgroup_per_tile(abq, kind):
    M, N, K = 200, 200, 13824
    x, w = operands(abq, 4, 4, True, M, N, K)
    xd, wt = abq.pack_i32(x, 4), abq.relayout_planes(abq.pack_i32(w, 4))
    ws = torch.empty(M * K, dtype=torch.uint8, device="cuda")
    assert parts(abq.Gemm(xd, wt, True, w_tiled=True, workspace=ws)) == 3
    xs, wsc = torch.full((M,), 2.0 ** -8, device="cuda"), torch.full((N,), 0.5, device="cuda")
    kw = dict(out_kind=abq.OUT_F16_SCALED, x_scale=xs, w_scale=wsc) if kind == "scaled" else dict(
        out_kind=abq.OUT_F16_TENSOR_F32SCALE, c_scale=torch.full((1,), 2.0 ** -9, device="cuda"))
    g = abq.Gemm(xd, wt, True, w_tiled=True, workspace=ws, **kw)
    assert parts(g) == 1
    got = g.run()
    sums = product(x, w)
    want = (sums.double() * 2.0 ** -9).half() if kind == "scaled" else sums.float().half() * 2.0 ** -9
    assert torch.equal(got, want)
