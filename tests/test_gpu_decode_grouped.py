"""GPU tests of the decode kernel with group scales on prepared operands at the edges of its plan: blocks of four K
tiles dealt out to the waves, one to six tiles of 16 weight rows per workgroup, one or two blocks in flight, several
rounds, and activations packed or quantised in the kernel.  Expected values are fp64 matmuls of the dequantised
operands; the bounds are those of test_gpu_quant_epilogue.py."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_quant_epilogue import assert_close_rel, fdev, planes_dev  # noqa: E402

pytestmark = pytest.mark.gpu


def operands(abq, oracle, rng, M, N, K, q, p, group, act):
    from oracle import quantizer as Q
    G = K // group
    x = rng.integers(-(1 << (q - 1)), 1 << (q - 1), (M, K)).astype(np.int32)
    w = rng.integers(-(1 << (p - 1)), 1 << (p - 1), (N, K)).astype(np.int32)
    # (scales that leave results of about one: a gate times its up row must stay within fp16)
    xs, wsc = rng.uniform(0.5, 1.5, M) / (1 << (q - 1)), rng.uniform(0.5, 1.5, (N, G)) / ((1 << (p - 1)) * K ** 0.5)
    xz = rng.integers(-3, 4, M).astype(np.float64)
    wz = rng.uniform(-1.5, 1.5, (N, G)).astype(np.float32).astype(np.float64)  # (no whole numbers)
    want = Q.dequant_matmul(x, xs, xz, w, wsc, wz, group)
    if act:
        b = want.reshape(M, N // 32, 2, 16)
        want = (b[:, :, 0] / (1.0 + np.exp(-b[:, :, 0])) * b[:, :, 1]).reshape(M, N // 2)
    wp = planes_dev(oracle.pack_i32(w, p))
    kw = dict(x_scale=fdev(xs), w_scale=fdev(wsc), group_size=group, w_zero=fdev(wz), x_zero=fdev(xz), x_tiled=True, w_tiled=True,
              x_group_sums=torch.from_numpy(x.reshape(M, G, group).sum(axis=2).astype(np.int32)).cuda(), act=int(act))
    kw["w_zero_term"] = abq.weight_zero_term(wp, True, kw["w_scale"], kw["w_zero"], group)
    return abq.relayout_planes(planes_dev(oracle.pack_i32(x, q))), abq.relayout_planes(wp), kw, want


@pytest.mark.parametrize("q,p", [(8, 2), (8, 4), (8, 8), (4, 4), (2, 2)])
@pytest.mark.parametrize("group", [128, 64])
# one to six tiles per workgroup by the width, the last workgroup ragged; one and two loads of activations per step (8 and 9
# rows); K of one tile, of blocks that are not full, of one and two blocks per wave and of more than two
@pytest.mark.parametrize("M,N,K,act", [(9, 4112, 640, False), (16, 8216, 256, False), (12, 12312, 384, False), (9, 16416, 128, True),
                                       (8, 4128, 4224, True), (10, 32, 4224, True), (1, 40, 16512, False), (11, 24, 16512, False)])
def test_tiles_blocks_and_rounds(abq, oracle, q, p, group, M, N, K, act):
    rng = np.random.default_rng(M + N + K + 10 * q + p)
    xt, wt, kw, want = operands(abq, oracle, rng, M, N, K, q, p, group, act)
    g = abq.Gemm(xt, wt, True, out_kind=abq.OUT_F16_SCALED, **kw)
    assert g.strategy == "decode_tiled", g.strategy
    got = g.run()
    torch.cuda.synchronize()
    assert_close_rel(got.cpu().numpy(), want)


@pytest.mark.parametrize("p", [2, 4, 8])
@pytest.mark.parametrize("symmetric", [True, False])
# rows held in registers (one; two to four), reloaded (more rows, or more blocks than are in flight), blocks that are not full
@pytest.mark.parametrize("M,N,K,act", [(1, 12312, 640, False), (1, 24608, 384, True), (1, 96, 8320, True), (1, 32, 16384, False),
                                       (3, 72, 4224, False), (4, 64, 4096, True), (5, 40, 640, False), (16, 24, 1024, False)])
def test_rows_quantised_in_the_kernel(abq, oracle, p, symmetric, M, N, K, act):
    """Bit for bit the result of the quantise-and-pack kernel and the GEMM on its records."""
    rng = np.random.default_rng(M + N + K + p)
    _, wt, kw, _ = operands(abq, oracle, rng, 1, N, K, 8, p, 128, act)
    gen = torch.Generator(device="cuda").manual_seed(K)
    x = (torch.randn((M, K), generator=gen, device="cuda") * torch.exp(torch.randn((M, 1), generator=gen, device="cuda"))).half()
    if M > 1:
        x[1, 5] = float("inf")  # the scale clamps, the element takes the largest code
    xt, xs, xz, sums = abq.quant_pack_f16(x, 8, symmetric=symmetric, tiled=True, group_size=128)
    term = None if symmetric else kw["w_zero_term"]
    kw.update(x_scale=xs, x_zero=None if symmetric else xz, x_group_sums=sums, w_zero_term=term)
    want = abq.Gemm(xt, wt, True, out_kind=abq.OUT_F16_SCALED, **kw).run()
    w_zero = kw.pop("w_zero")
    for name in ("x_zero", "x_group_sums", "w_zero_term"):
        del kw[name]
    g = abq.Gemm(xt, wt, True, out_kind=abq.OUT_F16_SCALED, **kw)
    g.set_dynamic_f16_activations(x, symmetric, w_zero=w_zero, w_zero_term=term)
    got = g.run()
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("q,p", [(8, 2), (8, 8), (4, 4), (2, 2)])
@pytest.mark.parametrize("group", [128, 64])
# blocks of two and three K tiles, the last one short; waves with an odd number of blocks, whose last is a round of its own (8-bit
# weights and groups of 64: three and two blocks, three each); one tile and several per workgroup by the waves
@pytest.mark.parametrize("M,N,K,act", [(9, 264, 1152, False), (16, 72, 2176, False), (5, 40, 2944, False), (16, 4128, 1408, True), (1, 24, 2048, False),
                                       (8, 40, 8320, False), (16, 32, 9216, True), (3, 8208, 512, False), (16, 8216, 256, False), (12, 4112, 8576, False)])
def test_short_blocks_and_odd_rounds(abq, oracle, q, p, group, M, N, K, act):
    rng = np.random.default_rng(M + N + K + 10 * q + p)
    xt, wt, kw, want = operands(abq, oracle, rng, M, N, K, q, p, group, act)
    g = abq.Gemm(xt, wt, True, out_kind=abq.OUT_F16_SCALED, **kw)
    assert g.strategy == "decode_tiled", g.strategy
    print(q, p, group, M, N, K, act, flush=True)
    got = g.run()
    torch.cuda.synchronize()
    assert_close_rel(got.cpu().numpy(), want)


@pytest.mark.parametrize("p", [2, 8])
# the same with rows quantised in the kernel: units of a block that is no whole wave, records past the end of K
@pytest.mark.parametrize("M,N,K,act", [(1, 40, 128, False), (1, 12312, 1152, False), (3, 24, 2688, False), (4, 64, 1920, True), (16, 40, 896, False),
                                       (1, 96, 8960, True)])
def test_rows_quantised_in_short_blocks(abq, oracle, p, M, N, K, act):
    test_rows_quantised_in_the_kernel(abq, oracle, p, False, M, N, K, act)
    test_rows_quantised_in_the_kernel(abq, oracle, p, True, M, N, K, act)
