"""GPU tests of the packing kernels at the edges of their plans: rows quantised by four, eight and sixteen waves and by one,
static packing of one and two units per thread, zero points folded into weight records four codes at a time and one by one,
against the oracle's packing and plain arithmetic on the CPU."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def planes_dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int32)).cuda()


@pytest.mark.parametrize("fp6", [False, True])
# lengths on either side of 2048 and 8192 elements, rows on either side of 256
@pytest.mark.parametrize("M,K", [(3, 2048), (5, 2176), (256, 2176), (257, 2176), (7, 8192), (2, 8320), (256, 8320), (257, 8320), (1, 16384)])
def test_quantised_rows(abq, oracle, fp6, M, K):
    rng = np.random.default_rng(M + K)
    x = (rng.standard_normal((M, K)) * np.exp(rng.standard_normal((M, 1)))).astype(np.float16)
    bits = 4 if fp6 else 8
    xt = torch.from_numpy(x).cuda()
    half = 1 << (bits - 1)
    scale = np.clip(np.abs(x.astype(np.float32)).max(1) / np.float32(half - 1), 1e-5, 1e4).astype(np.float32)
    codes = np.clip(np.rint(x.astype(np.float32) / scale[:, None]), -half, half - 1).astype(np.int32)
    planes = planes_dev(oracle.pack_i32(codes, bits))
    out = torch.empty(M * K * 8 // 32, dtype=torch.int32, device="cuda")
    xs = torch.empty(M, dtype=torch.float32, device="cuda")
    sums = torch.empty((M, K // 128), dtype=torch.int32, device="cuda")
    layout = abq.LAYOUT_FP6 if fp6 else abq.LAYOUT_TILED
    assert abq.lib().abq_quant_pack_f16(xt.data_ptr(), M, K, bits, 1, layout, out.data_ptr(), xs.data_ptr(), None, sums.data_ptr(), 128,
                                        torch.cuda.current_stream().cuda_stream) == 0
    want = abq.relayout_planes_fp6(planes, True) if fp6 else abq.relayout_planes(planes)
    torch.cuda.synchronize()
    assert np.array_equal(xs.cpu().numpy(), scale)
    assert torch.equal(out[: want.numel()].view(-1), want.view(-1))
    assert np.array_equal(sums.cpu().numpy(), codes.reshape(M, K // 128, 128).sum(2))


@pytest.mark.parametrize("fp6,bits", [(False, 8), (False, 4), (True, 4)])
@pytest.mark.parametrize("M,K", [(1, 128), (3, 1152), (510, 4096), (513, 4224)])
def test_static_packing(abq, oracle, fp6, bits, M, K):
    rng = np.random.default_rng(M + K + bits)
    half = 1 << (bits - 1)
    x = (rng.uniform(-half, half - 0.01, (M, K)) / 4).astype(np.float16)
    codes = np.trunc((x * np.float16(4.0)).astype(np.float32)).astype(np.int32)
    planes = planes_dev(oracle.pack_i32(codes, bits))
    want = abq.relayout_planes_fp6(planes, True) if fp6 else abq.relayout_planes(planes)
    out = torch.empty_like(want)
    xt, step = torch.from_numpy(x).cuda(), torch.full((1,), 4.0, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    L = abq.lib()
    rc = L.abq_pack_f16_fp6(xt.data_ptr(), step.data_ptr(), out.data_ptr(), M, K, bits, 1, st) if fp6 else \
        L.abq_pack_f16_tiled(xt.data_ptr(), step.data_ptr(), out.data_ptr(), M, K, bits, st)
    assert rc == 0
    torch.cuda.synchronize()
    assert torch.equal(out, want)


@pytest.mark.parametrize("bits,group", [(1, 128), (2, 128), (2, 64), (3, 96), (4, 128), (5, 32), (6, 256), (7, 128)])
@pytest.mark.parametrize("spread", [0, 70])  # zero points inside the range that is folded four codes at a time, and beyond
def test_folded_zero_points(abq, oracle, bits, group, spread):
    rows, K = 41, 768
    rng = np.random.default_rng(bits + group + spread)
    half, rb = 1 << (bits - 1), abq.lib().abq_folded_bits(bits)
    codes = rng.integers(-half, half, (rows, K)).astype(np.int32)
    zero = rng.integers(-half, half, (rows, K // group)).astype(np.float32)
    planes = planes_dev(oracle.pack_i32(codes, bits))
    if group in (64, 128):
        term = abq.weight_zero_term(planes, True, torch.ones((rows, K // group), device="cuda"), torch.from_numpy(zero).cuda(), group)
        assert np.array_equal(term.cpu().numpy(), (codes.reshape(rows, -1, group).sum(2) - group * zero).sum(1).astype(np.float32))
    if spread:
        zero[3, 0] = spread
    diff = codes - np.repeat(zero, group, axis=1).astype(np.int32)
    fits = diff.min() >= -(1 << (rb - 1)) and diff.max() < 1 << (rb - 1)
    zt = torch.from_numpy(zero).cuda()
    if not fits:
        with pytest.raises(ValueError):
            abq.relayout_planes_folded(planes, zt, group, True)
        return
    got = abq.relayout_planes_folded(planes, zt, group, True)
    assert torch.equal(got, abq.relayout_planes(planes_dev(oracle.pack_i32(diff, rb))))
