"""The kernels a loader brings weight matrices through, at the sizes where their variants begin and end: packing of int32
codes by whole lines (from 2^21 units of eight codes on, 4 bits from 2^20) and the activation zero point's term."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("rows,k", [(2047, 4096), (2048, 4096), (65551, 128), (2731, 3200), (4095, 4096), (4096, 4096), (131103, 128), (5461, 3200)])
def test_packing_of_large_matrices(abq, oracle, bits, rows, k):
    import torch
    g = torch.Generator(device="cuda").manual_seed(bits * 1000 + rows)
    # (bits above the packed ones are set in half of the codes: they must not reach the planes)
    codes = torch.randint(-(1 << 9), 1 << 9, (rows, k), generator=g, device="cuda", dtype=torch.int32)
    got = abq.pack_i32(codes, bits).cpu().numpy().view(np.uint32)
    assert np.array_equal(got, oracle.pack_i32(codes.cpu().numpy(), bits))


@pytest.mark.parametrize("group", [64, 128])
@pytest.mark.parametrize("n,k", [(1, 128), (33, 1024), (31, 2048), (17, 2176), (7, 4096), (5, 4224), (130, 11008)])
@pytest.mark.parametrize("bits,signed", [(2, True), (4, False), (8, True)])
def test_zero_point_term(abq, group, n, k, bits, signed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n + k)
    low = -(1 << (bits - 1)) if signed else 0
    codes = torch.randint(low, low + (1 << bits), (n, k), generator=g, device="cuda", dtype=torch.int32)
    scale = torch.rand((n, k // group), generator=g, device="cuda") + 0.5
    zero = torch.randint(-4, 5, (n, k // group), generator=g, device="cuda").float()
    got = abq.weight_zero_term(abq.pack_i32(codes, bits), signed, scale, zero, group).double()
    part = codes.double().view(n, -1, group).sum(2) - group * zero.double()
    want = (scale.double() * part).sum(1)
    # fp32 sum of G products of exact integers: (G + 1) roundings of 2^-24 of the terms' magnitudes
    bound = (k // group + 1) * 2.0 ** -24 * (scale.double() * part.abs()).sum(1)
    assert bool(((got - want).abs() <= bound + 1e-30).all())
