"""GPU tests of the group-scale kernel for 17 rows and more on prepared operands (weights streamed once for up to 64 rows)
at the edges of its plan: two to four blocks of 16 rows, several blocks of 64, one to six tiles of weight rows per
workgroup with the last one ragged, blocks of four K tiles that are not full, one and several blocks per wave.  Expected
values are fp64 matmuls of the dequantised operands; the bounds are those of test_gpu_quant_epilogue.py."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_decode_grouped import operands  # noqa: E402
from test_gpu_quant_epilogue import assert_close_rel  # noqa: E402

pytestmark = pytest.mark.gpu


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
    got = abq.Gemm(xt, wt, True, out_kind=abq.OUT_F16_SCALED, **kw).run()
    torch.cuda.synchronize()
    print(p, M, N, K, act, flush=True)
    assert_close_rel(got.cpu().numpy(), want)
    # without zero points
    for name in ("w_zero", "x_zero", "x_group_sums", "w_zero_term"):
        del kw[name]
    plain = abq.Gemm(xt, wt, True, out_kind=abq.OUT_F16_SCALED, **kw)
    first = plain.run().clone()
    assert torch.equal(plain.run().view(torch.int16), first.view(torch.int16))
    if not act:
        # rows do not depend on how many others there are: the decode kernel's results for sixteen of them
        lo = abq.Gemm(xt[:, :16].contiguous(), wt, True, out_kind=abq.OUT_F16_SCALED, **{**kw, "x_scale": kw["x_scale"][:16].contiguous()}).run()
        assert_close_rel(first[:16].cpu().numpy(), lo.double().cpu().numpy())
