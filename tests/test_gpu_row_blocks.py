"""Decode-shaped groups whose row counts lie around the 16-row blocks of the streaming kernels (1, 15,
16, 17, 31 and 32 rows; 33 takes the tile kernels), against the oracle: the down-projection bit for
bit, GroupedMatmulSwigluQuant within one int8 step and 1e-5 of the row scale."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _i8(rng, *shape):
    return rng.integers(-127, 128, size=shape, dtype=np.int8)


@pytest.mark.parametrize("counts", [[16, 1, 15], [17, 0, 16], [31, 32, 2, 18], [33, 17, 32]])
@pytest.mark.parametrize("K,N", [(512, 512), (464, 288), (64, 32)])
def test_row_blocks(cb, orc, counts, K, N):
    rng = np.random.default_rng(sum(counts) + K)
    E, M = len(counts), sum(counts)
    gl = np.cumsum(counts)
    x, w = _i8(rng, M, K), _i8(rng, E, K, N)
    ws = rng.uniform(0.001, 0.01, (E, N)).astype(np.float32)
    xs = rng.uniform(0.005, 0.02, M).astype(np.float32)
    d = [torch.from_numpy(v).to(DEV) for v in (x, w, ws, xs)]
    out = cb.grouped_matmul_quant(*d, gl.tolist())
    np.testing.assert_array_equal(out.view(torch.int16).cpu().numpy().view(np.uint16),
                                  orc.grouped_matmul_quant(x, w, ws, xs, gl))
    y, ys = cb.grouped_matmul_swiglu_quant(*d, gl.tolist())
    yr, ysr = orc.gmsq(x, w, ws, xs, gl)
    assert np.abs(y.cpu().numpy().astype(int) - yr).max() <= 1
    np.testing.assert_allclose(ys.cpu().numpy(), ysr, rtol=1e-5)
