"""Decode-shaped groups whose row counts lie around the 16-row blocks of the streaming kernels (1, 15,
16, 17, 31 and 32 rows; 33 takes the tile kernels), against the oracle: the int8 GEMMs bit for bit,
GroupedMatmulSwigluQuant within one int8 step and 1e-5 of the row scale.  At these sizes the
down-projection's own choice is a tile; the tests that force a grid for the persistent kernels keep it
from choosing one, so that they run the streaming kernel with one and with two row blocks."""
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


def bits16(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


# K off the 64-deep chunks and the waves' 256, N off the 256-column tiles and the lanes' 16-byte columns
SHAPES = [(64, 16), (464, 288), (80, 528), (1040, 272), (2048, 512)]


@pytest.mark.parametrize("counts", [[16, 1, 0, 15], [17, 0, 16], [31, 32, 2, 18], [0, 24, 0, 0, 32]])
@pytest.mark.parametrize("K,N", SHAPES)
def test_streaming_down_projection(cb, orc, overrides, counts, K, N):
    rng = np.random.default_rng(sum(counts) + K + N)
    E, M = len(counts), sum(counts)
    gl = np.cumsum(counts)
    x, w = _i8(rng, M, K), _i8(rng, E, K, N)
    ws = rng.uniform(0.001, 0.01, (E, N)).astype(np.float32)
    xs = rng.uniform(0.005, 0.02, M).astype(np.float32)
    overrides(persistent_grid=256)
    out = cb.grouped_matmul_quant(*[torch.from_numpy(v).to(DEV) for v in (x, w, ws, xs)], gl.tolist())
    np.testing.assert_array_equal(bits16(out), orc.grouped_matmul_quant(x, w, ws, xs, gl))


@pytest.mark.parametrize("M", [1, 16, 17, 31, 32])
@pytest.mark.parametrize("K,N", SHAPES)
@pytest.mark.parametrize("flags", ["plain", "i32", "full", "perchan_off", "bf16_scale"])
def test_streaming_quant_matmul(cb, orc, overrides, M, K, N, flags):
    rng = np.random.default_rng(M + K + N)
    x1, x2 = _i8(rng, M, K), _i8(rng, K, N)
    scale = torch.from_numpy(rng.uniform(0.001, 0.01, 1 if flags == "perchan_off" else N).astype(np.float32))
    if flags == "bf16_scale":
        scale = scale.to(torch.bfloat16)
    pt = None if flags == "i32" else rng.uniform(0.005, 0.02, M).astype(np.float32)
    off = rng.uniform(-1, 1, N).astype(np.float32) if flags == "full" else None
    bias = {"i32": rng.integers(-5000, 5000, N, dtype=np.int32), "full": rng.normal(size=N).astype(np.float32)}.get(flags)
    dt = "bfloat16" if flags in ("plain", "full") else "float16"
    opt = lambda a: None if a is None else torch.from_numpy(a).to(DEV)
    overrides(persistent_grid=256)
    out = cb.quant_matmul(opt(x1), opt(x2), scale.to(DEV), offset=opt(off), pertoken_scale=opt(pt), bias=opt(bias),
                          output_dtype=dt)
    ref = orc.quant_matmul(x1, x2, bits16(scale) if flags == "bf16_scale" else scale.numpy(), offset=off, pertoken=pt,
                           bias=bias, bias_dtype="i32" if flags == "i32" else "f32",
                           scale_dtype="bf16" if flags == "bf16_scale" else "f32",
                           out_dtype="bf16" if dt == "bfloat16" else "f16")
    np.testing.assert_array_equal(bits16(out).reshape(ref.shape), ref)


@pytest.mark.parametrize("counts", [[16, 0, 3], [17, 31], [32, 0, 18, 1]])
@pytest.mark.parametrize("K,N", SHAPES)
def test_streaming_int32(cb, orc, counts, K, N):
    rng = np.random.default_rng(sum(counts) * 3 + K)
    x, w = _i8(rng, sum(counts), K), _i8(rng, len(counts), K, N)
    gl = np.cumsum(counts).tolist()
    c = cb.grouped_matmul_int32(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV), gl).cpu().numpy()
    for e, (a, b) in enumerate(zip([0] + gl, gl)):
        if b > a:
            np.testing.assert_array_equal(c[a:b], orc.i8_gemm(x[a:b], w[e]), err_msg=f"group {e}")
