"""GPU parity of the tiled GEMMs (QuantMatmul, the int8 grouped down-projection and the 16-bit
GroupedMatmul), each tile forced in turn through the library's test override: row
counts around the 32-row fragments and the tile edges, partial column tiles (N off every tile
width), K of one 16-byte chunk, below, at and past a stage and the ring's depth, ragged and empty
groups, every dequant flag and a batch.  The int32 sums are exact and the dequant chain rounds in
the oracle's order, so the bar is bit equality; GroupedMatmul meets the bar of its own parity tests
(one output ulp plus 1e-6 of sum |x w|, the fp32 sum's bound) and is bit-identical for both weight
layouts."""
import numpy as np
import pytest
import torch

import test_gpu_gmm as gmm

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _i8(rng, *shape):
    return rng.integers(-127, 128, size=shape, dtype=np.int8)


def _dev(*arrays):
    return [torch.from_numpy(a).to(DEV) for a in arrays]


def bits16(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


@pytest.fixture(params=[1, 2, 3, 4, 5])  # 32 x 64, 64 x 128, 64 x 256, 128 x 128, 128 x 256
def tile(request, overrides):
    overrides(gmm_tile=request.param)
    return request.param


GROUPED = [
    # (counts, K, N)
    ([1, 0, 31, 33], 16, 16),
    ([64, 65, 0, 127], 144, 272),
    ([129, 2], 1040, 528),
    ([300, 0, 0, 7], 2048, 80),
]


@pytest.mark.parametrize("counts,K,N", GROUPED)
def test_tile_grouped(cb, orc, tile, counts, K, N):
    rng = np.random.default_rng(K + N)
    E, M = len(counts), sum(counts)
    x, w = _i8(rng, M, K), _i8(rng, E, K, N)
    ws = rng.uniform(0.001, 0.01, (E, N)).astype(np.float32)
    xs = rng.uniform(0.005, 0.02, M).astype(np.float32)
    gl = np.cumsum(counts)
    out = cb.grouped_matmul_quant(*_dev(x, w, ws, xs), gl.tolist())
    np.testing.assert_array_equal(bits16(out), orc.grouped_matmul_quant(x, w, ws, xs, gl))


@pytest.mark.parametrize("M,K,N", [(1, 256, 64), (32, 400, 144), (200, 640, 496)])
@pytest.mark.parametrize("flags", ["plain", "i32", "full", "perchan_off"])
def test_tile_quant_matmul(cb, orc, tile, M, K, N, flags):
    rng = np.random.default_rng(M + K)
    x1, x2 = _i8(rng, M, K), _i8(rng, K, N)
    scale = rng.uniform(0.001, 0.01, 1 if flags == "perchan_off" else N).astype(np.float32)
    pt = None if flags == "i32" else rng.uniform(0.005, 0.02, M).astype(np.float32)
    off = rng.uniform(-1, 1, N).astype(np.float32) if flags == "full" else None
    bias = {"i32": rng.integers(-5000, 5000, N, dtype=np.int32), "full": rng.normal(size=N).astype(np.float32)}.get(flags)
    dt = "bfloat16" if flags in ("plain", "full") else "float16"
    opt = lambda a: None if a is None else torch.from_numpy(a).to(DEV)
    out = cb.quant_matmul(*_dev(x1, x2, scale), offset=opt(off), pertoken_scale=opt(pt), bias=opt(bias), output_dtype=dt)
    ref = orc.quant_matmul(x1, x2, scale, offset=off, pertoken=pt, bias=bias,
                           bias_dtype="i32" if flags == "i32" else "f32", out_dtype="bf16" if dt == "bfloat16" else "f16")
    np.testing.assert_array_equal(bits16(out), ref)


def test_tile_batched(cb, tile):
    rng = np.random.default_rng(3)
    x1, x2 = _i8(rng, 3, 70, 272), _i8(rng, 3, 272, 144)
    scale = rng.uniform(0.001, 0.01, 144).astype(np.float32)
    bias = rng.integers(-5000, 5000, (3, 1, 144), dtype=np.int32)
    d = _dev(x1, x2, scale, bias)
    out = cb.quant_matmul(*d[:3], bias=d[3], output_dtype="bfloat16")
    acc = np.matmul(x1.astype(np.int64), x2.astype(np.int64)).astype(np.float32) + bias.astype(np.float32)
    ref = torch.from_numpy(acc * scale).to(torch.bfloat16)
    assert torch.equal(out.cpu(), ref)


@pytest.mark.parametrize("t", [1, 2, 3, 4, 5, 6])  # as above, then 256 x 256
@pytest.mark.parametrize("counts,K,N", [([1, 0, 33, 64], 8, 24), ([127, 130, 2], 200, 264), ([257, 0, 31], 1032, 72)])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_tile_grouped_matmul(cb, orc, overrides, t, counts, K, N, dtype):
    overrides(gmm_tile=t)
    x, w, b, ends = gmm._inputs(counts, K, N, dtype, False, "f32", K + N)
    args = dict(bias=b.to(DEV), split_item=2)
    y = cb.grouped_matmul(x.to(DEV), w.to(DEV), ends, **args)[0]
    yt = cb.grouped_matmul(x.to(DEV), w.transpose(1, 2).contiguous().to(DEV), ends, transpose_weight=True, **args)[0]
    assert torch.equal(y.view(torch.int16), yt.view(torch.int16))
    ref = orc.grouped_matmul(gmm.host(x, dtype), gmm.host(w, dtype), ends, b.numpy(), dtype=dtype, bias_dtype="f32")
    gmm._check(y, ref, dtype, x.float(), w.float(), ends, False)


@pytest.mark.parametrize("counts,K,N", [([1, 0, 33, 300], 1152, 264), ([256, 257, 31], 1208, 72), ([513], 1600, 776)])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("bias", ["f32", None])
def test_grouped_matmul_long_k_layouts(cb, orc, overrides, counts, K, N, dtype, bias):
    """From K of 1152 on the 256 x 256 tile of a [N][K] weight is a kernel of its own: the oracle's result, and the
    bits of the [K][N] kernel."""
    overrides(gmm_tile=6)
    x, w, b, ends = gmm._inputs(counts, K, N, dtype, False, bias, K + N)
    args = dict(bias=None if b is None else b.to(DEV), split_item=2)
    y = cb.grouped_matmul(x.to(DEV), w.to(DEV), ends, **args)[0]
    yt = cb.grouped_matmul(x.to(DEV), w.transpose(1, 2).contiguous().to(DEV), ends, transpose_weight=True, **args)[0]
    assert torch.equal(y.view(torch.int16), yt.view(torch.int16))
    ref = orc.grouped_matmul(gmm.host(x, dtype), gmm.host(w, dtype), ends, None if b is None else b.numpy(), dtype=dtype,
                             bias_dtype=bias or "f32")
    gmm._check(yt, ref, dtype, x.float(), w.float(), ends, False)


@pytest.mark.parametrize("off", [1, 2, 4])  # elements: y at 2, 4 and 8 bytes past a 16-byte boundary
def test_grouped_matmul_unaligned_output(cb, off):
    """An output off 16-byte alignment (possible through the C ABI) takes the kernel with single-value
    stores and leaves its neighbours alone."""
    x, w, b, ends = gmm._inputs([70, 3], 64, 40, "bf16", False, "f32", 5)
    xd, wd, bd = x.to(DEV), w.to(DEV), b.to(DEV)
    ref = cb.grouped_matmul(xd, wd, ends, bias=bd, split_item=2)[0]
    buf = torch.full((73 * 40 + 16,), 7.0, dtype=torch.bfloat16, device=DEV)
    rc = cb._lib.load().cb_grouped_matmul(
        xd.data_ptr(), wd.data_ptr(), bd.data_ptr(), cb._lib.CB_DT_BFLOAT16, cb._lib.CB_DT_FLOAT32,
        cb._lib.int64_array(ends), 2, 73, 64, 40, 2, 0, buf.data_ptr() + 2 * off, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    got = buf[off:off + 73 * 40].view(73, 40).float()
    # the two kernels sum in different orders: at most one bf16 step apart
    assert ((got - ref.float()).abs() <= ref.float().abs() * 2.0 ** -7 + 1e-5).all()
    assert (buf[:off] == 7).all() and (buf[off + 73 * 40:] == 7).all()
