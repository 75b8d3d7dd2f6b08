"""The 16-bit encoder, bit for bit against its definition in numpy float32: row scale, 256 error-feedback
runs per row, and the row lengths, row counts and alignments at which its staging changes form.
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

F32 = np.float32
HALF_MAX = {torch.float16: 32752.0, torch.bfloat16: float.fromhex("0x1.fep126")}


def round16(v, dtype):
    return torch.from_numpy(np.ascontiguousarray(v)).to(dtype)


def encode(tod, dtype, order):
    nrows, n = tod.shape
    scale = np.maximum(np.abs(tod).max(axis=1) / F32(HALF_MAX[dtype]), np.finfo(F32).tiny).astype(F32)
    with np.errstate(over="ignore"):
        x = tod / scale[:, None]
    if order == 0:
        return round16(x, dtype), scale
    run = -(-n // 256)
    pad = np.zeros((nrows, 256 * run), F32)
    pad[:, :n] = x
    x = pad.reshape(nrows * 256, run)
    out = torch.empty(x.shape, dtype=dtype)
    e1 = np.zeros(x.shape[0], F32)
    e2 = e1.copy()
    for i in range(run):
        v = x[:, i] + (e1 if order == 1 else F32(2) * e1 - e2)
        out[:, i] = round16(v, dtype)
        e2, e1 = e1, v - out[:, i].float().numpy()
    return out.reshape(nrows, 256 * run)[:, :n].contiguous(), scale


# One block per row (short rows, or at least 256 rows) and several; runs of one sample, of whole tiles
# of 32, of tiles and a rest; lengths that are no multiple of 4; a last group of runs that is cut short.
SHAPES = [(1, 1), (3, 5), (2, 255), (2, 257), (1, 8192), (2, 8448), (300, 421), (257, 1024), (1, 16384), (1, 16388),
          (3, 20000), (2, 33001), (5, 65536)]


@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_encode_bits(gmm, dev, shape, dtype, order):
    rng = np.random.default_rng(shape[0] * 7 + shape[1])
    tod = (rng.standard_normal(shape) * np.exp(rng.uniform(-12, 12, (shape[0], 1)))).astype(F32)
    tod[0, ::5] = 0.0
    tod[-1, ::3] *= F32(1e-30)               # quotients that a reciprocal may not give exactly
    ref, scale = encode(tod, dtype, order)
    for offset in (0, 1):                    # 16-byte aligned input or not
        buf = torch.empty(tod.size + offset, dtype=torch.float32, device=dev)
        src = buf[offset:].view(shape)
        src.copy_(torch.from_numpy(tod))
        got, sc = gmm.encode_tod16(src, dtype, error_feedback=order)
        assert np.array_equal(sc.cpu().numpy(), scale)
        assert torch.equal(got.cpu().view(torch.int16), ref.view(torch.int16))


# Rows whose runs are kept in registers, up to 2048 samples (independent rounding: 256), and the next.
@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("shape", [(2000, 1), (700, 33), (9, 64), (70, 65), (5, 128), (40, 129), (1, 256), (300, 256), (2, 512), (3, 769), (1, 2047), (257, 2048), (3, 2049)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_encode_short_rows(gmm, dev, shape, dtype, order):
    nrows, n = shape
    rng = np.random.default_rng(nrows + 3 * n)
    tod = (rng.standard_normal(shape) * np.exp(rng.uniform(-12, 12, (nrows, 1)))).astype(F32)
    tod[rng.random(shape) < 0.1] = -0.0
    tod[1::3][rng.random(tod[1::3].shape) < 0.02] = np.nan       # left out of the scale, no feedback from them
    tod[2::5, n // 3] = np.inf
    scale = np.maximum(np.fmax.reduce(np.abs(tod), axis=1) / F32(HALF_MAX[dtype]), np.finfo(F32).tiny).astype(F32)
    scale = np.fmax(scale, np.finfo(F32).tiny)
    with np.errstate(invalid="ignore"):
        x = tod / scale[:, None]
        run = -(-n // 256)
        pad = np.zeros((nrows, 256 * run), F32)
        pad[:, :n] = x
        pad = pad.reshape(nrows * 256, run)
        ref = torch.empty(pad.shape, dtype=dtype)
        e1 = np.zeros(pad.shape[0], F32)
        e2 = e1.copy()
        for i in range(run):
            v = pad[:, i] if order == 0 else pad[:, i] + (e1 if order == 1 else F32(2) * e1 - e2)
            ref[:, i] = round16(v, dtype)
            e = v - ref[:, i].float().numpy()
            e2, e1 = e1, np.where(np.isfinite(e), e, F32(0))
    ref = ref.reshape(nrows, 256 * run)[:, :n]
    got, sc = gmm.encode_tod16(torch.from_numpy(tod).to(dev), dtype, error_feedback=order)
    got = got.cpu()
    assert np.array_equal(sc.cpu().numpy(), scale)
    nan = torch.isnan(ref)
    assert torch.equal(torch.isnan(got), nan)
    assert torch.equal(got.view(torch.int16)[~nan], ref.contiguous().view(torch.int16)[~nan])
