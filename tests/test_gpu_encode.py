"""The MXINT8 and MXFP8 encoders, bit for bit against the oracle: ragged rows
and columns, an input at 4-byte alignment, block maxima over the whole exponent
range (subnormal ones and those next to the hardware arithmetic's lower end
included), rounding ties, negative values that round to zero, all-zero
blocks."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import hotarubi_amd as hb
import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 31), (4, 32), (5, 40), (7, 100), (33, 129),
                                       (254, 64)])
def test_encode_exponent_range(gpu, rows, cols, fp8):
    rng = np.random.default_rng(rows * 1000 + cols)
    blocks, quads = (cols + 31) // 32, (rows + 3) // 4
    x = rng.standard_normal((rows, blocks * 32))
    x = np.where(rng.random(x.shape) < 0.3, np.round(x * 32) / 32 + 1 / 64, x)
    # one exponent per block, swept over the range: fields 0 (subnormal) .. 254
    e = (np.arange(rows * blocks).reshape(rows, blocks, 1) * 37 + 3) % 255 - 127
    with np.errstate(over="ignore", under="ignore"):
        v = np.ldexp(x.reshape(rows, blocks, 32) / 4, e + 1) * \
            np.exp2(-rng.integers(0, 3, (rows, blocks, 32)) * 4.0)
        v = np.clip(v, -3.4e38, 3.4e38).astype(np.float32)
    v[rng.random((rows, blocks)) < 0.05] = -0.0
    x = np.ascontiguousarray(v.reshape(rows, -1)[:, :cols])
    flat = torch.empty(x.size + 1, dtype=torch.float32, device=DEV)
    flat[1:].copy_(torch.from_numpy(x.reshape(-1)))
    out = torch.full((quads * blocks, 144), 0xAB, dtype=torch.uint8, device=DEV)
    print("encode", rows, cols, fp8, flush=True)
    (hb.encode_mxfp8 if fp8 else hb.encode_mxint8)(flat[1:], rows, cols, out, gpu)
    xp = np.zeros((quads * 4, cols), np.float32)
    xp[:rows] = x
    enc = oracle.encode_mxfp8 if fp8 else oracle.encode_mxint8
    q, ex = enc(oracle.f32_bits(xp))
    assert np.array_equal(out.cpu().numpy(), oracle.pack_abuf(q.view(np.int8), ex))
    # a rejected call leaves the next one's answer alone
    bad = torch.full((4, 32), float("nan"), device=DEV)
    with pytest.raises(hb.HbError):
        (hb.encode_mxfp8 if fp8 else hb.encode_mxint8)(bad, 4, 32, out, gpu)
    (hb.encode_mxfp8 if fp8 else hb.encode_mxint8)(flat[1:], rows, cols, out, gpu)
