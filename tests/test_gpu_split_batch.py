"""Batches of small fast layers on the split kernel's tiles: each layer's
result is bitwise that of its own launch (the same tiles, splits and order of
sums), and within the fast-mode tolerance of the oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import hotarubi_amd as hb
import oracle
from helpers import (EP_ADD, EP_ADDP, EP_MULP, EP_RELU, block_abs_sums, check_fast, mxfp4_weights,
                     oracle_linear_mt, random_a_words, w8_planes_from_int8)

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


# (m, n, kb, layers): one and several K splits, partial row and column tiles,
# exactly two tiles to a CU on 256 CUs (512), a single step.
@pytest.mark.parametrize("panels", [False, True])
@pytest.mark.parametrize("w8", [False, True])
@pytest.mark.parametrize("m,n,kb,layers", [(17, 96, 2, 2), (50, 192, 2, 32), (50, 64, 6, 9),
                                           (160, 128, 13, 20), (33, 32, 1, 256), (61, 160, 35, 3)])
def test_batch_equals_single_launches(gpu, m, n, kb, layers, w8, panels):
    rng = np.random.default_rng(m * n + kb + layers)
    quads, L = (m + 3) // 4, layers
    a = np.stack([random_a_words(rng, m, kb) for _ in range(L)])
    if m > 40:
        a[L - 1, 0, 128] = 60  # the last layer's first row leaves the fast window
    if w8:
        w = [np.stack(x) for x in zip(*[w8_planes_from_int8(rng.integers(-127, 128, (n, kb * 32)))
                                        for _ in range(L)])]
        modes = [1, 2]
    else:
        w = [np.stack([oracle.pack_wbuf(*mxfp4_weights(rng, n, kb * 32)) for _ in range(L)])]
        modes = [0]
    a_d, w_d = dev(a), [dev(x) for x in w]
    if panels:
        packed = [torch.empty((L, hb.panel_bytes(n, kb)), dtype=torch.uint8, device=DEV) for _ in w]
        for src, dst in zip(w_d, packed):
            for i in range(L):
                hb.pack_weights(src[i], n, kb, dst[i], ctx=gpu)
        w_d = packed
    scale = (rng.random((L, n)) * 0.02).astype(np.float32)
    bias = rng.standard_normal((L, n)).astype(np.float32)
    x2 = rng.standard_normal((L, m, n)).astype(np.float32)
    s_d, b_d, x_d = dev(scale), dev(bias), dev(x2)
    start = rng.standard_normal((L, m, n)).astype(np.float32)
    pieces = [(kb - kb // 2, kb // 2), (0, kb - kb // 2)] if kb > 2 else None
    print("split batch", (m, n, kb, layers, w8, panels), flush=True)

    def descs(c, q):
        return [hb.linear_desc(m, n, kb, a_d[i], [x[i] for x in w_d], modes, c[i], pieces=pieces,
                               onto=True, ops=[(EP_MULP, s_d[i]), (EP_ADDP, b_d[i]),
                                               (EP_ADD, x_d[i]), (EP_RELU, None)],
                               mode=hb.FAST, q_out=q[i], panels=panels) for i in range(L)]
    c1, c2 = dev(start), dev(start)
    q1 = torch.zeros((L, quads * (n // 32), 144), dtype=torch.uint8, device=DEV)
    q2 = torch.ones_like(q1)
    hb.linear_batched(descs(c1, q1), gpu)
    for d in descs(c2, q2):
        hb.launch(d, gpu)
    torch.cuda.synchronize()
    assert torch.equal(c1.view(torch.int32), c2.view(torch.int32)) and torch.equal(q1, q2)
    for i in (0, L - 1):
        ops = [(EP_MULP, scale[i].view(np.uint32)), (EP_ADDP, bias[i].view(np.uint32)),
               (EP_ADD, x2[i].view(np.uint32)), (EP_RELU, None)]
        want, wq = oracle_linear_mt(m, n, kb, a[i], [x[i] for x in w], modes, ops=ops,
                                    pieces=pieces, onto=start[i].view(np.uint32), quantize=True)
        bound = block_abs_sums(m, n, kb, a[i], [x[i] for x in w], modes, pieces)
        # (after MULP the layer's own error shrinks with the scale; the ops
        # add one rounding each)
        check_fast(c1[i].cpu().numpy().view(np.uint32), want,
                   bound=bound + 4 * 2.0 ** -6 * (np.abs(x2[i]) + np.abs(bias[i]) + 1))
