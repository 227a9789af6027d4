"""MXFP4 layers on waves of their own (32 rows x 64 or 128 columns): the edges
of the wave tiles, odd and single block counts, a piece list that starts past
block 0, C and operands at 4-byte alignment, layers that start from C, every
op, the requantize, and a scale byte outside the fast window (the tile is then
exact); within the fast-mode tolerance of the oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers
import hotarubi_amd as hb
import oracle
from helpers import (EP_ACT, EP_ACT_MUL, EP_ADD, EP_ADDP, EP_COPY, EP_MULP, EP_RELU, EP_SCALE,
                     check_fast, mxfp4_weights, oracle_linear_mt, random_a_words)

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def unaligned(x):
    """x's values on the GPU at an address that is 4 past a multiple of 16."""
    flat = torch.empty(x.size + 1, dtype=torch.float32, device=DEV)
    out = flat[1:].view(x.shape)
    out.copy_(torch.from_numpy(np.ascontiguousarray(x)))
    return out


# (m, n, blocks, first block, kb_total, layers): 64-column waves with partial
# row and column tiles, one block, an odd count, a range of the blocks, at
# most 5 column tiles over many rows (1,057 x 160: 3 of 64, not 2 of 128);
# 128-column waves (at least 512 of them, 4 steps and more) with a partly used
# last column tile, and for a fold of 24 steps that fits one round of the CUs
# in 128 columns and not in 64 (15 layers of 132 x 640: 150 workgroups, not
# 300).
SHAPES = [(1030, 72, 1, 0, 1, 1), (1025, 64, 9, 0, 9, 1), (1057, 160, 6, 2, 9, 1),
          (2049, 96, 13, 0, 13, 1), (170, 200, 5, 0, 5, 3), (65, 416, 7, 0, 7, 43),
          (97, 352, 8, 4, 13, 43), (132, 640, 48, 0, 48, 15)]


@pytest.mark.parametrize("panels", [False, True])
@pytest.mark.parametrize("ops", ["none", "onto", "vectors", "operands", "acts"])
@pytest.mark.parametrize("m,n,blocks,first,kb,layers", SHAPES)
def test_wave_tiles(gpu, m, n, blocks, first, kb, layers, ops, panels):
    rng = np.random.default_rng(m * 7 + n + kb + len(ops))
    quads, L, quant = (m + 3) // 4, layers, n % 32 == 0 and ops != "onto"
    onto = ops in ("onto", "operands")
    pieces = [(first, blocks)] if blocks != kb else None
    a = [random_a_words(rng, m, kb) for _ in range(L)]
    if ops == "operands":
        a[L - 1].reshape(quads, kb, 144)[0, first, 128] = 60  # row 0 leaves the fast window
    w = [oracle.pack_wbuf(*mxfp4_weights(rng, n, kb * 32)) for _ in range(L)]
    w_d = dev(np.stack(w))
    if panels:
        packed = torch.empty((L, hb.panel_bytes(n, kb)), dtype=torch.uint8, device=DEV)
        for i in range(L):
            hb.pack_weights(w_d[i], n, kb, packed[i], ctx=gpu)
        w_d = packed
    a_d = dev(np.stack(a))
    f = lambda *shape: rng.standard_normal(shape).astype(np.float32)
    scale, bias, x2, x3, start = f(L, n) * 0.02, f(L, n), f(L, m, n), f(L, m, n), f(L, m, n)
    s_d, b_d, x_d, x3_d, c = dev(scale), dev(bias), unaligned(x2), dev(x3), unaligned(start)
    imm = int(np.float32(0.03).view(np.uint32))
    tbuf = helpers.activation_table("silu")
    # per layer: (kind, device operand, host operand)
    plan = {"none": lambda i: [], "onto": lambda i: [],
            "vectors": lambda i: [(EP_MULP, s_d[i], scale[i]), (EP_ADDP, b_d[i], bias[i]),
                                  (EP_RELU, None, None)],
            "operands": lambda i: [(EP_SCALE, imm, imm), (EP_ADD, x_d[i], x2[i]),
                                   (EP_COPY, None, None), (EP_ADD, x3_d[i], x3[i])],
            "acts": lambda i: [(EP_MULP, s_d[i], scale[i]), (EP_ACT, None, None),
                               (EP_ACT_MUL, x_d[i], x2[i])]}[ops]
    bits = lambda v: v.view(np.uint32) if isinstance(v, np.ndarray) else v
    q = torch.ones((L, quads * (n // 32), 144), dtype=torch.uint8, device=DEV) if quant else None
    t_d = dev(tbuf.view(np.int64)) if ops == "acts" else None
    descs = [hb.linear_desc(m, n, kb, a_d[i], [w_d[i]], [0], c[i], pieces=pieces, onto=onto,
                            ops=[(k, d) for k, d, _ in plan(i)], tbuf=t_d, mode=hb.FAST,
                            q_out=q[i] if quant else None, panels=panels) for i in range(L)]
    print("wave", (m, n, blocks, first, kb, layers, ops, panels), flush=True)
    if L == 1:
        hb.launch(descs[0], gpu)
    else:
        hb.linear_batched(descs, gpu)
    torch.cuda.synchronize()
    for i in sorted({0, L - 1}):
        want, wq = oracle_linear_mt(m, n, kb, a[i], [w[i]], [0],
                                    ops=[(k, bits(h)) for k, _, h in plan(i)], pieces=pieces,
                                    onto=start[i].view(np.uint32) if onto else None,
                                    tbuf=tbuf if ops == "acts" else None, quantize=quant)
        got = c[i].cpu().numpy().view(np.uint32)
        gq = q[i].cpu().numpy() if quant else None
        # Per row, as every fast kernel: the rounding of a step's sums is
        # relative to the planes' sums 32 h w and r w, which a block's own sum
        # may cancel (so no bound per element from the block sums); a row's
        # largest output is of their size.
        check_fast(got, want, gq, wq)
        if ops == "operands" and i == L - 1:
            # the wave that saw the byte folds exactly; the fast ops are one
            # IEEE rounding each, as the engine's away from the range's ends
            assert np.array_equal(got[:32, :64], want[:32, :64])


@pytest.mark.parametrize("panels", [False, True])
@pytest.mark.parametrize("layers", [1, 3])
def test_a_words_before_their_w_blocks(gpu, layers, panels):
    """W blocks 16..19 of 20 against A words 0..3: the layer's A base, moved by
    the piece's place, lies before A's first byte, and nothing may be read
    there.  With vector ops and no table, whose unused loads take A's bytes."""
    rng = np.random.default_rng(layers + 10 * panels)
    m, n, kb, first, blocks = (1030 if layers == 1 else 170), 200, 20, 16, 4
    a = [random_a_words(rng, m, blocks) for _ in range(layers)]
    codes = [mxfp4_weights(rng, n, kb * 32) for _ in range(layers)]
    w_d = dev(np.stack([oracle.pack_wbuf(*c) for c in codes]))
    if panels:
        packed = torch.empty((layers, hb.panel_bytes(n, kb)), dtype=torch.uint8, device=DEV)
        for i in range(layers):
            hb.pack_weights(w_d[i], n, kb, packed[i], ctx=gpu)
        w_d = packed
    bias = rng.standard_normal(n).astype(np.float32)
    a_d, b_d = dev(np.stack(a)), dev(bias)
    c = torch.zeros((layers, m, n), device=DEV)
    descs = [hb.linear_desc(m, n, kb, a_d[i], [w_d[i]], [0], c[i], pieces=[(first, blocks, 0)],
                            a_stride=blocks, ops=[(EP_ADDP, b_d), (EP_RELU, None)], mode=hb.FAST,
                            panels=panels) for i in range(layers)]
    print("A before its W blocks", (m, n, layers, panels), flush=True)
    hb.linear_batched(descs, gpu)
    torch.cuda.synchronize()
    for i in range(layers):
        w = oracle.pack_wbuf(*[x[..., first * (x.shape[-1] // kb):] for x in codes[i]])
        want, _ = oracle_linear_mt(m, n, blocks, a[i], [w], [0],
                                   ops=[(EP_ADDP, bias.view(np.uint32)), (EP_RELU, None)])
        check_fast(c[i].cpu().numpy().view(np.uint32), want)
