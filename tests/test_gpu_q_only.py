"""Layers that keep only their requantized MXINT8 words (C = NULL with
q_out), on an MI355X: the NPU keeps a layer's FP32 result in FBUF and
stores only the ABUF words of the requantize (tools/iss/vec_engine.cpp:
447-458), so the FP32 C need not reach memory.  On every kernel route that
can requantize, the words equal those of the same layer with C given, bit
for bit, and those equal the oracle's (bitwise in exact mode, within the
fast-mode bound otherwise).  The API rejects C = NULL without q_out, with
`onto`, and for pieces at different A offsets (their launches meet in C),
and C or q_out not 4-byte aligned."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers
import hotarubi_amd as hb
from test_gpu_bench_routes import DEV, dev, host, mxfp4_planes, say, to_panels, w8_planes

pytestmark = pytest.mark.gpu


def q_only(gpu, m, n, kb, mode, seed, w8=False, layers=1, ops=None, tbuf=None, panels=False,
           w8_panels=False, fp8=False, pieces=None):
    rng = np.random.default_rng(seed)
    a_h, w_h, w_d = [], [], []
    for _ in range(layers):
        a_h.append(helpers.activations_fp8(rng, m, kb * 32)[1] if fp8
                   else helpers.activations(rng, m, kb * 32)[1])
        planes, modes = w8_planes(rng, n, kb) if w8 else mxfp4_planes(rng, n, kb)
        w_h.append(planes)
    a_d = dev(np.stack(a_h))
    for planes in w_h:
        d = [dev(p) for p in planes]
        if w8_panels:
            pan = torch.empty((hb.w8_panel_bytes(n, kb),), dtype=torch.uint8, device=DEV)
            hb.pack_w8(d[0], d[1], n, kb, pan, ctx=gpu)
            d = [pan, pan]
        elif panels:
            d = [to_panels(gpu, x, n, kb) for x in d]
        w_d.append(d)
    ops = ops or []
    dev_ops = [(k, dev(v.view(np.float32)) if isinstance(v, np.ndarray) else v) for k, v in ops]
    tb_d = dev(tbuf.view(np.int64)) if tbuf is not None else None
    qwords = (m + 3) // 4 * (n // 32)
    results = []
    for with_c in (True, False):
        c = torch.zeros((layers, m, n), dtype=torch.float32, device=DEV) if with_c else None
        q = torch.full((layers, qwords, 144), 0xA5, dtype=torch.uint8, device=DEV)
        descs = [hb.linear_desc(m, n, kb, a_d[i], w_d[i], modes, c[i] if with_c else None,
                                ops=dev_ops, tbuf=tb_d, q_out=q[i], mode=mode, panels=panels,
                                w8_panels=w8_panels, a_fp8=fp8, pieces=pieces)
                 for i in range(layers)]
        torch.cuda.synchronize()
        say("q only", dict(m=m, n=n, kb=kb, mode=mode, w8=w8, layers=layers, panels=panels,
                           w8_panels=w8_panels, fp8=fp8, with_c=with_c))
        hb.linear_batched(descs, gpu)
        results.append(host(q).copy())
    assert np.array_equal(results[0], results[1])
    for i in (0, layers - 1):
        _, wq = helpers.oracle_linear_mt(m, n, kb, a_h[i], w_h[i], modes, ops=ops, tbuf=tbuf,
                                         quantize=True, a_fp8=fp8, pieces=pieces)
        if mode == hb.EXACT:
            assert np.array_equal(results[1][i], wq.reshape(qwords, 144))
        else:
            helpers.check_requantized(results[1][i], wq)


def relu_bias(rng, n):
    return [(hb.EP_ADDP, np.asarray(rng.normal(0, 0.1, n), np.float32).view(np.uint32)),
            (hb.EP_RELU, None)]


def test_wave_kernel_128_columns(gpu):
    """4512 x 960 x 960 MXFP4 (the SmolVLA prefix's q at B = 32)."""
    q_only(gpu, 4512, 960, 30, hb.FAST, seed=900)


def test_wave_kernel_panels_narrow_ops(gpu):
    """The backbone's stage-1 3x3 conv: 67,584 x 64 x 576 over panels, bias
    and ReLU."""
    q_only(gpu, 67584, 64, 18, hb.FAST, seed=901, panels=True,
           ops=relu_bias(np.random.default_rng(1), 64))


@pytest.mark.parametrize("panels", [False, True])
def test_tile_kernel_128_rows(gpu, panels):
    """4096 x 2048 x 160 MXFP4 in two pieces: 256 tiles of 128 rows."""
    q_only(gpu, 4096, 2048, 5, hb.FAST, seed=908, panels=panels, pieces=[(0, 2), (2, 3)],
           ops=relu_bias(np.random.default_rng(5), 2048))


def test_k_split_and_epilogue_kernel(gpu):
    """1100 x 512 x 512, W8: 2 K splits over workgroups, finished by the
    epilogue kernel."""
    q_only(gpu, 1100, 512, 16, hb.FAST, seed=902, w8=True)


def test_split_kernel(gpu):
    """141 rows: the single-launch split kernel, with a bias."""
    q_only(gpu, 141, 960, 30, hb.FAST, seed=903, ops=relu_bias(np.random.default_rng(2), 960)[:1])


def test_skinny_kernel_batched(gpu):
    """A batch of 16-row layers: the skinny kernel."""
    q_only(gpu, 16, 256, 12, hb.FAST, seed=904, layers=4)


@pytest.mark.parametrize("m", [200, 1000])
def test_exact(gpu, m):
    """Exact mode: the exact tile kernel's epilogue, bias and ReLU."""
    q_only(gpu, m, 320, 13, hb.EXACT, seed=905 + m, ops=relu_bias(np.random.default_rng(3), 320))


def test_w8_panels_gelu(gpu):
    """SigLIP's MLP up over W8 panels: bias, GELU and the requantize."""
    rng = np.random.default_rng(4)
    ops = [(hb.EP_MULP, np.asarray(rng.uniform(0.001, 0.02, 3072), np.float32).view(np.uint32)),
           (hb.EP_ADDP, np.asarray(rng.normal(0, 0.1, 3072), np.float32).view(np.uint32)),
           (hb.EP_ACT, None)]
    q_only(gpu, 2048, 3072, 24, hb.FAST, seed=906, w8=True, w8_panels=True, ops=ops,
           tbuf=helpers.activation_table("gelu"))


@pytest.mark.parametrize("m", [141, 2000])
def test_mxfp8(gpu, m):
    """MXFP8 activations: the split kernel (141 rows) and, past 1,024 rows
    with a requantize, the per-output exact fold of the epilogue kernel."""
    q_only(gpu, m, 256, 8, hb.FAST, seed=907 + m, fp8=True)


def test_rejections(gpu):
    a = torch.zeros((4 * 4, 144), dtype=torch.uint8, device=DEV)  # 4 quads x a_stride 4
    w = torch.zeros((4 * 2, 144), dtype=torch.uint8, device=DEV)
    c = torch.zeros((16, 32), dtype=torch.float32, device=DEV)
    q = torch.zeros((4, 144), dtype=torch.uint8, device=DEV)
    for kw in (dict(c=None), dict(c=None, q_out=q, onto=True),
               dict(c=None, q_out=q, a_stride=4, pieces=[(0, 1, 0), (1, 1, 3)]),
               dict(q_out=q.data_ptr() + 2),  # q_out not 4-byte aligned
               dict(c=c.data_ptr() + 2)):  # C not 4-byte aligned
        args = dict(m=16, n=32, kb_total=2, a=a, planes=[w], modes=[0], c=c)
        args.update(kw)
        with pytest.raises(hb.HbError) as err:
            hb.linear(gpu, **args)
        assert err.value.code == hb.HB_EINVAL
