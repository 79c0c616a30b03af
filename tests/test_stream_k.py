"""The keyed GEMM's stream-K split with fewer key slots than workgroups: the
sum over a tile's segments reads only those that a workgroup wrote.

The schedule is checked on the CPU for every slot count up to twice the
workgroups (tests/cpp/stream_k.cxx).  On the device the partial buffer is left
dirty by a larger call, then problems of a few dozen pairs run through it: one
tree, the grouped graph, and learned orders, whose classes hold a few slots each.
Bars: against the FP64 M2L per pair, a BF16x3 sum of same-signed terms, 3 x 2^-17
relative for p and eight times that for F (terms of both signs); learned orders
against the same orders without stream-K, which adds the same FP32 products in
another order: the same bars.
"""
import os
import shutil
import subprocess

import numpy as np
import pytest

from conftest import ROOT
from minimal_amd import fmm
from minimal_amd.inputs import BODY_DTYPE, plummer_background, rel_l2

torch = pytest.importorskip("torch")

BOUND = 3 * 2.0 ** -17


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ missing")
def test_schedule(tmp_path):
    exe = str(tmp_path / "stream_k")
    subprocess.run(["g++", "-std=c++17", "-O2", os.path.join(ROOT, "tests", "cpp", "stream_k.cxx"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def _blobs(seed, n=60):
    """Two blobs in opposite corners: few pairs on each of several levels."""
    rng = np.random.default_rng(seed)
    b = np.zeros(2 * n, BODY_DTYPE)
    b["X"][:n] = rng.random((n, 3)) * 0.3
    b["X"][n:] = 0.7 + rng.random((n, 3)) * 0.3
    b["q"] = (0.5 + rng.random(2 * n)) / (2 * n)
    return b


def _dirty():
    b = plummer_background(20000, 3)
    b["q"] = 1e3 * np.abs(b["q"])
    return b


def _exact(b0, P):
    f = fmm.FMM(P=P, ncrit=40, theta=0.4, m2l_precision=fmm.PREC_FP64)
    b = b0.copy()
    f.evaluate(b)
    w = f.work_counts()
    f.close()
    assert 0 < w["m2l_pairs"] < 128  # slots <= pairs < workgroups (256, or 128 per row block)
    return b


def _close(b, ref):
    assert np.array_equal(b["X"], ref["X"])
    assert rel_l2(b["p"], ref["p"]) <= BOUND
    assert rel_l2(b["F"], ref["F"]) <= 8 * BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("P", [4, 10, 12, 16])
def test_few_slots(gpu, monkeypatch, P):
    monkeypatch.setenv("EXAFMM_GEMM_SK_ONLY", "1")
    f = fmm.FMM(P=P, ncrit=40, theta=0.4)
    for seed in range(3):
        d = _dirty()
        f.evaluate(d)
        b = _blobs(seed)
        f.evaluate(b)
        _close(b, _exact(_blobs(seed), P))


@pytest.mark.gpu
def test_few_slots_grouped(gpu):
    probs = [(_blobs(10 + i), (6, 12)[i % 2]) for i in range(4)]
    ctxs = [fmm.FMM(P=P, ncrit=40, theta=0.4) for _, P in probs]

    def evaluate(sets):
        devs = []
        for f, x in zip(ctxs, sets):
            d = torch.from_numpy(x.view(np.uint8).copy()).cuda()
            torch.cuda.synchronize()
            f.evaluate(d.data_ptr(), n=len(x), on_device=True)
            f.synchronize()
            devs.append(d)
        return devs

    large = evaluate([_dirty()] * len(probs))
    g = fmm.Graph(ctxs, grouped=True)
    g.launch()
    g.synchronize()
    g.close()  # its partial buffer returns to the allocator
    devs = evaluate([b for b, _ in probs])
    g = fmm.Graph(ctxs, grouped=True)
    for _ in range(3):
        g.launch()
        g.synchronize()
        for (b, P), d in zip(probs, devs):
            _close(d.cpu().numpy().view(BODY_DTYPE), _exact(b, P))
        x = torch.ones(1 << 20, device="cuda").sum()
        assert float(x) == float(1 << 20)
    g.close()


@pytest.mark.gpu
def test_few_slots_learned(gpu, monkeypatch):
    t = fmm.FMM(P=14, ncrit=64, theta=0.4)
    t.build_tree(plummer_background(20000, 8))
    t.upward()
    t.horizontal()
    t.train_order_model(nsamples=2048, epochs=20)
    w = t.order_model()
    t.close()
    _exact(_blobs(0), 14)
    orders = set()
    for tol in (-3.0, -4.5, -6.0):
        out = []
        # one sum over all classes, a sum per class, no stream-K
        for env, how in (("EXAFMM_GEMM_SK_ONLY", "1"), ("EXAFMM_GEMM_SK_ONLY", "class"), ("EXAFMM_GEMM_NO_SK", "1")):
            with monkeypatch.context() as m:
                m.setenv(env, how)
                f = fmm.FMM(P=14, ncrit=40, theta=0.4, order_policy=fmm.ORDER_LEARNED)
                f.set_order_model(w, tol)
                d = _dirty()
                f.evaluate(d)
                b = _blobs(0)
                f.evaluate(b)
                orders |= set(np.nonzero(f.order_stats())[0])
                f.close()
            out.append(b)
        _close(out[0], out[2])
        _close(out[1], out[2])
    assert len(orders) > 1
