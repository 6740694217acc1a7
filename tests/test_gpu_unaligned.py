"""Rows at any float's address: contiguous rows of an odd number of ids (and a
base pointer off 16 bytes) in every sampling mode, softmax, attention softmax
and verification.  The 16-byte loads they take must stay inside the row: the
last row ends with its buffer, and the entries around the rows are huge, so a
read past either end would be chosen.  Everything identical to the oracle."""
import ctypes

import numpy as np
import pytest

import pz_oracle as po
import pzsample as pz
from conftest import to_dev

pytestmark = pytest.mark.gpu

MODES = {
    "greedy": dict(temperature=0.0),
    "greedy_rep": dict(temperature=0.0, rep_penalty=1.3),
    "categorical": dict(temperature=0.9),
    "topk": dict(temperature=0.8, top_k=40, top_p=0.9),
    "topp": dict(temperature=0.7, top_p=0.9),
}


# vocabularies with remainders 1, 2, 3 and 0 of four, below one load, at a
# segment's and a tile's edge; batches of one workgroup and several per row
@pytest.mark.parametrize("B,V", [(3, 2), (3, 7), (2, 257), (5, 4097), (1, 4098), (9, 16387),
                                 (300, 1023), (2, 50257), (33, 32003)])
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_modes(torch_cuda, B, V, shift):
    print(f"case unaligned B={B} V={V} shift={shift}", flush=True)
    x = pz.synth_normal(B, V, 3.0, 0xA11 + V)
    H = 16
    hist = pz.synth_uniform_ids(B, H, V, 0xA12)
    u = pz.synth_draws(B, 0xA13)
    flat = np.full(B * V + 8, 1e30, np.float32)
    flat[shift:shift + B * V] = x.ravel()
    d_flat = to_dev(torch_cuda, flat)
    d_x = d_flat[shift:shift + B * V]
    d_h = to_dev(torch_cuda, hist)
    with pz.Sampler(B, V, max_hist=H) as s:
        for name, kw in MODES.items():
            ids, p = s.sample(d_x, B, V, V, [pz.row_params(**kw)], u=u, d_hist=d_h, H=H,
                              want_p=True)
            want, wp, _, _ = po.sample_batch(x, [po.params(**kw)], u=u, hist=hist)
            assert (ids == want).all(), (name, np.nonzero(ids != want)[0][:5])
            if not name.startswith("greedy"):
                assert (p.view(np.uint32) == wp.view(np.uint32)).all(), name


@pytest.mark.parametrize("rows,n", [(5, 3), (9, 101), (6, 333), (7, 1001), (5, 2049), (3, 8191),
                                    (2, 20001)])
@pytest.mark.parametrize("shift", [0, 1, 2])
def test_softmaxes(torch_cuda, rows, n, shift):
    print(f"case unaligned softmax rows={rows} n={n} shift={shift}", flush=True)
    x = pz.synth_normal(rows, n, 2.0, 0xA21 + n)
    want = x.copy()
    o = po.oracle()
    for row in want:
        o.orc_softmax(row.ctypes.data_as(ctypes.c_void_p), n)
    flat = np.full(rows * n + 8, 1e30, np.float32)
    flat[shift:shift + rows * n] = x.ravel()
    d_in = to_dev(torch_cuda, flat)
    with pz.Sampler(rows, n) as s:
        for call in (s.softmax, s.attn_softmax):
            d_out = torch_cuda.full((rows * n + 8,), -7.0, dtype=torch_cuda.float32, device="cuda")
            a, b = d_in[shift:shift + rows * n], d_out[shift:shift + rows * n]
            torch_cuda.cuda.synchronize()
            call(a, b, rows, n, n, n)
            s.sync()
            got = d_out.cpu().numpy()
            assert (got[shift:shift + rows * n].view(np.uint32) ==
                    want.ravel().view(np.uint32)).all()
            assert (got[:shift] == -7.0).all() and (got[shift + rows * n:] == -7.0).all()


@pytest.mark.parametrize("V", [257, 4099, 20001])
def test_verification(torch_cuda, V):
    B, K = 3, 2
    print(f"case unaligned verify V={V}", flush=True)
    tgt = pz.synth_normal(B * (K + 1), V, 2.5, 0xA31).reshape(B, K + 1, V)
    dft = pz.synth_perturb(np.ascontiguousarray(tgt[:, :K]).reshape(B * K, V), 0.5,
                           0xA32).reshape(B, K, V)
    ids = pz.synth_draft_ids(dft.reshape(B * K, V), 0.8, 0xA33).reshape(B, K)
    ua, ur = pz.synth_draws(B * K, 0xA34).reshape(B, K), pz.synth_draws(B, 0xA35)
    with pz.Sampler(B, V) as s:
        acc, out = s.spec_verify(to_dev(torch_cuda, tgt), to_dev(torch_cuda, dft), B, K, V, V,
                                 True, 0.8, ids, ua, ur)
    wacc, wout, _ = po.spec_verify(tgt, dft, K, True, 0.8, ids, ua, ur)
    assert (acc == wacc).all() and (out == wout).all()
