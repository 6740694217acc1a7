"""pz_softmax_batch over whole vocabulary rows (softmax.c:4-23 after
apply_temperature): rows split over workgroups above 6144 entries, one
workgroup per row below and where the sampler's workspace does not hold the
rows.  Every probability must be bit-identical to the oracle's, whatever the
path, and the padding of the output stays unwritten."""
import ctypes

import numpy as np
import pytest

import pz_oracle as po
import pzsample as pz
from conftest import to_dev

pytestmark = pytest.mark.gpu


def oracle_rows(x, T, div):
    o = po.oracle()
    want = x.copy()
    for row in want:
        p = row.ctypes.data_as(ctypes.c_void_p)
        o.orc_apply_temperature(p, row.size, ctypes.c_float(T), div)
        o.orc_softmax(p, row.size)
    return want


# the split's edges: one entry past the limit, segment and slice remainders,
# scalar rows (odd strides), one row, more rows than a launch's target
@pytest.mark.parametrize("B,V,ld", [(3, 6144, 6144), (3, 6145, 6145), (5, 6400, 6404),
                                    (1, 50257, 50257), (7, 8191, 8200), (2, 16385, 16388),
                                    (600, 7001, 7004), (33, 128256, 128256)])
@pytest.mark.parametrize("div", [0, 1])
def test_softmax_rows(torch_cuda, B, V, ld, div):
    if div and B > 33:
        pytest.skip("the temperature's form does not depend on the batch")
    print(f"case softmax B={B} V={V} ld={ld} div={div}", flush=True)
    rng = np.random.default_rng(V + div)
    x = (rng.standard_normal((B, V), dtype=np.float32) * 2.0).astype(np.float32)
    if B >= 3:
        x[0, V // 3] = np.nan           # a NaN: every output NaN
        x[1, V - 1] = 40.0              # the maximum is the last entry
        x[2, :V // 2] = -np.inf         # an empty first half
    if B >= 5:
        x[3, 5] = np.inf                # an infinite maximum
        x[4] = np.float32(np.finfo(np.float32).min)  # the lowest value everywhere
    want = oracle_rows(x, 0.7, div)
    full = np.full((B, ld), 1e30, np.float32)
    full[:, :V] = x
    with pz.Sampler(B, V) as s, pz.Sampler(1, 16) as small:
        for q in (s, small):  # the second holds no such rows: one workgroup each
            q.set_temp_mode(div)
            d_in = to_dev(torch_cuda, full)
            d_out = torch_cuda.full((B, ld), -7.0, dtype=torch_cuda.float32, device="cuda")
            q.softmax(d_in, d_out, B, V, ld, ld, temperature=0.7)
            q.softmax(d_in, d_in, B, V, ld, ld, temperature=0.7)  # in place
            q.sync()
            got, inp = d_out.cpu().numpy(), d_in.cpu().numpy()
            for r in (got, inp):
                ok = (r[:, :V].view(np.uint32) == want.view(np.uint32)) | (
                    np.isnan(r[:, :V]) & np.isnan(want))
                assert ok.all(), np.argwhere(~ok)[:5]
            assert (got[:, V:] == -7.0).all() and (inp[:, V:] == 1e30).all()
