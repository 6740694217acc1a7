"""LM head on the device (pz_lm_head_bf16) and its fused greedy epilogue
(pz_lm_head_argmax_bf16).

Logits: against the exact product (float64 of the same bf16 weights and fp32
activations), within the fp32 summation bound the header states:
|gpu - exact| <= n * 2^-24 * sum_j |w_ij x_bj| (any order of n fp32 adds and
products is inside it).  Fused ids: bit for bit the reference argmax
(orc_argmax, argmax.c:3-13) of the unfused kernel's logits, and the ids the
batched sampler's greedy path gives on those logits."""
import numpy as np
import pytest

import pz_oracle as po
import pzsample as pz
from conftest import to_dev

pytestmark = pytest.mark.gpu


def bf16_bits(a):
    """fp32 -> bf16 bit patterns, round to nearest even."""
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    r = (u + 0x7FFF + ((u >> 16) & 1)) >> 16
    return r.astype(np.uint16)


def bf16_to_f64(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def weights(V, n, seed, scale=0.02):
    rng = np.random.default_rng(seed)
    return bf16_bits(rng.standard_normal((V, n), dtype=np.float32) * scale)


def exact(wb, x):
    """float64 product and the summation bound, row blocks of W."""
    V = wb.shape[0]
    B = x.shape[0]
    xd = x.astype(np.float64)
    out = np.empty((B, V))
    bound = np.empty((B, V))
    step = max(1, (1 << 25) // wb.shape[1])  # 256 MiB of float64 per block
    for r0 in range(0, V, step):
        wd = bf16_to_f64(wb[r0:r0 + step])
        out[:, r0:r0 + step] = xd @ wd.T
        bound[:, r0:r0 + step] = np.abs(xd) @ np.abs(wd).T
    return out, bound


def run(torch, wb, x, s, offset=0):
    V, n = wb.shape
    B = x.shape[0]
    if offset:
        flat = np.zeros(V * n + offset, np.uint16)
        flat[offset:] = wb.ravel()
        d_flat = to_dev(torch, flat.view(np.int16))
        d_w = d_flat.data_ptr() + 2 * offset
    else:
        d_flat = to_dev(torch, wb.view(np.int16))
        d_w = d_flat.data_ptr()
    d_x = to_dev(torch, x)
    d_l = torch.full((B, V), -7.0, dtype=torch.float32, device="cuda")
    d_i = torch.full((B,), -9, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    s.lm_head(d_w, V, n, d_x, B, n, d_l, V)
    s.lm_head_argmax(d_w, V, n, d_x, B, n, d_i)
    s.sync()
    logits = d_l.cpu().numpy()
    ids = d_i.cpu().numpy()
    # the batched sampler's greedy path on the same device logits
    gids, _ = s.sample(d_l, B, V, V, [pz.row_params(temperature=0.0)])
    del d_flat
    return logits, ids, gids


def check(label, wb, x, logits, ids, gids, check_logits=True):
    n = wb.shape[1]
    if check_logits:
        ex, bound = exact(wb, x)
        err = np.abs(logits.astype(np.float64) - ex)
        tol = n * 2.0 ** -24 * bound + 1e-30
        worst = float((err / tol).max())
        print(f"{label}: max |err| / bound = {worst:.4f}, max |err| = {err.max():.3e}", flush=True)
        assert (err <= tol).all(), label
    o = po.oracle()
    want = np.array([o.orc_argmax(np.ascontiguousarray(r).ctypes.data_as(po._P), r.size)
                     for r in logits], np.int32)
    assert (ids == want).all(), (label, ids, want)
    assert (gids == ids).all(), (label, gids, ids)


@pytest.mark.parametrize("B", [1, 3, 8, 17])
def test_lm_head_batches(torch_cuda, B):
    V, n = 32000, 2048
    print(f"case lmhead V={V} n={n} B={B}", flush=True)
    wb = weights(V, n, 0x1A0 + B)
    x = np.random.default_rng(B).standard_normal((B, n), dtype=np.float32)
    with pz.Sampler(32, V) as s:
        check(f"B{B}", wb, x, *run(torch_cuda, wb, x, s))


def test_lm_head_full_vocab(torch_cuda):
    """BitNet b1.58-2B-4T shape: vocab 128256, hidden 2560, one sequence."""
    V, n = 128256, 2560
    print(f"case lmhead full V={V} n={n}", flush=True)
    wb = weights(V, n, 0x1B0)
    x = np.random.default_rng(7).standard_normal((1, n), dtype=np.float32)
    with pz.Sampler(4, V) as s:
        check("full", wb, x, *run(torch_cuda, wb, x, s))


@pytest.mark.parametrize("n,offset", [(2050, 0), (2048, 1), (37, 0), (24576, 0)])
def test_lm_head_odd_shapes(torch_cuda, n, offset):
    """n not a multiple of 8 and a weight pointer off 16-byte alignment (the
    element-load path), a tiny n, and the largest n the LDS tile holds."""
    V = 4099
    print(f"case lmhead n={n} offset={offset}", flush=True)
    wb = weights(V, n, 0x1C0 + n)
    x = np.random.default_rng(n).standard_normal((5, n), dtype=np.float32)
    with pz.Sampler(8, V) as s:
        check(f"n{n}o{offset}", wb, x, *run(torch_cuda, wb, x, s, offset=offset))


def test_fused_argmax_ties_and_nan(torch_cuda):
    V, n = 3000, 512
    rng = np.random.default_rng(0x1D0)
    w = rng.standard_normal((V, n), dtype=np.float32) * 0.01
    x = rng.standard_normal((4, n), dtype=np.float32)
    # rows 1500 and 700 identical and dominant for x[0]: equal logits, lowest id
    w[1500] = np.sign(x[0]) * 0.5
    w[700] = w[1500]
    # x[1] NaN: every logit NaN, argmax returns 0
    x[1, 3] = np.nan
    # an inf weight in row 0: logit 0 is -inf for x[0] and x[3], NaN for
    # x[2] (inf times a zero activation)
    w[0, 5] = np.inf
    x[0, 5] = -1.0
    x[2, 5] = 0.0
    # x[3] zero but for that one activation, which meets a zero weight in
    # every other row: logit 0 = -inf, every other logit +0 or -0, so the
    # first of them (id 1) wins
    w[1:, 5] = 0.0
    x[3] = 0.0
    x[3, 5] = -1.0
    wb = bf16_bits(w)
    print("case lmhead ties and nan", flush=True)
    with pz.Sampler(8, V) as s:
        logits, ids, gids = run(torch_cuda, wb, x, s)
    assert ids[0] == 700
    assert ids[1] == 0 and np.isnan(logits[1]).all()
    assert np.isnan(logits[2, 0]) and ids[2] == 0
    assert ids[3] == 1
    check("ties", wb, x, logits, ids, gids, check_logits=False)


# edges of the matrix-core paths: batch blocks of 16 .. 256, two chunks of 256,
# row tiles of 256, k below one step, off a step and off a stage, with and
# without the workspace (tests/test_lmhead_tiles.py says which path each takes)
TILE_CASES = [
    (4, 1, 8), (16, 129, 40), (17, 255, 96), (32, 4099, 1048), (33, 257, 72), (64, 512, 2560),
    (65, 1000, 104), (128, 4099, 2056), (129, 300, 32), (256, 4099, 264), (257, 513, 160),
    (530, 1025, 64), (9, 1025, 2048), (40, 800, 4096), (20, 40000, 136), (100, 70001, 72),
    (200, 70001, 24), (90, 700, 24576), (5, 66000, 328), (16, 66000, 40), (32, 66001, 72),
    (17, 300, 248)]
# vocabularies for which the other tile shapes are chosen: the 256 x 256 tile
# with an odd number of k-steps and an end off a step, the 64-row tile, and W
# past the Infinity Cache in every tile that then loads it non-temporally
LARGE_CASES = [
    (200, 33000, 40), (256, 65003, 72), (229, 40001, 104), (48, 33000, 40), (64, 40001, 104),
    (8, 131201, 1032), (20, 131201, 1032), (60, 131201, 1032), (100, 131201, 1032)]


@pytest.mark.parametrize("B,V,n", TILE_CASES)
def test_lm_head_matrix_core_tiles(torch_cuda, B, V, n):
    """The GEMM's edges, unfused against float64 and fused against the argmax of
    the unfused logits; row V // 2 holds an infinite weight (its logits are
    +-inf by the sign of the activation it meets)."""
    torch = torch_cuda
    print(f"case lmhead tiles B={B} V={V} n={n}", flush=True)
    rng = np.random.default_rng(B * 7 + n)
    w = rng.standard_normal((V, n), dtype=np.float32) * 0.02
    x = rng.standard_normal((B, n), dtype=np.float32)
    r = V // 2
    wb = bf16_bits(w)
    finite = wb.copy()
    wb[r, n - 1] = 0x7F80
    finite[r] = 0
    with pz.Sampler(B, max(V, 16)) as s:
        logits, ids, gids = run(torch, wb, x, s)
        # rows longer than their entries, off 16 bytes
        ld, ldx = V + 3, n + 5
        d_w = to_dev(torch, wb.view(np.int16))
        d_x = torch.full((B, ldx), float("nan"), dtype=torch.float32, device="cuda")
        d_x[:, :n] = to_dev(torch, x)
        d_l = torch.full((B, ld), -7.0, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        s.lm_head(d_w.data_ptr(), V, n, d_x, B, ldx, d_l, ld)
        s.sync()
        padded = d_l.cpu().numpy()
    assert (logits[:, r] == np.copysign(np.inf, x[:, n - 1])).all()
    assert (padded[:, :V].view(np.int32) == logits.view(np.int32)).all()
    assert (padded[:, V:] == -7.0).all()
    want = np.array([po.oracle().orc_argmax(
        np.ascontiguousarray(q).ctypes.data_as(po._P), q.size) for q in logits], np.int32)
    assert (ids == want).all() and (gids == ids).all()
    logits[:, r] = 0.0
    ex, bound = exact(finite, x)
    err = np.abs(logits.astype(np.float64) - ex)
    tol = n * 2.0 ** -24 * bound + 1e-30
    print(f"B{B} V{V} n{n}: max |err| / bound = {float((err / tol).max()):.4f}", flush=True)
    assert (err <= tol).all()


# row lengths around the multiples of 2048 (rows of W a multiple of 4 KiB
# apart) and short ones with and without the workspace, batches in every tile
# of the GEMM and in more than one chunk
@pytest.mark.parametrize("n", [64, 72, 256, 264, 2048, 2056, 2560, 4096, 6144])
def test_equal_rows_give_equal_logits(torch_cuda, n):
    """From four batch rows on, a logit depends on its row of W and its
    activations alone: not on where the row lies in the vocabulary, on the
    batch row or on the batch.  Equal rows of W in different row tiles tie, so
    the fused argmax returns the lowest of their ids."""
    torch = torch_cuda
    rng = np.random.default_rng(n)
    period, V = 200, 1100
    base = bf16_bits(rng.standard_normal((period, n), dtype=np.float32) * 0.02)
    wb = np.ascontiguousarray(np.tile(base, (V // period + 1, 1))[:V])
    x7 = rng.standard_normal((7, n), dtype=np.float32)
    first = None
    with pz.Sampler(300, V) as s:
        for B in (4, 16, 40, 64, 100, 130, 256, 300):
            print(f"case lmhead equal rows n={n} B={B}", flush=True)
            logits, ids, gids = run(torch, wb, np.ascontiguousarray(x7[np.arange(B) % 7]), s)
            bits = logits.view(np.int32)
            if first is None:
                first = run(torch, base, x7, s)[0].view(np.int32)
            want = first[np.arange(B) % 7][:, np.arange(V) % period]
            assert (bits == want).all(), (B, np.argwhere(bits != want)[:3])
            assert (ids < period).all() and (gids == ids).all()


@pytest.mark.parametrize("B", [4, 37])
def test_rows_past_the_parts_workspace(torch_cuda, B):
    """Rows of W longer than the workspace of the activations' parts serves
    (131072 weights): the call queues its launches and nothing else -- no
    device memory is taken -- and the sums are the ones of shorter rows, so
    eight more zero weights change no bit."""
    torch = torch_cuda
    V, n = 300, 131072
    print(f"case lmhead long rows B={B}", flush=True)
    rng = np.random.default_rng(B)
    w = rng.standard_normal((V, n), dtype=np.float32) * 0.02
    x = rng.standard_normal((B, n), dtype=np.float32)
    wb = bf16_bits(w)
    longer = np.concatenate([wb, np.zeros((V, 8), np.uint16)], axis=1)
    xl = np.concatenate([x, rng.standard_normal((B, 8), dtype=np.float32)], axis=1)
    with pz.Sampler(64, V) as s:
        logits, ids, gids = run(torch, wb, x, s)
        check(f"long{B}", longer, xl, *run(torch, longer, xl, s))
        got = run(torch, longer, xl, s)
        assert (got[0].view(np.int32) == logits.view(np.int32)).all()
        assert (got[1] == ids).all()
        longer[V // 2, n + 7] = 0x7F80
        got = run(torch, longer, xl, s)[0]
        assert (got[:, V // 2] == np.copysign(np.inf, xl[:, n + 7])).all()
    # twice the length: nothing is allocated (the first call loads the kernels)
    d_w = torch.zeros((16, 2 * n + 8), dtype=torch.int16, device="cuda")
    d_x = torch.ones((B, 2 * n + 8), dtype=torch.float32, device="cuda")
    d_l = torch.empty((B, 16), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    with pz.Sampler(64, V) as s:
        s.lm_head(d_w.data_ptr(), 16, n, d_x, B, n, d_l, 16)
        s.sync()
        free = torch.cuda.mem_get_info()[0]
        s.lm_head(d_w.data_ptr(), 16, 2 * n + 8, d_x, B, 2 * n + 8, d_l, 16)
        s.sync()
        assert torch.cuda.mem_get_info()[0] == free
    assert (d_l == 0).all()


@pytest.mark.parametrize("B,V,n", LARGE_CASES)
def test_lm_head_large_tiles(torch_cuda, B, V, n):
    """The tile shapes of large vocabularies: W repeats 331 rows, one of them
    with an infinite weight, so every logit is known from the first 331 (those
    against float64); rows longer than their entries, off 16 bytes."""
    torch = torch_cuda
    print(f"case lmhead large tiles B={B} V={V} n={n}", flush=True)
    rng = np.random.default_rng(B + n)
    P, r = 331, 100
    base = bf16_bits(rng.standard_normal((P, n), dtype=np.float32) * 0.02)
    x = rng.standard_normal((B, n), dtype=np.float32)
    finite = base.copy()
    finite[r] = 0
    base[r, n - 1] = 0x7F80
    d_w = to_dev(torch, base.view(np.int16)).repeat(V // P + 1, 1)[:V].contiguous()
    ld, ldx = V + 3, n + 5
    d_x = torch.full((B, ldx), float("nan"), dtype=torch.float32, device="cuda")
    d_x[:, :n] = to_dev(torch, x)
    d_l = torch.full((B, ld), -7.0, dtype=torch.float32, device="cuda")
    d_i = torch.full((B,), -9, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    with pz.Sampler(B, V) as s:
        s.lm_head(d_w.data_ptr(), V, n, d_x, B, ldx, d_l, ld)
        s.lm_head_argmax(d_w.data_ptr(), V, n, d_x, B, ldx, d_i)
        s.sync()
    logits = d_l.cpu().numpy()
    ids = d_i.cpu().numpy()
    first = logits[:, :P].copy()
    assert (logits[:, :V].view(np.int32) == first.view(np.int32)[:, np.arange(V) % P]).all()
    assert (logits[:, V:] == -7.0).all()
    want = np.array([po.oracle().orc_argmax(
        np.ascontiguousarray(q).ctypes.data_as(po._P), q.size) for q in first], np.int32)
    assert (ids == want).all()
    assert (first[:, r] == np.copysign(np.inf, x[:, n - 1])).all()
    first[:, r] = 0.0
    ex, bound = exact(finite, x)
    err = np.abs(first.astype(np.float64) - ex)
    tol = n * 2.0 ** -24 * bound + 1e-30
    print(f"B{B} V{V} n{n}: max |err| / bound = {float((err / tol).max()):.4f}", flush=True)
    assert (err <= tol).all()
