"""What a host program has the sampler do, as cases that can be timed.

Every case is one pass through the C ABI (include/pz_sampler.h) as a decode
loop calls it: batched sampling from [B, V] fp32 logits that sit in HBM,
speculative verification, softmax of attention scores and of whole rows, and
the bf16 LM head that produces the logits.  Sizes are those of the bench's
workloads (vocabularies 49152, 128256, 151936; hidden size 2560; 32 heads) and
serving batches between them.

A case's "op":
  sample    pz_sample_batch (synchronous: ids in host memory); "mode" greedy,
            topk (chained with top-p when top_p < 1), topp or categorical
  step      pz_sample_step: the RNG states, uniforms and EOS flags on the device
  spec      pz_spec_verify
  softmax   pz_softmax_batch
  attn      pz_attn_softmax, "ragged": every row has its own length
  lmhead    pz_lm_head_bf16, or with "fused" pz_lm_head_argmax_bf16
"""
import ctypes
import functools
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "project-zero_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import pzsample as pz  # noqa: E402

_MOST = 1024 * 128256  # logits of the largest sampling batch


def listed():
    return [
        # one sequence at a time, as the reference's own loop samples: latency
        dict(name="chain_1x49152", op="sample", mode="topk", B=1, V=49152, ld=49152, H=64,
             top_k=40, top_p=0.95, temperature=0.8, rep=1.1, pres=0.0, freq=0.0),
        # nucleus sampling of a serving batch
        dict(name="topp_64x128256", op="sample", mode="topp", B=64, V=128256, ld=128256, H=0,
             top_k=0, top_p=0.9, temperature=0.7, rep=1.0, pres=0.0, freq=0.0),
        # the full chat chain: penalties, top-k, top-p
        dict(name="topk_256x151936", op="sample", mode="topk", B=256, V=151936, ld=151936, H=512,
             top_k=20, top_p=0.8, temperature=1.0, rep=1.0, pres=0.5, freq=0.3),
        # the largest batch: greedy with a repetition penalty, bound by HBM
        dict(name="greedy_1024x128256", op="sample", mode="greedy", B=1024, V=128256, ld=128256,
             H=256, top_k=0, top_p=1.0, temperature=0.0, rep=1.15, pres=0.0, freq=0.0),
        # a mid-size decode step without an aligned row (50257 ids, contiguous
        # rows): plain sampling at temperature 1, everything on the device
        dict(name="step_48x50257", op="step", mode="categorical", B=48, V=50257, ld=50257, H=0,
             top_k=0, top_p=1.0, temperature=1.0, rep=1.0, pres=0.0, freq=0.0),
        # verification of four drafts for 32 sequences
        dict(name="spec_32x4x128256", op="spec", B=32, K=4, V=128256, bonus=True,
             temperature=0.8),
        # probabilities of every token (scoring, log-probabilities)
        dict(name="softmax_64x128256", op="softmax", B=64, V=128256, ld=128256, temperature=1.0),
        # attention scores of a decode step: 64 sequences x 32 heads, each at
        # its own position
        dict(name="attn_2048x4096", op="attn", rows=2048, n=4096, ragged=True),
        # attention scores of one sequence with a long context
        dict(name="attn_32x32768", op="attn", rows=32, n=32768, ragged=False),
        # the LM head of one sequence, of a small and of a large batch
        dict(name="lmhead_1x2560x128256", op="lmhead", B=1, n=2560, V=128256, fused=False),
        dict(name="lmhead_argmax_32x2560x128256", op="lmhead", B=32, n=2560, V=128256, fused=True),
        dict(name="lmhead_256x2560x128256", op="lmhead", B=256, n=2560, V=128256, fused=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["sample", "sample", "step", "spec", "softmax", "attn", "lmhead", "lmhead"])
    V = _log(rng, 8192, 200000)
    if op in ("sample", "step"):
        mode = rng.choice(["greedy", "topk", "topp", "categorical"])
        B = min(_log(rng, 1, 1024), _MOST // V)
        ld = V if rng.random() < 0.5 else (V + 63) // 64 * 64
        pen = mode in ("greedy", "topk") and rng.random() < 0.7
        return dict(op=op, mode=mode, B=B, V=V, ld=ld,
                    H=rng.choice([64, 256, 512]) if pen else 0,
                    top_k=rng.choice([10, 20, 40, 50, 100]) if mode == "topk" else 0,
                    top_p=rng.choice([0.8, 0.9, 0.95]) if mode == "topp" else
                    rng.choice([0.9, 1.0]) if mode == "topk" else 1.0,
                    temperature=0.0 if mode == "greedy" else rng.choice([0.7, 0.8, 1.0]),
                    rep=rng.choice([1.0, 1.1]) if pen else 1.0,
                    pres=0.5 if pen else 0.0, freq=rng.choice([0.0, 0.3]) if pen else 0.0)
    if op == "spec":
        K = rng.randint(1, 8)
        B = max(1, min(_log(rng, 1, 64), _MOST // (V * (2 * K + 1))))
        return dict(op=op, B=B, K=K, V=V, bonus=rng.random() < 0.8,
                    temperature=rng.choice([0.6, 0.8, 1.0]))
    if op == "softmax":
        return dict(op=op, B=min(_log(rng, 1, 256), _MOST // V), V=V,
                    ld=V if rng.random() < 0.5 else (V + 63) // 64 * 64,
                    temperature=rng.choice([0.7, 1.0]))
    if op == "attn":
        n = _log(rng, 64, 32768)
        rows = rng.choice([8, 16, 32]) * _log(rng, 1, 64)
        return dict(op=op, rows=max(8, min(rows, (1 << 23) // n)), n=n, ragged=rng.random() < 0.5)
    n = 64 * rng.randint(16, 64)  # hidden sizes 1024 .. 4096
    V = min(_log(rng, 32000, 200000), 128256 * 2560 // n)
    return dict(op=op, B=_log(rng, 1, 256), n=n, V=V, fused=rng.random() < 0.5)


@functools.lru_cache(maxsize=1)
def _sampler(max_batch, max_vocab, max_hist):
    """One handle per program: its stream and workspaces outlive the inputs."""
    return pz.Sampler(max_batch, max_vocab, max_hist=max_hist)


def _normal(g, shape, sigma):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(sigma)


def _logits(g, case, rows, ld):
    """Logits as the bench draws them: N(0, 3^2), N(0, 2^2) with a few strong
    tokens, or 2.5 x Gumbel."""
    mode, V = case.get("mode", "topp"), case["V"]
    if mode == "greedy":
        return _normal(g, (rows, ld), 3.0)
    if mode == "topk":
        e = torch.empty((rows, ld), device="cuda").exponential_(generator=g)
        return e.clamp_(min=1e-30).log_().mul_(-2.5)
    x = _normal(g, (rows, ld), 2.0)
    at = torch.randint(0, V, (rows, 5), generator=g, device="cuda")
    up = torch.rand((rows, 5), generator=g, device="cuda").mul_(4.0).add_(8.0)
    return x.scatter_add_(1, at, up)


def _history(g, case):
    """Generated ids so far, Zipf(1.1) over the vocabulary."""
    cdf = torch.arange(1, case["V"] + 1, device="cuda", dtype=torch.float64).pow_(-1.1).cumsum_(0)
    u = torch.rand((case["B"], case["H"]), generator=g, device="cuda", dtype=torch.float64)
    ids = torch.searchsorted(cdf, u * cdf[-1].item())
    return ids.clamp_(max=case["V"] - 1).to(torch.int32).contiguous()


def _params(case):
    return [pz.row_params(temperature=case["temperature"], top_k=case["top_k"],
                          top_p=case["top_p"], rep_penalty=case["rep"],
                          presence_penalty=case["pres"], frequency_penalty=case["freq"])]


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 2654435761 % (1 << 62) + 1)
    host = np.random.default_rng(seed + 1)
    op, st = case["op"], {"case": case}
    if op in ("sample", "step"):
        B, V, ld, H = case["B"], case["V"], case["ld"], case["H"]
        s = st["s"] = _sampler(B, V, H)
        st["logits"] = _logits(g, case, B, ld)
        st["hist"] = _history(g, case) if H else None
        if op == "sample":
            st["u"] = host.random(B, dtype=np.float32)
            st["call"] = s.caller(B, V, ld, _params(case), H)
        else:
            s.set_eos([2, V - 1])
            states = host.integers(1, 1 << 63, B, dtype=np.int64)
            st["params"] = _params(case)
            st["state"] = torch.from_numpy(states).cuda()
            st["ids"] = torch.empty(B, dtype=torch.int32, device="cuda")
            st["p"] = torch.empty(B, dtype=torch.float32, device="cuda")
            st["eos"] = torch.empty(B, dtype=torch.uint8, device="cuda")
    elif op == "spec":
        B, K, V = case["B"], case["K"], case["V"]
        KT = K + (1 if case["bonus"] else 0)
        st["s"] = _sampler(B, V, 0)
        st["target"] = _normal(g, (B, KT, V), 2.5)
        st["draft"] = st["target"][:, :K].contiguous()
        st["draft"] += _normal(g, (B, K, V), 0.5)
        q = torch.softmax(st["draft"].reshape(B * K, V) / case["temperature"], dim=1)
        ids = torch.multinomial(q, 1, generator=g).reshape(B, K)
        st["draft_ids"] = np.ascontiguousarray(ids.cpu().numpy().astype(np.int32))
        st["u_acc"] = host.random((B, K), dtype=np.float32)
        st["u_res"] = host.random(B, dtype=np.float32)
        st["acc"] = np.empty(B, np.int32)
        st["out"] = np.empty((B, K + 1), np.int32)
    elif op == "softmax":
        st["s"] = _sampler(case["B"], case["V"], 0)
        st["x"] = _logits(g, case, case["B"], case["ld"])
        st["out"] = torch.zeros_like(st["x"])
    elif op == "attn":
        rows, n = case["rows"], case["n"]
        st["s"] = _sampler(1, 16, 0)
        st["x"] = _normal(g, (rows, n), 3.0)
        st["out"] = torch.zeros_like(st["x"])
        st["len"] = (torch.randint(1, n + 1, (rows,), generator=g, device="cuda")
                     .to(torch.int32) if case["ragged"] else None)
    else:
        B, V, n = case["B"], case["V"], case["n"]
        st["s"] = _sampler(B, V, 0)
        st["w"] = _normal(g, (V, n), 0.02).to(torch.bfloat16)
        st["x"] = _normal(g, (B, n), 1.0)
        if case["fused"]:
            st["ids"] = torch.empty(B, dtype=torch.int32, device="cuda")
        else:
            st["logits"] = torch.empty((B, V), dtype=torch.float32, device="cuda")
    return st


def _ok(rc):
    if rc != pz.PZ_OK:
        raise RuntimeError(f"the sampler returned {rc}")


def run(st):
    """The asynchronous calls run on the sampler's stream and return buffers
    that a later wait makes valid, as for a C caller."""
    c, s = st["case"], st["s"]
    op = c["op"]
    if op == "sample":
        hist = st["hist"].data_ptr() if st["hist"] is not None else None
        return st["call"](st["logits"].data_ptr(), st["u"], hist)
    if op == "step":
        s.sample_step(st["logits"], c["B"], c["V"], c["ld"], st["params"], st["state"],
                      st["ids"], st["p"], st["eos"], st["hist"], c["H"])
        return st["ids"], st["p"], st["eos"], st["state"]
    lib, h = s.lib, s.h
    if op == "spec":
        host = [st[k].ctypes.data_as(ctypes.c_void_p)
                for k in ("draft_ids", "u_acc", "u_res", "acc", "out")]
        _ok(lib.pz_spec_verify(h, st["target"].data_ptr(), st["draft"].data_ptr(), c["B"],
                               c["K"], c["V"], c["V"], int(c["bonus"]), c["temperature"], *host))
        return st["acc"], st["out"]
    if op == "softmax":
        _ok(lib.pz_softmax_batch(h, st["x"].data_ptr(), c["ld"], st["out"].data_ptr(), c["ld"],
                                 c["B"], c["V"], c["temperature"]))
        return st["out"]
    if op == "attn":
        d_len = st["len"].data_ptr() if st["len"] is not None else None
        _ok(lib.pz_attn_softmax(h, st["x"].data_ptr(), c["n"], st["out"].data_ptr(), c["n"],
                                c["rows"], c["n"], d_len))
        return st["out"]
    w, x = st["w"].data_ptr(), st["x"].data_ptr()
    if c["fused"]:
        _ok(lib.pz_lm_head_argmax_bf16(h, w, c["V"], c["n"], x, c["B"], c["n"],
                                       st["ids"].data_ptr()))
        return st["ids"]
    _ok(lib.pz_lm_head_bf16(h, w, c["V"], c["n"], x, c["B"], c["n"], st["logits"].data_ptr(),
                            c["V"]))
    return st["logits"]


def work(case):
    op = case["op"]
    if op in ("sample", "step"):
        # each row read once, its history, uniform or state, and outputs
        return {"bytes": case["B"] * (4 * case["V"] + 4 * case["H"] + (8 if op == "sample" else 25)),
                "flops": 0}
    if op == "spec":
        rows = 2 * case["K"] + (1 if case["bonus"] else 0)
        return {"bytes": case["B"] * (4 * rows * case["V"] + 12 * case["K"] + 12), "flops": 0}
    if op == "softmax":
        return {"bytes": 8 * case["B"] * case["V"], "flops": 0}
    if op == "attn":
        per = (case["n"] + 1) / 2 if case["ragged"] else case["n"]
        return {"bytes": 8 * case["rows"] * per, "flops": 0}
    B, V, n = case["B"], case["V"], case["n"]
    return {"bytes": 2 * V * n + 4 * B * n + (4 * B if case["fused"] else 4 * B * V),
            "flops": 2 * B * V * n}


def tolerance(case):
    """Everything but the LM head is defined bit for bit (sequential fp32 sums
    in id order, the reference's exponential), so ids and probabilities are
    exact.  The LM head's fp32 sums may be taken in any order."""
    if case["op"] == "lmhead":
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.005}
    return "exact"


def _softmax64(x, lens=None):
    """Row softmax in 64 bits, zeros from each row's length on."""
    y = x.double()
    if lens is not None:
        at = torch.arange(x.shape[1], device=x.device)
        y = y.masked_fill(at[None, :] >= lens[:, None], -math.inf)
    return torch.softmax(y, dim=1)


def exact(case, seed):
    op = case["op"]
    if op in ("softmax", "attn", "lmhead"):
        st = prepare(case, seed)
    if op == "softmax":
        out = torch.zeros_like(st["x"], dtype=torch.float64)
        V = case["V"]
        out[:, :V] = _softmax64(st["x"][:, :V].double() / case["temperature"])
        return out
    if op == "attn":
        return _softmax64(st["x"], st["len"])
    if op == "lmhead":
        x = st["x"].double()
        out = torch.empty((case["B"], case["V"]), dtype=torch.float64, device="cuda")
        step = max(1, (1 << 27) // case["n"])
        for r in range(0, case["V"], step):
            out[:, r:r + step] = x @ st["w"][r:r + step].double().t().contiguous()
        return torch.argmax(out, dim=1).to(torch.int32) if case["fused"] else out
    # drawn ids and their probabilities are defined by sequential fp32 sums
    # and have no value in 64 bits
    return None
