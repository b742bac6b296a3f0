"""The workloads whose speed this library is kept to, and how to run and check one.

A case is a dict of plain values:

  B, Lq, Lk, Hq, Hkv, d   sizes ([B, L, H, d] tensors; flex: [B, H, L, d])
  dtype                   "bf16", "fp16" or "fp32" (Q, K and V)
  out                     "fp32" (the default output dtype) or "same" (the input's)
  grad                    True: forward and backward, False: forward alone
  api                     "map" (masked_attention_via_map) or "flex" (flex_attention)
  kernel                  "default" (softmax scale 1/sqrt(d)) or "threshold" (scale 1,
                          which runs at precision "highest")
  unit                    True: N(0, 1) inputs, False: N(0, 1) times d^-0.25
  mask                    "none"; "causal"; "window" (causal, q - k <= window);
                          "docs" (packed documents of mean length `docs`, causal);
                          "sparse" (random 128 x 128 tiles per head at `density`, the
                          diagonal ones on, causal inside those); "strided"
                          (q % period == k % period, causal)

prepare() makes what a training or serving step has in hand (tensors on the GPU
and the mask's function or block mask), run() is one step through the public
functions, exact() the same in float64 by plain torch operations.
"""
import math
import random

import numpy as np
import torch

import jaxmodules_amd as jm
from jaxmodules_amd import masks

TILE = 128
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(B, L, H, d, *, Lk=None, Hkv=None, dtype="bf16", out="fp32", grad=True, api="map", kernel="default",
          unit=False, mask="causal", **more):
    return dict(B=B, Lq=L, Lk=Lk or L, Hq=H, Hkv=Hkv or H, d=d, dtype=dtype, out=out, grad=grad, api=api,
                kernel=kernel, unit=unit, mask=mask, **more)


def listed():
    cases = {
        # A call as small as the test suites and unit-sized models make: float32 (the
        # arrays' default type), forward only; latency and launches are all it costs.
        "fp32_causal_small_fwd": _case(2, 128, 8, 64, dtype="fp32", grad=False, unit=True),
        # One layer of a small model's training step in bf16: still mostly launches.
        "bf16_small_flex_train": _case(2, 1024, 8, 64, api="flex", out="same"),
        # A mid-sized model trained in float32, the type a program has that sets none.
        "fp32_causal_train": _case(2, 2048, 8, 64, dtype="fp32", unit=True),
        # The headline workload: one long causal sequence, training.
        "bf16_causal_8k_train": _case(1, 8192, 32, 128),
        # A prompt batch served with grouped KV heads: forward only, 16-bit output.
        "bf16_gqa_prefill": _case(4, 4096, 32, 128, Hkv=8, out="same", grad=False),
        # Sliding-window training over long sequences (short rows of tiles).
        "bf16_window_16k_train": _case(2, 16384, 16, 128, mask="window", window=512),
        # Block-sparse training, a tile table of its own for each head, d = 64.
        "bf16_block_sparse_train": _case(1, 8192, 32, 64, mask="sparse", density=0.25),
        # Packed documents, a long context, training.
        "bf16_documents_32k_train": _case(1, 32768, 8, 128, mask="docs", docs=2048),
        # The strided mask of very long sequences (every 2048th key), float16.
        "fp16_strided_128k_train": _case(1, 131072, 1, 64, dtype="fp16", unit=True, mask="strided", period=2048),
        # Cross attention of odd lengths and a head dimension the kernels pad.
        "fp16_cross_ragged_train": _case(2, 1000, 12, 80, Lk=1511, dtype="fp16", mask="none"),
        # Wide heads: d = 256 in bf16, training.
        "bf16_wide_heads_train": _case(1, 4096, 8, 256),
        # The sharp kernel (scale 1), which runs at "highest" precision, training.
        "bf16_threshold_train": _case(1, 2048, 8, 64, kernel="threshold", unit=True),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sized(rng, cap, make):
    """make(rng) until its work is at most `cap` flop."""
    while True:
        c = make(rng)
        if work(c)["flops"] <= cap:
            return c


def draw(rng: random.Random):
    def heads(r):
        hkv = r.choice((1, 2, 4, 8))
        return hkv * r.choice((1, 1, 2, 4)), hkv

    def causal(r):       # training or prefill in 16 bits, every common head dimension
        hq, hkv = heads(r)
        return _case(r.choice((1, 1, 2, 3, 4)), _log(r, 256, 8192), hq, r.choice((64, 64, 96, 128, 128)), Hkv=hkv,
                     dtype=r.choice(("bf16", "bf16", "fp16")), out=r.choice(("fp32", "same")),
                     grad=r.random() < 0.7, mask=r.choice(("causal", "causal", "none")))

    def flex(r):         # the same through flex_attention (lengths of whole blocks of 128)
        hq, hkv = heads(r)
        return _case(r.choice((1, 2, 4)), 128 * _log(r, 2, 32), hq, r.choice((64, 128)), Hkv=hkv, api="flex",
                     out=r.choice(("fp32", "same")), grad=r.random() < 0.7, mask=r.choice(("causal", "none")))

    def window(r):
        hq, hkv = heads(r)
        return _case(r.choice((1, 2)), _log(r, 1024, 16384), hq, r.choice((64, 128)), Hkv=hkv, mask="window",
                     window=_log(r, 64, 2048))

    def docs(r):
        return _case(r.choice((1, 2)), _log(r, 2048, 32768), r.choice((4, 8)), r.choice((64, 128)), mask="docs",
                     docs=_log(r, 128, 4096))

    def sparse(r):
        return _case(1, _log(r, 1024, 8192), r.choice((8, 16, 32)), r.choice((64, 128)), mask="sparse",
                     density=round(r.uniform(0.1, 0.5), 3))

    def strided(r):
        period = 2 ** r.randint(6, 11)
        return _case(1, period * r.randint(8, 64), r.choice((1, 2)), 64, dtype=r.choice(("fp16", "bf16")),
                     unit=True, mask="strided", period=period)

    def cross(r):
        hq, hkv = heads(r)
        return _case(r.choice((1, 2, 4)), _log(r, 16, 1500) * 2 + 1, hq, r.choice((40, 64, 80, 128)), Lk=_log(r, 33, 3000),
                     Hkv=hkv, dtype=r.choice(("fp16", "bf16")), mask="none")

    def fp32(r):
        hq, hkv = heads(r)
        return _case(r.choice((1, 2, 4)), _log(r, 64, 4096), hq, r.choice((32, 64, 64, 128)), Hkv=hkv, dtype="fp32",
                     grad=r.random() < 0.7, unit=True, mask=r.choice(("causal", "causal", "none", "window")),
                     window=256)

    def wide(r):
        hq, hkv = heads(r)
        return _case(r.choice((1, 2)), _log(r, 128, 4096), hq, r.choice((160, 192, 256, 256)), Hkv=hkv,
                     dtype=r.choice(("bf16", "bf16", "fp16")), grad=r.random() < 0.7,
                     mask=r.choice(("causal", "none")))

    def threshold(r):
        return _case(r.choice((1, 2)), _log(r, 64, 4096), r.choice((2, 4, 8)), r.choice((64, 128)),
                     dtype=r.choice(("bf16", "bf16", "fp32")), kernel="threshold", unit=True,
                     mask=r.choice(("causal", "none")))

    # 16-bit problems on the matrix cores up to the headline workload's size; the
    # float32-precision ones up to the time of the listed wide-head step
    make, cap = rng.choice(((causal, 1.9e12), (flex, 1.9e12), (window, 1.9e12), (docs, 1.9e12), (sparse, 1.9e12),
                            (strided, 1.9e12), (cross, 1.9e12), (fp32, 1.2e11), (wide, 2.0e11), (threshold, 5e10)))
    return _sized(rng, cap, make)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _doc_ids(case, seed):
    """Document id of each position: geometric lengths of mean `docs`, at least 64."""
    rng = np.random.default_rng([seed, 71])
    lens = []
    while sum(lens) < case["Lq"]:
        lens.append(max(64, int(rng.geometric(1.0 / case["docs"]))))
    return np.repeat(np.arange(len(lens)), lens)[:case["Lq"]]


def _tiles(case, seed):
    """[H, tiles, tiles] 0 / 1 / 2 (diagonal: causal inside), as masks.tile_table takes them."""
    rng = np.random.default_rng([seed, 73])
    nt = -(-case["Lq"] // TILE)
    t = (rng.random((case["Hq"], nt, nt)) < case["density"]).astype(np.uint8)
    t[:, np.arange(nt), np.arange(nt)] = 2
    return t


def _tensors(case, seed):
    """Q, K, V and the upstream gradient (None without a backward), [B, L, H, d]
    or, for flex, [B, H, L, d]."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dt, d = DTYPES[case["dtype"]], case["d"]
    scale = 1.0 if case["unit"] else d ** -0.25

    def rand(L, H, dtype, s):
        shape = (case["B"], H, L, d) if case["api"] == "flex" else (case["B"], L, H, d)
        return (torch.randn(shape, generator=gen, device="cuda") * s).to(dtype)

    q = rand(case["Lq"], case["Hq"], dt, scale)
    k = rand(case["Lk"], case["Hkv"], dt, scale)
    v = rand(case["Lk"], case["Hkv"], dt, scale)
    do = rand(case["Lq"], case["Hq"], dt if case["out"] == "same" else torch.float32, 1.0) if case["grad"] else None
    return q, k, v, do


def prepare(case, seed):
    q, k, v, do = _tensors(case, seed)
    if case["grad"]:
        q, k, v = (x.requires_grad_() for x in (q, k, v))
    call = dict(out_dtype=DTYPES[case["dtype"]] if case["out"] == "same" else None)
    mask = case["mask"]
    if case["api"] == "flex":
        if mask == "causal":
            call["block_mask"] = jm.BlockMask.causal_mask(1, 1, case["Lq"], case["Lk"], TILE)
        call["enable_gqa"] = case["Hq"] != case["Hkv"]
    else:
        if mask == "causal":
            call["is_causal"] = True
        elif mask == "window":
            call["mask_fn"] = masks.intersect(masks.causal(), masks.window(case["window"], 0))
            if case["window"] + 2 * TILE <= case["Lk"]:  # a wider one than the sequence is refused
                call["window_size"], call["block_size"] = (case["window"], 0), TILE
        elif mask == "docs":
            call["mask_fn"] = masks.intersect(masks.documents(_doc_ids(case, seed)), masks.causal())
        elif mask == "sparse":
            call["mask_fn"] = masks.intersect(masks.tile_table(_tiles(case, seed)), masks.causal())
        elif mask == "strided":
            call["mask_fn"] = masks.intersect(masks.same_residue(case["period"]), masks.causal())
        if case["Lq"] != case["Lk"]:  # lengths that differ are padded to a common block
            call["block_size"] = TILE
        if case["kernel"] == "threshold":
            call["kernel_fn"] = jm.threshold_kernel()
    return dict(fn=jm.flex_attention if case["api"] == "flex" else jm.masked_attention_via_map,
                q=q, k=k, v=v, do=do, call=call)


def run(state):
    q, k, v, do = state["q"], state["k"], state["v"], state["do"]
    o = state["fn"](q, k, v, **state["call"])
    if do is None:
        return {"o": o}
    dq, dk, dv = torch.autograd.grad(o, (q, k, v), do)
    return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what it has to give
# ---------------------------------------------------------------------------


def _pairs(case):
    """Allowed (query, key) pairs of one (batch, head), on average over the seeds
    where the mask is drawn."""
    n, m = case["Lq"], case["Lk"]
    mask = case["mask"]
    if mask == "none":
        return n * m
    q = np.arange(n)
    if mask == "causal":
        return int(np.minimum(q + 1, m).sum())
    if mask == "window":
        return int(np.minimum(q + 1, case["window"] + 1).sum())
    if mask == "strided":
        return int((q // case["period"] + 1).sum())
    if mask == "docs":
        tot = 0
        for s in range(4):
            lens = np.bincount(_doc_ids(case, s)).astype(np.int64)
            tot += int((lens * (lens + 1) // 2).sum())
        return tot // 4
    nt = -(-n // TILE)
    diag = sum(w * (w + 1) // 2 for w in [min(TILE, n - TILE * i) for i in range(nt)])
    off = n * n - sum(min(TILE, n - TILE * i) ** 2 for i in range(nt))
    return int(diag + case["density"] * off)


def work(case):
    """The unmasked pairs' products (4 d forward, 10 d backward a pair) and every
    input read and output written once."""
    B, Hq, Hkv, d = case["B"], case["Hq"], case["Hkv"], case["d"]
    flops = (14 if case["grad"] else 4) * d * B * Hq * _pairs(case)
    es = 4 if case["dtype"] == "fp32" else 2
    eo = es if case["out"] == "same" else 4
    nq, nk = B * Hq * case["Lq"] * d, B * Hkv * case["Lk"] * d
    bytes_ = es * (nq + 2 * nk) + eo * nq
    if case["grad"]:
        bytes_ += eo * nq + es * (nq + 2 * nk)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """Relative errors against exact() measured on the listed cases and draws, times
    about four: 16-bit outputs are rounded to 8 (bf16) or 11 (fp16) significant
    bits, 1.7e-3 or 2.1e-4 of their norm, and the 16-bit kernels' operands to 11
    bits; float32 sums are 1e-7 to 1e-6 off."""
    if case["dtype"] == "fp32":
        return {"rel": 5e-6}
    if case["dtype"] == "fp16":
        return {"rel": 1.5e-3}
    return {"rel": 8e-3}


def _allowed(case, seed, q0, q1, h, aux):
    """Boolean [q1 - q0, Lk] on the GPU, or None where every pair is allowed."""
    mask = case["mask"]
    if mask == "none":
        return None
    q = torch.arange(q0, q1, device="cuda")[:, None]
    k = torch.arange(case["Lk"], device="cuda")[None, :]
    m = q >= k
    if mask == "window":
        m &= q - k <= case["window"]
    elif mask == "docs":
        m &= aux[q] == aux[k]
    elif mask == "strided":
        m &= (q - k) % case["period"] == 0
    elif mask == "sparse":
        t = aux[h][q // TILE, k // TILE]
        m = (t == 1) | ((t == 2) & m)
    return m


def exact(case, seed):
    q, k, v, do = _tensors(case, seed)
    if case["api"] == "flex":
        q, k, v, do = (None if x is None else x.transpose(1, 2) for x in (q, k, v, do))
    d = case["d"]
    scale = 1.0 if case["kernel"] == "threshold" else 1.0 / math.sqrt(d)
    aux = None
    if case["mask"] == "docs":
        aux = torch.from_numpy(_doc_ids(case, seed)).cuda()
    elif case["mask"] == "sparse":
        aux = torch.from_numpy(_tiles(case, seed)).cuda()
    G = case["Hq"] // case["Hkv"]
    f64 = dict(dtype=torch.float64, device="cuda")
    o = torch.empty(q.shape, **f64)
    if case["grad"]:
        dq = torch.empty(q.shape, **f64)
        dk, dv = torch.zeros(k.shape, **f64), torch.zeros(v.shape, **f64)
    chunk = max(128, min(2048, (1 << 27) // case["Lk"]))
    for b in range(case["B"]):
        for h in range(case["Hq"]):
            hk = h // G
            kh, vh = k[b, :, hk].double(), v[b, :, hk].double()
            for q0 in range(0, case["Lq"], chunk):
                q1 = min(case["Lq"], q0 + chunk)
                qc = q[b, q0:q1, h].double()
                s = (qc @ kh.T).mul_(scale)
                ok = _allowed(case, seed, q0, q1, h, aux)
                if ok is not None:
                    s.masked_fill_(~ok, float("-inf"))
                s.sub_(s.amax(1, keepdim=True)).exp_()
                p = s.div_(s.sum(1, keepdim=True))
                oc = p @ vh
                o[b, q0:q1, h] = oc
                if case["grad"]:
                    g = do[b, q0:q1, h].double()
                    dv[b, :, hk] += p.T @ g
                    ds = (g @ vh.T).sub_((g * oc).sum(1, keepdim=True)).mul_(p).mul_(scale)
                    dq[b, q0:q1, h] = ds @ kh
                    dk[b, :, hk] += ds.T @ qc
    out = {"o": o}
    if case["grad"]:
        out.update(dq=dq, dk=dk, dv=dv)
    if case["api"] == "flex":
        out = {n: x.transpose(1, 2) for n, x in out.items()}
    return out
