"""The work this library is timed on: a decode step's attention at several
batch sizes, context lengths and pool formats, prefill attention, cache
maintenance (gather, block copy and append), a layer's projections and whole
greedy generations, each through the Python entry points.

A case is a dict with an "op" and that op's sizes.  ``prepare`` makes what a
serving program holds before the call, ``run`` makes one pass, ``exact``
repeats it in float64 with plain torch.
"""
from __future__ import annotations

import math

import torch

from rustral_amd import kv, model

DEV = "cuda:0"
BS = 16  # tokens per block
TOP = {"int8": 127.0, "fp8": 448.0}
ELEM = {"f32": 4, "bf16": 2, "int8": 1, "fp8": 1}
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16}


def listed() -> list[dict]:
    heads = dict(hq=32, hkv=8, d=128)  # Llama-3-8B's attention layer
    return [
        # one user's chat turn: latency and launches are all there is
        dict(name="decode_single", op="decode", seqs=1, lo=300, hi=300, kv="bf16",
             append=True, **heads),
        # one GPU's share of a 64-sequence batch over 8 GPUs, the step's K/V row
        # appended by the attention call as a model's layer does it
        dict(name="decode_share", op="decode", seqs=8, lo=512, hi=4096, kv="bf16", append=True,
             **heads),
        # the headline: one decode step's attention for 64 sequences
        dict(name="decode_batch", op="decode", seqs=64, lo=512, hi=4096, kv="bf16", append=False,
             **heads),
        # long documents: few sequences, split-K over many partitions
        dict(name="decode_long", op="decode", seqs=8, lo=16384, hi=65536, kv="bf16", append=False,
             **heads),
        # the 64-sequence batch over a quantized cache, with its append
        dict(name="decode_int8", op="decode", seqs=64, lo=512, hi=4096, kv="int8", append=True,
             **heads),
        # new requests admitted together: 25 prompts of 128 tokens
        dict(name="prefill_admit", op="prefill", seqs=25, new=128, cached=0, kv="bf16", **heads),
        # one chunk of 512 tokens of 8 long prompts, 3,584 tokens already cached
        dict(name="prefill_chunk", op="prefill", seqs=8, new=512, cached=3584, kv="bf16",
             **heads),
        # the batch's cache read back into contiguous tensors (eviction, hand-over)
        dict(name="gather_batch", op="gather", seqs=64, lo=512, hi=4096, kv="bf16", out="bf16",
             hkv=8, d=128),
        # a scheduler step's cache upkeep in 8 layers: a quarter of the blocks
        # relocated, then one token of 64 sequences appended
        dict(name="cache_step", op="cache", layers=8, blocks=2048, pairs=512, tokens=64,
             kv="bf16", hkv=8, d=128),
        # a decode step's attention input (layer norm, q / k / v, append) for 64
        # sequences at Llama-3-8B's layer sizes
        dict(name="qkv_batch", op="qkv", tokens=64, d_model=4096, kv="bf16", ln=True, **heads),
        # the same layer's output projection
        dict(name="linear_out", op="linear", rows=64, n_in=4096, n_out=4096, bias=False),
        # the small decoder end to end: 32 prompt tokens, 64 new ones
        dict(name="generate", op="generate", prompt=32, new=64, batch_seed=0),
    ]


def _log(rng, lo: int, hi: int) -> int:
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    op = rng.choice(["decode", "decode", "decode", "prefill", "gather", "cache", "qkv", "linear",
                     "generate"])
    hkv, group, d = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4, 4, 8]), rng.choice([64, 128])
    heads = dict(hq=hkv * group, hkv=hkv, d=d)
    row = 2 * hkv * d  # K and V elements of one token
    if op == "decode":
        fmt = rng.choice(["bf16", "bf16", "f32", "int8", "fp8"])
        hi = _log(rng, 64, 65536)
        room = int(1.0e9 / (row * ELEM[fmt] * hi))  # at most about the long case's bytes
        seqs = _log(rng, 1, max(1, min(64, room)))
        return dict(op=op, seqs=seqs, lo=_log(rng, max(1, hi // 16), hi), hi=hi, kv=fmt,
                    append=fmt != "f32" and rng.random() < 0.5, **heads)
    if op == "prefill":
        new, cached = _log(rng, 2, 512), rng.choice([0, 0, _log(rng, 16, 3584)])
        return dict(op=op, seqs=_log(rng, 1, 8 if new > 128 else 25), new=new, cached=cached,
                    kv=rng.choice(["bf16", "bf16", "f32"]), **heads)
    if op == "gather":
        fmt = rng.choice(["bf16", "f32", "int8", "fp8"])
        out = rng.choice(["bf16", "f32"]) if fmt == "bf16" else "f32"
        hi = _log(rng, 64, 4096)
        return dict(op=op, seqs=_log(rng, 1, 64 if out == "bf16" else 32),
                    lo=_log(rng, max(1, hi // 8), hi), hi=hi, kv=fmt, out=out, hkv=hkv, d=d)
    if op == "cache":
        blocks = _log(rng, 64, 2048)
        return dict(op=op, layers=rng.randint(1, 8), blocks=blocks, pairs=_log(rng, 1, blocks // 4),
                    tokens=_log(rng, 1, blocks // 4), kv=rng.choice(["bf16", "f32"]),
                    hkv=hkv // 2 or 1, d=d)
    if op == "qkv":
        d_model = 32 * _log(rng, 4, 128) + rng.choice([0, 0, 4, 7])
        return dict(op=op, tokens=_log(rng, 1, 64), d_model=d_model,
                    kv=rng.choice(["bf16", "f32"]), ln=rng.random() < 0.75, **heads)
    if op == "linear":
        n_in, n_out = _log(rng, 128, 8192), _log(rng, 32, 4096)
        return dict(op=op, rows=_log(rng, 1, 64 if n_in <= 4096 else 32),
                    n_in=n_in if rng.random() < 0.3 else 4 * (n_in // 4), n_out=n_out,
                    bias=rng.random() < 0.5)
    prompt = rng.randint(1, 64)
    return dict(op=op, prompt=prompt, new=rng.randint(1, min(64, 128 - prompt)),
                batch_seed=rng.randint(0, 9))


# ---- inputs ------------------------------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(1_000_003 * (seed % 1_000_000) + 17)


def _lens(case: dict) -> list[int]:
    """Context lengths, uniform in [lo, hi]: part of the case, so that every
    seed of a case is the same amount of work."""
    g = torch.Generator().manual_seed(7 * case["seqs"] + 31 * case["hi"] + case["lo"])
    return torch.randint(case["lo"], case["hi"] + 1, (case["seqs"],), generator=g).tolist()


def _tables(lens: list[int], g: torch.Generator):
    """Block tables over randomly permuted blocks, the lengths, and the pool's
    block count (a few blocks stay free)."""
    need = [-(-n // BS) for n in lens]
    nb = sum(need) + 8
    perm = torch.randperm(nb, generator=g, device=DEV).to(torch.int32)
    tab = torch.full((len(lens), max(need)), -1, dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(need):
        tab[b, :n] = perm[at:at + n]
        at += n
    return tab, torch.tensor(lens, dtype=torch.int32, device=DEV), nb


def _randn(shape, g: torch.Generator, dtype=torch.float32) -> torch.Tensor:
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _quantize(x: torch.Tensor, fmt: str):
    """Rows of x (last dim) as bytes and one fp32 scale per row."""
    amax = x.abs().amax(-1, keepdim=True)
    y = x * (TOP[fmt] / amax)
    if fmt == "int8":
        b = y.round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
    else:
        b = y.clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    return b, (amax / TOP[fmt]).squeeze(-1).contiguous()


def _pools(nb: int, hkv: int, d: int, fmt: str, g: torch.Generator):
    """K and V pools of N(0, 1) rows, with scale pools for the 1-byte formats."""
    k, v = (_randn((nb, hkv, BS, d), g) for _ in range(2))
    if fmt in TOP:
        (kb, ks), (vb, vs) = _quantize(k, fmt), _quantize(v, fmt)
        return kb, vb, ks, vs
    return k.to(TORCH[fmt]), v.to(TORCH[fmt]), None, None


def prepare(case: dict, seed: int) -> dict:
    g = _gen(seed)
    st = dict(case=case)
    if case["op"] in ("decode", "prefill", "gather"):
        lens = ([case["cached"] + case["new"]] * case["seqs"] if case["op"] == "prefill"
                else _lens(case))
        st["tab"], st["ctx"], nb = _tables(lens, g)
        st["k"], st["v"], st["ks"], st["vs"] = _pools(nb, case["hkv"], case["d"], case["kv"], g)
    if case["op"] == "decode":
        B, hq, hkv, d = case["seqs"], case["hq"], case["hkv"], case["d"]
        st["q"], st["out"] = _randn((B, hq, d), g), torch.empty((B, hq, d), device=DEV)
        if case["append"]:
            st["kn"], st["vn"] = _randn((B, hkv, d), g), _randn((B, hkv, d), g)
        st["max_context"] = st["tab"].shape[1] * BS
        need = kv.workspace_bytes(B, hq, d, st["max_context"])
        st["ws"] = torch.empty(max(need, 16), dtype=torch.uint8, device=DEV)
    elif case["op"] == "prefill":
        rows = case["seqs"] * case["new"]
        st["q"] = _randn((rows, case["hq"], case["d"]), g)
        st["out"] = torch.empty_like(st["q"])
        st["start"] = torch.arange(0, rows + 1, case["new"], dtype=torch.int32, device=DEV)
    elif case["op"] == "gather":
        per = [n * case["hkv"] * case["d"] for n in lens]
        off = [sum(per[:i]) for i in range(len(per))]
        st["off"] = torch.tensor(off, dtype=torch.int64, device=DEV)
        st["total"] = sum(per)
        st["ko"], st["vo"] = (torch.empty(st["total"], dtype=TORCH[case["out"]], device=DEV)
                              for _ in range(2))
    elif case["op"] == "cache":
        n, nb, hkv, d = case["layers"], case["blocks"], case["hkv"], case["d"]
        dt = TORCH[case["kv"]]
        st["k"], st["v"] = (torch.empty((n, nb, hkv, BS, d), dtype=dt, device=DEV)
                            for _ in range(2))
        for p in (st["k"], st["v"]):
            for layer in range(n):
                p[layer] = _randn((nb, hkv, BS, d), g, dt)
        # disjoint sources, destinations and appended blocks
        perm = torch.randperm(nb, generator=g, device=DEV)
        src, dst = perm[:case["pairs"]].sort()[0], perm[case["pairs"]:2 * case["pairs"]].sort()[0]
        st["pairs"] = torch.stack([src, dst], 1).to(torch.int32).contiguous()
        blk = perm[2 * case["pairs"]:2 * case["pairs"] + case["tokens"]]
        row = torch.randint(0, BS, (case["tokens"],), generator=g, device=DEV)
        st["slots"] = (blk * BS + row).to(torch.int64)
        st["kn"], st["vn"] = (_randn((n, case["tokens"], hkv, d), g) for _ in range(2))
    elif case["op"] == "qkv":
        t, dm, hkv, d = case["tokens"], case["d_model"], case["hkv"], case["d"]
        st["x"] = _randn((t, dm), g)
        std = 0.02
        st["wq"] = _randn((case["hq"] * d, dm), g) * std
        st["wk"], st["wv"] = (_randn((hkv * d, dm), g) * std for _ in range(2))
        st["ln"] = (1 + 0.1 * _randn((dm,), g), 0.1 * _randn((dm,), g)) if case["ln"] else None
        nb = 2 * t + 8
        st["k"], st["v"] = (torch.zeros((nb, hkv, BS, d), dtype=TORCH[case["kv"]], device=DEV)
                            for _ in range(2))
        blk = torch.randperm(nb, generator=g, device=DEV)[:t]
        row = torch.randint(0, BS, (t,), generator=g, device=DEV)
        st["slots"] = (blk * BS + row).to(torch.int64)
    elif case["op"] == "linear":
        st["x"] = _randn((case["rows"], case["n_in"]), g)
        st["w"] = _randn((case["n_out"], case["n_in"]), g) * 0.02
        st["b"] = _randn((case["n_out"],), g) if case["bias"] else None
    elif case["op"] == "generate":
        st["cfg"] = model.config()
        st["params"] = model.init_params(st["cfg"], seed=case["batch_seed"] + 10 * (seed % 1000))
        st["dec"] = model.Decoder(st["cfg"], st["params"])
        st["prompt"] = torch.randint(0, st["cfg"].vocab, (case["prompt"],), generator=g,
                                     device=DEV).to(torch.int32).cpu().numpy()
    return st


# ---- one pass ------------------------------------------------------------------------

def run(st: dict):
    case = st["case"]
    op = case["op"]
    if op == "decode":
        common = dict(max_context=st["max_context"], out=st["out"], workspace=st["ws"])
        if case["kv"] in TOP:
            scales = (st["ks"], st["vs"])
            if case["append"]:
                kv.decode_attention_append_q(st["q"], st["k"], st["v"], *scales, st["kn"],
                                             st["vn"], st["tab"], st["ctx"], None, case["kv"],
                                             **common)
                return st["out"], st["k"], st["v"], st["ks"], st["vs"]
            kv.decode_attention_q(st["q"], st["k"], st["v"], *scales, st["tab"], st["ctx"], None,
                                  case["kv"], **common)
            return (st["out"],)
        if case["append"]:
            kv.decode_attention_append(st["q"], st["k"], st["v"], st["kn"], st["vn"], st["tab"],
                                       st["ctx"], **common)
            return st["out"], st["k"], st["v"]
        kv.decode_attention(st["q"], st["k"], st["v"], st["tab"], st["ctx"], **common)
        return (st["out"],)
    if op == "prefill":
        return kv.prefill_attention(st["q"], st["k"], st["v"], st["tab"], st["start"], st["ctx"],
                                    max_q_len=case["new"], out=st["out"])
    if op == "gather":
        packed = dict(out_offsets=st["off"], out_total=st["total"], k_out=st["ko"],
                      v_out=st["vo"])
        if case["kv"] in TOP:
            return kv.gather_q(st["k"], st["v"], st["ks"], st["vs"], st["tab"], st["ctx"],
                               case["kv"], **packed)
        return kv.gather(st["k"], st["v"], st["tab"], st["ctx"], out_dtype=TORCH[case["out"]],
                         **packed)
    if op == "cache":
        kv.copy_blocks(st["k"], st["v"], st["pairs"])
        kv.append(st["k"], st["v"], st["kn"], st["vn"], st["slots"])
        return st["k"], st["v"]
    if op == "qkv":
        ln_g, ln_b = st["ln"] if st["ln"] else (None, None)
        q = model.qkv_append(st["x"], st["wq"], st["wk"], st["wv"], st["k"], st["v"], st["slots"],
                             ln_g=ln_g, ln_b=ln_b)
        return q, st["k"], st["v"]
    if op == "linear":
        return model.linear(st["x"], st["w"], st["b"])
    return st["dec"].generate(st["prompt"], case["new"], logits=True)


# ---- what a pass cannot do without -----------------------------------------------------

def work(case: dict) -> dict:
    op = case["op"]
    if op in ("decode", "gather"):
        lens, hkv, d = _lens(case), case["hkv"], case["d"]
        row = d * ELEM[case["kv"]] + (4 if case["kv"] in TOP else 0)
        pool = sum(lens) * 2 * hkv * row
        if op == "gather":
            return dict(bytes=pool + sum(lens) * 2 * hkv * d * ELEM[case["out"]], flops=0)
        new = case["seqs"] * 2 * hkv * (4 * d + row) if case["append"] else 0
        return dict(bytes=pool + 8 * case["seqs"] * case["hq"] * d + new + 4 * sum(lens) // BS,
                    flops=4 * d * case["hq"] * sum(lens))
    if op == "prefill":
        n, L, d = case["new"], case["cached"] + case["new"], case["d"]
        pairs = n * case["cached"] + n * (n + 1) // 2
        return dict(bytes=case["seqs"] * (8 * n * case["hq"] * d
                                          + 2 * L * case["hkv"] * d * ELEM[case["kv"]]),
                    flops=4 * d * case["hq"] * pairs * case["seqs"])
    if op == "cache":
        row = case["hkv"] * case["d"]
        e = ELEM[case["kv"]]
        return dict(bytes=2 * case["layers"] * row * (2 * case["pairs"] * BS * e
                                                      + case["tokens"] * (4 + e)), flops=0)
    if op == "qkv":
        cols, dm = (case["hq"] + 2 * case["hkv"]) * case["d"], case["d_model"]
        out = case["hq"] * 4 + 2 * case["hkv"] * ELEM[case["kv"]]
        return dict(bytes=4 * cols * dm + case["tokens"] * (4 * dm + out * case["d"]),
                    flops=2 * case["tokens"] * cols * dm)
    if op == "linear":
        r, i, o = case["rows"], case["n_in"], case["n_out"]
        return dict(bytes=4 * (i * o + r * i + r * o), flops=2 * r * i * o)
    cfg = model.CONFIG0
    n = 2 * (4 * cfg["d_model"] ** 2 + 2 * cfg["d_model"] * cfg["d_ff"])
    head = cfg["vocab"] * cfg["d_model"]
    steps = case["prompt"] + case["new"] - 1
    return dict(bytes=4 * (n + 2 * head + case["new"] * cfg["vocab"]),
                flops=2 * (n * steps + head * case["new"]))


# Largest relative errors: four times what the library shows against float64
# (2-norm; element over the larger of its value and the result's RMS).  bf16
# pool rows of a projection may also round the other way where a sum lies
# within its error of a tie: one step (2^-7) in about a thousandth of them.
TOLERANCE = {
    "decode": {"rel": 1.5e-5, "max": 1.2e-4},
    "prefill": {"rel": 2.6e-5, "max": 1.8e-4},
    "qkv": {"rel": 5e-6, "max": 7e-5},
    "linear": {"rel": 5e-6, "max": 3.5e-5},
    "generate": {"rel": 4e-6, "max": 2e-5},
}


def tolerance(case: dict):
    if case["op"] in ("gather", "cache"):  # copies, and one product per dequantized element
        return "exact"
    if case["op"] == "qkv" and case["kv"] == "bf16":
        return {"rel": 4e-4, "max": 8e-3}
    return TOLERANCE[case["op"]]


# ---- the same in float64 -----------------------------------------------------------------

def _values(pool: torch.Tensor, scale, fmt: str) -> torch.Tensor:
    if fmt not in TOP:
        return pool.double()
    b = pool.view(torch.int8 if fmt == "int8" else torch.float8_e4m3fn)
    return b.float().double() * scale.double().unsqueeze(-1)


def _contiguous(st: dict, pool: str, b: int, n: int) -> torch.Tensor:
    """Sequence b's first n rows [hkv, n, d] in float64."""
    ids = st["tab"][b, :-(-n // BS)].long()
    scale = st[pool + "s"][ids] if st[pool + "s"] is not None else None
    x = _values(st[pool][ids], scale, st["case"]["kv"])  # [blocks, hkv, BS, d]
    return x.transpose(0, 1).reshape(x.shape[1], -1, x.shape[3])[:, :n]


def _attend(q, k, v, first=None):
    """q [n, hq, d] over k, v [hkv, L, d]: row i sees positions 0 .. first + i
    (all of them without first)."""
    n, hq, d = q.shape
    hkv = k.shape[0]
    qg = q.double().reshape(n, hkv, hq // hkv, d).permute(1, 2, 0, 3)
    out = torch.empty((hkv, hq // hkv, n, d), dtype=torch.float64, device=q.device)
    for h in range(hkv):
        s = (qg[h].reshape(-1, d) @ k[h].T.contiguous() / math.sqrt(d)).view(-1, n, k.shape[1])
        if first is not None:
            pos = torch.arange(k.shape[1], device=q.device)
            s = s.masked_fill(pos > first + torch.arange(n, device=q.device)[:, None], -math.inf)
        out[h] = (s.softmax(-1).reshape(-1, k.shape[1]) @ v[h].contiguous()).view(-1, n, d)
    return out.permute(2, 0, 1, 3).reshape(n, hq, d)


def _write_rows(pool: torch.Tensor, slots: torch.Tensor, rows: torch.Tensor) -> None:
    """Rows [tokens, hkv, ...] to slots of a layer's pool [nb, hkv, BS, ...]."""
    pool[slots // BS, :, slots % BS] = rows.to(pool.dtype)


def _layer_norm(x, g, b, eps=1e-5):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], g.double(), b.double(), eps)


def exact(case: dict, seed: int):
    st = prepare(case, seed)
    op = case["op"]
    if op == "decode":
        lens = st["ctx"].tolist()
        pools = ()
        if case["append"]:
            p = torch.tensor(lens, device=DEV) - 1
            blk = st["tab"].long().gather(1, (p // BS)[:, None])[:, 0]
            slots = blk * BS + p % BS
            names = ["k", "v"]
            for n in names:
                rows = st[n + "n"]
                if case["kv"] in TOP:
                    rows, scale = _quantize(rows, case["kv"])
                    _write_rows(st[n + "s"], slots, scale)
                _write_rows(st[n], slots, rows)
            pools = tuple(st[n] for n in (names + ["ks", "vs"] if case["kv"] in TOP else names))
        out = torch.stack([_attend(st["q"][b:b + 1], _contiguous(st, "k", b, n),
                                   _contiguous(st, "v", b, n))[0] for b, n in enumerate(lens)])
        return (out, *pools)
    if op == "prefill":
        n, L = case["new"], case["cached"] + case["new"]
        return torch.cat([_attend(st["q"][b * n:(b + 1) * n], _contiguous(st, "k", b, L),
                                  _contiguous(st, "v", b, L), case["cached"])
                          for b in range(case["seqs"])])
    if op == "gather":
        return tuple(torch.cat([_contiguous(st, pool, b, n).reshape(-1)
                                for b, n in enumerate(st["ctx"].tolist())]) for pool in "kv")
    if op == "cache":
        src, dst = st["pairs"].long().T
        for p, new in ((st["k"], st["kn"]), (st["v"], st["vn"])):
            for layer in range(case["layers"]):
                p[layer][dst] = p[layer][src]
                _write_rows(p[layer], st["slots"], new[layer])
        return st["k"], st["v"]
    if op == "qkv":
        x = st["x"].double()
        if st["ln"]:
            x = _layer_norm(x, *st["ln"])
        k, v = st["k"].double(), st["v"].double()
        for p, w in ((k, st["wk"]), (v, st["wv"])):
            _write_rows(p, st["slots"], (x @ w.double().T).view(-1, case["hkv"], case["d"]))
        return x @ st["wq"].double().T, k, v
    if op == "linear":
        y = st["x"].double() @ st["w"].double().T
        return y if st["b"] is None else y + st["b"].double()
    return _generate64(st)


def _generate64(st: dict):
    """Greedy generation with a float64 decoder and a contiguous cache."""
    cfg, new = st["cfg"], st["case"]["new"]
    d, f, heads = cfg.d_model, cfg.d_ff, cfg.n_heads
    kvd = cfg.n_kv_heads * (d // heads)
    flat = torch.from_numpy(st["params"]).double()
    at = 0

    def take(*shape):
        nonlocal at
        n = math.prod(shape)
        at += n
        return flat[at - n:at].view(shape)

    embed = take(cfg.vocab, d)
    shapes = dict(g1=(d,), h1=(d,), wq=(d, d), bq=(d,), wk=(kvd, d), bk=(kvd,), wv=(kvd, d),
                  bv=(kvd,), wo=(d, d), bo=(d,), g2=(d,), h2=(d,), w1=(f, d), b1=(f,), w2=(d, f),
                  b2=(d,))
    layers = [{n: take(*s) for n, s in shapes.items()} for _ in range(cfg.n_layers)]
    gf, hf, head = take(d), take(d), take(cfg.vocab, d)
    i = torch.arange(d)
    angle = torch.arange(cfg.max_seq)[:, None] / 10000.0 ** ((i // 2 * 2).double() / d)
    pe = torch.where(i % 2 == 0, angle.sin(), angle.cos())
    ids = torch.from_numpy(st["prompt"]).long()
    cache = [[torch.zeros((0, cfg.n_kv_heads, d // heads), dtype=torch.float64)] * 2
             for _ in layers]
    tokens, logits, at_pos = [], [], 0
    for _ in range(new):
        n = len(ids)
        x = embed[ids] + pe[at_pos:at_pos + n]
        for w, c in zip(layers, cache):
            h = _layer_norm(x, w["g1"], w["h1"], cfg.eps)
            for j, (m, b) in enumerate((("wk", "bk"), ("wv", "bv"))):
                c[j] = torch.cat([c[j], (h @ w[m].T + w[b]).view(n, cfg.n_kv_heads, -1)])
            q = (h @ w["wq"].T + w["bq"]).view(n, heads, -1)
            o = _attend(q, c[0].transpose(0, 1), c[1].transpose(0, 1), at_pos)
            x = x + o.reshape(n, d) @ w["wo"].T + w["bo"]
            h = _layer_norm(x, w["g2"], w["h2"], cfg.eps) @ w["w1"].T + w["b1"]
            x = x + torch.nn.functional.gelu(h, approximate="tanh") @ w["w2"].T + w["b2"]
        logits.append(_layer_norm(x[-1], gf, hf, cfg.eps) @ head.T)
        tokens.append(int(logits[-1].argmax()))
        at_pos += n
        ids = torch.tensor([tokens[-1]])
    return torch.tensor(tokens, dtype=torch.int32).numpy(), torch.stack(logits).numpy()
