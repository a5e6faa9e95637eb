"""The timed workloads of the erasure-coding engine, one pass each through its public entry points.

Four kinds of work, as a training job's checkpoint path meets them:

  flat    k equal-size shards on the GPU: ``xor_encode``, ``rs_encode``, ``reconstruct``, or the same call
          prepared once as a ``ShardPlan``.  ``place`` "own": every shard a tensor of its own; "views": the
          shards lie back to back in one flat fp32 buffer (an optimizer's or a gradient buffer cut in k), so
          they start at any multiple of 4 bytes, and a rebuild writes into that buffer in place.
  ragged  a rank's ordered tensor list cut into units and stripes: ``StripeLayout.encode``, a prepared decode,
          a prepared parity update.  ``place`` "own": tensors at 64-byte starts; "views": back to back in one
          flat buffer.
  save    ``GpuSliceCodec.encode``: the whole save of a rank's state, coded on the GPU and staged to host memory.
  load    ``GpuSliceCodec.decode``: slices in host memory back to tensors on the GPU, lost positions rebuilt.

Bytes stand in for serialized state: fp32 or bf16 normal values.
"""
import math
import random

import numpy as np
import torch

import __graft_entry__

KiB, MiB = 1 << 10, 1 << 20
TOP_BYTES = 20_800_000_000   # one rank's checkpoint buffer of a 1.3B-parameter GPT


def _pkg():
    return __graft_entry__.load_package()


def listed():
    return [
        # the smallest call: XOR parity of a few small shards (an RNG or scheduler state), latency only
        {"name": "xor4_64k", "kind": "flat", "op": "xor", "call": "eager", "place": "own",
         "k": 4, "m": 1, "e": 1, "nbytes": 64 * KiB},
        # serialized blobs have odd byte sizes: the size smoke() codes
        {"name": "rs63_1m_odd", "kind": "flat", "op": "encode", "call": "eager", "place": "own",
         "k": 6, "m": 3, "e": 3, "nbytes": MiB + 5},
        # the benchmark's headline: optimizer-state shards coded again and again through one plan
        {"name": "rs63_256m", "kind": "flat", "op": "encode", "call": "plan", "place": "own",
         "k": 6, "m": 3, "e": 3, "nbytes": 256 * MiB},
        # a load that lost three of nine shards of a flat fp32 buffer and rebuilds them in place
        {"name": "rs63_rebuild_views", "kind": "flat", "op": "decode", "call": "eager", "place": "views",
         "k": 6, "m": 3, "e": 3, "nbytes": 24 * MiB + 4},
        # a wide code over many ranks' shards (k and m past the fully unrolled kernels)
        {"name": "rs24_8_32m", "kind": "flat", "op": "encode", "call": "eager", "place": "own",
         "k": 24, "m": 8, "e": 8, "nbytes": 32 * MiB},
        # a small state of small tensors (norms, biases, adapters) in small units
        {"name": "ragged42_small", "kind": "ragged", "op": "encode", "place": "own", "dtype": "bf16",
         "k": 4, "m": 2, "e": 2, "unit": 4 * KiB, "n": 300, "lo": 256, "hi": 64 * KiB, "sizes": 1},
        # a rank's whole ragged state, 64 KiB units: the save's parity
        {"name": "ragged124", "kind": "ragged", "op": "encode", "place": "own", "dtype": "fp32",
         "k": 12, "m": 4, "e": 4, "unit": 64 * KiB, "n": 900, "lo": 4 * KiB, "hi": 64 * MiB, "sizes": 2},
        # the load of the same state with four positions of every stripe lost
        {"name": "ragged124_decode", "kind": "ragged", "op": "decode", "place": "own", "dtype": "fp32",
         "k": 12, "m": 4, "e": 4, "unit": 64 * KiB, "n": 900, "lo": 4 * KiB, "hi": 64 * MiB, "sizes": 3},
        # a save in which about one byte in a hundred changed: fold the change in, refresh the old copies
        {"name": "ragged124_update", "kind": "ragged", "op": "update", "place": "own", "dtype": "fp32",
         "k": 12, "m": 4, "e": 4, "unit": 64 * KiB, "n": 900, "lo": 4 * KiB, "hi": 64 * MiB, "sizes": 4},
        # tensors that are views of one flat fp32 buffer, at any multiple of 4 bytes
        {"name": "ragged124_views", "kind": "ragged", "op": "encode", "place": "views", "dtype": "fp32",
         "k": 12, "m": 4, "e": 4, "unit": 64 * KiB, "n": 600, "lo": 4 * KiB, "hi": 64 * MiB, "sizes": 5},
        # the largest: one data-parallel rank's whole checkpoint buffer in large units
        {"name": "rank82_20g", "kind": "ragged", "op": "encode", "place": "own", "dtype": "bf16",
         "k": 8, "m": 2, "e": 2, "unit": 4 * MiB, "n": 1, "lo": TOP_BYTES, "hi": TOP_BYTES, "sizes": 6},
        # the whole save of a state: coded, staged to host memory, as k + m slices
        {"name": "save124_1g", "kind": "save", "op": "save", "place": "own", "dtype": "fp32",
         "k": 12, "m": 4, "e": 4, "unit": 64 * KiB, "n": 150, "lo": 4 * KiB, "hi": 64 * MiB, "sizes": 7},
    ]


def _log(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def _code(rng):
    """(k, m): mostly the codes of the unrolled kernels, sometimes wider ones up to 32 + 16."""
    if rng.random() < 0.75:
        return rng.choice([(2, 1), (4, 1), (4, 2), (5, 3), (6, 3), (7, 2), (8, 2), (8, 4), (10, 4), (12, 4), (16, 4)])
    return rng.choice([(20, 4), (24, 4), (10, 6), (6, 8), (16, 6), (16, 8), (24, 8), (20, 12), (32, 16)])


def draw(rng):
    kind = rng.choice(["flat", "flat", "flat", "flat", "ragged", "ragged", "ragged", "ragged", "save", "load"])
    k, m = _code(rng)
    e = rng.randint(1, m)
    if kind == "flat":
        op = rng.choice(["xor", "encode", "encode", "decode", "decode"])
        if op == "xor":
            m = e = 1
        place = rng.choice(["own", "own", "views"])
        n = _log(rng, 4 * KiB, min(256 * MiB, 2 * 1024 * MiB // k))
        if place == "views":
            n = n // 4 * 4
        elif rng.random() < 0.5:
            n = n // 16 * 16
        return {"kind": "flat", "op": op, "call": rng.choice(["eager", "eager", "plan"]) if op == "encode" else "eager",
                "place": place, "k": k, "m": m, "e": e, "nbytes": n}
    unit = rng.choice([4, 16, 64, 64, 256, 1024, 4096]) * KiB
    sizes = rng.randrange(1 << 20)
    if kind == "ragged":
        hi = _log(rng, 32 * KiB, 64 * MiB)
        n = max(1, min(_log(rng, 20, 2000), 4_000_000_000 // max(1, hi // 4)))
        return {"kind": "ragged", "op": rng.choice(["encode", "encode", "decode", "update"]),
                "place": rng.choice(["own", "own", "views"]), "dtype": rng.choice(["fp32", "bf16"]),
                "k": k, "m": m, "e": e, "unit": unit, "n": n, "lo": 512, "hi": hi, "sizes": sizes}
    hi = _log(rng, 256 * KiB, 64 * MiB)
    return {"kind": kind, "op": kind, "place": "own", "dtype": rng.choice(["fp32", "bf16"]), "k": k, "m": m, "e": e,
            "unit": min(unit, 256 * KiB), "n": rng.randint(10, 50), "lo": 512, "hi": hi, "sizes": sizes}


# ------------------------------------------------------------------ inputs --

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1_000_003 + 17)
    return g


def _state_bytes(nbytes, g, dtype="fp32"):
    """``nbytes`` bytes of normal values on the GPU, as uint8 (its storage may be a few bytes longer)."""
    kind, width = (torch.bfloat16, 2) if dtype == "bf16" else (torch.float32, 4)
    x = torch.empty(-(-nbytes // width), dtype=kind, device="cuda")
    x.normal_(0.0, 0.02, generator=g)
    return x.view(torch.uint8)[:nbytes]


def _lost(c):
    """The e lost positions among k + m: always a data position, then any."""
    r = random.Random(c["k"] * 4096 + c["m"] * 64 + c["e"])
    first = r.randrange(c["k"])
    rest = [p for p in range(c["k"] + c["m"]) if p != first]
    return sorted([first] + r.sample(rest, c["e"] - 1))


def _flat_shards(c, seed):
    g, k, n = _generator(seed), c["k"], c["nbytes"]
    if c["place"] == "views":
        flat = torch.empty(k * n // 4, dtype=torch.float32, device="cuda")
        flat.normal_(0.0, 0.02, generator=g)
        return [flat[j * n // 4: (j + 1) * n // 4] for j in range(k)]
    return [_state_bytes(n, g) for _ in range(k)]


def _sizes(c):
    """Tensor byte sizes, log-uniform on [lo, hi], whole elements."""
    r, w = random.Random(c["sizes"]), 2 if c["dtype"] == "bf16" else 4
    return [max(w, (c["hi"] if c["lo"] == c["hi"] else _log(r, c["lo"], c["hi"])) // w * w) for _ in range(c["n"])]


def _tensors(c, seed):
    """(block, tensors): the tensors are views of the uint8 block, at 64-byte starts or back to back."""
    step = 1 if c["place"] == "views" else 64
    starts, at = [], 0
    for s in _sizes(c):
        starts.append(at)
        at += -(-s // step) * step
    block = _state_bytes(at, _generator(seed), c["dtype"])
    kind = torch.bfloat16 if c["dtype"] == "bf16" else torch.float32
    return block, [block[a: a + s].view(kind) for a, s in zip(starts, _sizes(c))]


def _changed(c):
    """Indices of tensors that hold about one byte in a hundred of the state (at least one tensor)."""
    sizes = _sizes(c)
    order, most, got, have = list(range(len(sizes))), sum(sizes) / 100, [], 0
    random.Random(c["sizes"] + 1).shuffle(order)
    for i in order:
        if have + sizes[i] <= most:
            got.append(i)
            have += sizes[i]
    return sorted(got) or [min(order, key=lambda i: sizes[i])]


def prepare(case, seed):
    c, ec = case, _pkg()
    if c["kind"] == "flat":
        return _prepare_flat(c, seed, ec)
    if c["kind"] in ("save", "load"):
        from megatron_lm_amd.checkpoint import GpuSliceCodec
        _, tensors = _tensors(c, seed)
        codec = GpuSliceCodec(c["k"], c["m"], c["unit"])
        state = {"case": c, "codec": codec, "tensors": tensors, "slices": None}
        if c["kind"] == "load":
            meta, slices = codec.encode(tensors)
            lost = set(_lost(c))
            state.update(meta=meta, tensors=None, read={p: s for p, s in enumerate(slices) if p not in lost})
        return state
    block, tensors = _tensors(c, seed)
    lay = ec.StripeLayout(tensors, c["k"], c["m"], c["unit"])
    parity = lay.alloc_parity()
    state = {"case": c, "block": block, "layout": lay, "parity": parity}
    if c["op"] == "encode":
        return state
    lay.encode(parity)
    if c["op"] == "decode":
        lost = _lost(c)
        gone = [lay.unit_view(s * c["k"] + p) for p in lost if p < c["k"]
                for s in range(lay.n_stripes) if s * c["k"] + p < lay.n_units]
        torch._foreach_zero_(gone)
        for p in lost:
            if p >= c["k"]:
                parity[:, p - c["k"]].zero_()
        state["plan"] = lay.plan_decode(parity, lost)
        return state
    new = [tensors[i] for i in _changed(c)]
    old = [t.clone() for t in new]
    g = _generator(seed + 7)
    for t in new:
        t.add_(torch.empty_like(t).normal_(0.0, 0.001, generator=g))
    units, olds = [], []
    first = np.cumsum([0] + [-(-s // c["unit"]) for s in _sizes(c)])
    for i, o in zip(_changed(c), old):
        flat = o.view(torch.uint8)
        for u in range(int(first[i + 1] - first[i])):
            units.append(int(first[i]) + u)
            olds.append(flat[u * c["unit"]: (u + 1) * c["unit"]])
    state.update(plan=lay.plan_update(parity, units, olds), new=new, old=old)
    return state


def _prepare_flat(c, seed, ec):
    shards = _flat_shards(c, seed)
    state = {"case": c, "ec": ec, "shards": shards}
    if c["op"] == "decode":
        coded = ec.rs_encode(shards, c["m"])
        if c["place"] == "views":   # the parity shards, too, lie back to back
            coded = torch.cat(coded).chunk(c["m"])
        word, lost = list(shards) + list(coded), _lost(c)
        state["out"] = None
        if c["place"] == "views":   # rebuilt in place
            state["out"] = [word[p].zero_() for p in lost]
        state["shards"] = [None if p in lost else t for p, t in enumerate(word)]
    elif c["call"] == "plan":
        state["plan"] = ec.ShardPlan(ec.cauchy_matrix(c["k"], c["m"]), shards)
    return state


def run(state):
    c = state["case"]
    if c["kind"] == "flat":
        ec = state["ec"]
        if c["op"] == "xor":
            return ec.xor_encode(state["shards"])
        if c["op"] == "decode":
            got = ec.reconstruct(state["shards"], c["k"], c["m"], out=state["out"])
            return [got[p] for p in sorted(got)]
        return state["plan"]() if "plan" in state else ec.rs_encode(state["shards"], c["m"])
    if c["kind"] == "save":
        if state["slices"] is not None:   # the last save's slices were written out: hand their memory back
            state["codec"].release(state["slices"])
        _, state["slices"] = state["codec"].encode(state["tensors"])
        return state["slices"]
    if c["kind"] == "load":
        return state["codec"].decode(state["meta"], state["read"], torch.device("cuda", 0))
    lay, parity = state["layout"], state["parity"]
    if c["op"] == "encode":
        return lay.encode(parity)
    lay.run(state["plan"])
    if c["op"] == "decode":
        return [state["block"], parity]
    torch._foreach_copy_(state["old"], state["new"])   # the next change is against these bytes
    return [parity] + state["old"][:8]


# ------------------------------------------------------------- work, checks --

def _unit_lengths(c):
    """[stripes, k] valid bytes of each unit."""
    ln = []
    for s in _sizes(c):
        ln += [c["unit"]] * (s // c["unit"]) + ([s % c["unit"]] if s % c["unit"] else [])
    ln += [0] * (-len(ln) % c["k"])
    return np.array(ln, np.int64).reshape(-1, c["k"])


def work(case):
    c = case
    k, m, e = c["k"], c["m"], c["e"]
    if c["kind"] == "flat":
        return {"bytes": (k + (e if c["op"] == "decode" else m)) * c["nbytes"], "flops": 0.0}
    ln = _unit_lengths(c)
    stripes, data = ln.shape[0], int(ln.sum())
    if c["kind"] in ("save", "load"):
        return {"bytes": data + (k + m if c["kind"] == "save" else k) * stripes * c["unit"], "flops": 0.0}
    if c["op"] == "encode":
        return {"bytes": data + m * stripes * c["unit"], "flops": 0.0}
    if c["op"] == "decode":
        lost = _lost(c)
        read = [p for p in range(k + m) if p not in lost][:k]
        part = [int(ln[:, p].sum()) if p < k else stripes * c["unit"] for p in read + lost]
        return {"bytes": sum(part), "flops": 0.0}
    sizes, per = _sizes(c), c["unit"]
    first = np.cumsum([0] + [-(-s // per) for s in sizes])
    hit = np.zeros(ln.size, bool)
    for i in _changed(c):
        hit[first[i]: first[i + 1]] = True
    new = np.where(hit.reshape(ln.shape), ln, 0)
    # new, old and the changed stripes' parity read, the parity and the refreshed old copies written
    return {"bytes": 3 * int(new.sum()) + 2 * m * int(new.max(axis=1).sum()), "flops": 0.0}


def tolerance(case):
    return "exact"   # bytes


def _tables():
    """256 x 256 products over GF(2^8) mod x^8+x^4+x^3+x^2+1, on the GPU."""
    exp, log, x = np.zeros(510, np.uint8), np.zeros(256, np.int64), 1
    for i in range(255):
        exp[i] = exp[i + 255] = x
        log[x] = i
        x = (x << 1) ^ (0x11D if x & 0x80 else 0)
    a = np.arange(1, 256)
    mul = np.zeros((256, 256), np.uint8)
    mul[1:, 1:] = exp[log[a][:, None] + log[a][None, :]]
    inv = np.zeros(256, np.int64)
    inv[1:] = exp[(255 - log[a]) % 255]
    return torch.from_numpy(mul).cuda(), inv


def _parity(rows, m):
    """The m Cauchy parity rows of k uint8 tensors of one length, by table lookup."""
    mul, inv = _tables()
    k, n = len(rows), rows[0].numel()
    out = [torch.zeros(n, dtype=torch.uint8, device="cuda") for _ in range(m)]
    for a in range(0, n, 32 * MiB):
        b = min(n, a + 32 * MiB)
        for j, r in enumerate(rows):
            at = r[a:b].to(torch.int64)
            for i in range(m):
                out[i][a:b] ^= mul[int(inv[(k + i) ^ j])][at]
    return out


def exact(case, seed):
    c = case
    if c["kind"] == "flat":
        if (c["k"] + c["m"]) * c["nbytes"] > 4096 * MiB:
            return None
        shards = _flat_shards(c, seed)
        rows = [t.view(torch.uint8) for t in shards]
        if c["op"] == "xor":
            total = rows[0].clone()
            for r in rows[1:]:
                total ^= r
            return total
        parity = _parity(rows, c["m"])
        if c["op"] == "encode":
            return parity
        return [((shards if c["place"] == "views" else rows) + parity)[p] for p in _lost(c)]
    if sum(_sizes(c)) > 1024 * MiB or c["op"] == "update":
        return None
    block, tensors = _tensors(c, seed)
    if c["kind"] == "load":
        return tensors
    k, m, unit = c["k"], c["m"], c["unit"]
    units = []
    for t in tensors:
        flat = t.view(torch.uint8)
        units.append(torch.nn.functional.pad(flat, (0, -flat.numel() % unit)).view(-1, unit))
    units = torch.cat(units)
    units = torch.nn.functional.pad(units, (0, 0, 0, -units.shape[0] % k)).view(-1, k, unit)
    rows = [units[:, j].reshape(-1) for j in range(k)]
    parity = _parity(rows, m)
    if c["kind"] == "save":
        return [r.cpu().numpy() for r in rows + parity]
    stacked = torch.stack([p.view(-1, unit) for p in parity], dim=1)
    return stacked if c["op"] == "encode" else [block, stacked]
