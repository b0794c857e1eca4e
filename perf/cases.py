"""Performance cases of the Gated DeltaNet operators.

Each case is one pass through the public entry points ``gdn_amd.decode.kernel``
and ``gdn_amd.prefill.kernel``, called as a serving program calls them:
destination-passing, on torch's current stream, without a host synchronisation.
The distributions are those of the repository's own benchmark inputs: q and k
N(0,1) L2-normalised per head, v and the raw gates a, b N(0,1), A_log
U(0, ln 16), dt_bias U(0, 1), recurrent states N(0, 0.05).

A case's plain values:

* ``op``      "decode" or "prefill"
* ``hqk``, ``hv``  q/k heads and v-heads (head size is always 128)
* decode:  ``batch`` rows of ``tokens`` tokens each (1: a plain step; more:
  multi-token / speculative decode), through ``layers`` layers with tensors of
  their own; ``graph``: the step is captured once as a HIP graph and replayed,
  as a serving loop does
* prefill: ``lens`` comma-separated sequence lengths of the packed batch;
  ``state``: the sequences continue from states (chunked or resumed prefill)
  instead of starting fresh; ``cu`` the offsets' integer type; ``workspace``:
  the caller owns the workspace instead of using the per-stream cache;
  ``slow``: the first heads whose decay is near one (long memory)
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "gated-delta-network_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from gdn_amd import decode, prefill  # noqa: E402

D = 128  # head size


def _decode(name, batch, tokens=1, hqk=4, hv=8, layers=1, graph=False):
    c = {"op": "decode", "batch": batch, "tokens": tokens, "hqk": hqk, "hv": hv,
         "layers": layers, "graph": graph}
    return dict(c, name=name) if name else c


def _prefill(name, lens, hqk=4, hv=8, state=False, cu="int32", workspace=False, slow=0):
    c = {"op": "prefill", "lens": ",".join(str(n) for n in lens), "hqk": hqk, "hv": hv,
         "state": state, "cu": cu, "workspace": workspace, "slow": slow}
    return dict(c, name=name) if name else c


# 64 prompts of a busy server's queue, packed: ragged, 9 to 607 tokens.
_SHORT = (37, 182, 64, 401, 23, 96, 255, 130, 18, 311, 77, 149, 45, 512, 88, 203,
          29, 117, 366, 61, 154, 9, 240, 83, 128, 19, 475, 102, 58, 271, 35, 190,
          66, 333, 14, 144, 91, 52, 220, 607, 40, 73, 161, 111, 26, 288, 134, 57,
          197, 31, 420, 69, 121, 16, 248, 94, 173, 48, 355, 80, 139, 22, 209, 63)


def listed():
    return [
        # One user's step: the smallest call, latency and host path.
        _decode("decode_b1", 1),
        # A small batch's step through a stack of layers, replayed as a graph
        # (the launch-bound serving loop).
        _decode("decode_b8_graph12", 8, layers=12, graph=True),
        # The reference's headline step.
        _decode("decode_b64", 64),
        # The largest published batch: 1 GiB of state traffic.
        _decode("decode_b512", 512),
        # Speculative decode: four draft tokens per row.
        _decode("decode_b64_t4", 64, tokens=4),
        # The unsharded head layout (16 q/k, 32 v heads), a ragged batch size.
        _decode("decode_b13_h32", 13, hqk=16, hv=32),
        # A short prompt: the smallest prefill, one partial chunk.
        _prefill("prefill_1x61", (61,)),
        # A packed batch of many short prompts with resumed states.
        _prefill("prefill_64_short", _SHORT, state=True),
        # An ordinary prompt, fresh state, caller-owned workspace.
        _prefill("prefill_1x1024", (1024,), workspace=True),
        # The mixed-length batch of the reference's workloads, resumed states.
        _prefill("prefill_varlen6", (6, 49, 294, 1800, 2040, 61), state=True, cu="int64"),
        # One long prompt.
        _prefill("prefill_1x8192", (8192,), workspace=True),
        # Long-context batch with long-memory heads: the largest prefill.
        _prefill("prefill_4x8192", (8192,) * 4, state=True, workspace=True, slow=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "step", "multi", "single", "single", "packed", "packed"))
    hqk, hv = rng.choice(((4, 8), (4, 8), (4, 8), (16, 32), (2, 8), (8, 8)))
    if kind == "step":
        batch = max(1, _log_int(rng, 1, 512) * 8 // max(hv, 8))
        graph = batch * hv <= 512 and rng.random() < 0.3
        return _decode(None, batch, hqk=hqk, hv=hv, layers=rng.randint(4, 12) if graph else 1,
                       graph=graph)
    if kind == "multi":
        return _decode(None, max(1, _log_int(rng, 1, 128) * 8 // max(hv, 8)),
                       tokens=rng.randint(2, 16), hqk=hqk, hv=hv)
    opts = {"hqk": hqk, "hv": hv, "state": rng.random() < 0.5,
            "cu": rng.choice(("int32", "int64")), "workspace": rng.random() < 0.5,
            "slow": rng.choice((0, 0, 2))}
    if kind == "single":
        return _prefill(None, (_log_int(rng, 1, 8192 * 8 // max(hv, 8)),), **opts)
    n = _log_int(rng, 2, 64)
    mean = _log_int(rng, 8, 12288 * 8 // max(hv, 8) / n)
    spread = rng.choice((1.2, 3.0, 8.0))  # nearly equal lengths .. one long among short ones
    lens = [mean * math.exp(rng.uniform(-1.0, 1.0) * math.log(spread)) for _ in range(n)]
    fit = min(1.0, 12288 * 8 / max(hv, 8) / sum(lens))
    return _prefill(None, [max(1, int(round(x * fit))) for x in lens], **opts)


def _lens(case):
    return [int(n) for n in case["lens"].split(",")]


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _unit(gen, dev, *shape):
    x = torch.randn(shape, generator=gen, device=dev)
    return (x / x.norm(dim=-1, keepdim=True)).to(torch.bfloat16)


def _inputs(case, seed):
    """The input tensors of each layer's call, made from the seed alone."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(seed)
    hqk, hv = case["hqk"], case["hv"]

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=dev)

    def uniform(*shape):
        return torch.rand(shape, generator=gen, device=dev)

    layers = []
    for _ in range(case.get("layers", 1)):
        if case["op"] == "decode":
            lead, n, with_state = (case["batch"], case["tokens"]), case["batch"], True
        else:
            lens = _lens(case)
            lead, n, with_state = (sum(lens),), len(lens), case["state"]
        x = {"q": _unit(gen, dev, *lead, hqk, D), "k": _unit(gen, dev, *lead, hqk, D),
             "v": normal(*lead, hv, D).to(torch.bfloat16),
             "state": normal(n, hv, D, D) * 0.05 if with_state else None,
             "A_log": uniform(hv) * math.log(16.0),
             "a": normal(*lead, hv).to(torch.bfloat16), "dt_bias": uniform(hv),
             "b": normal(*lead, hv).to(torch.bfloat16)}
        slow = case.get("slow", 0)
        if slow:
            x["A_log"][:slow] = -6.0 - uniform(slow)
        layers.append(x)
    return layers


def _call_decode(layer):
    decode.kernel(layer["q"], layer["k"], layer["v"], layer["state"], layer["A_log"], layer["a"],
                  layer["dt_bias"], layer["b"], layer["scale"], layer["output"],
                  layer["new_state"])


def prepare(case, seed):
    layers = _inputs(case, seed)
    hv = case["hv"]
    for x in layers:
        x["scale"] = 1.0 / math.sqrt(D)
        x["output"] = torch.empty_like(x["v"])
        n = case["batch"] if case["op"] == "decode" else len(_lens(case))
        x["new_state"] = torch.empty((n, hv, D, D), dtype=torch.float32, device=x["q"].device)
    st = {"op": case["op"], "layers": layers, "graph": None}
    if case["op"] == "prefill":
        lens, dev = _lens(case), layers[0]["q"].device
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        st["cu"] = torch.tensor(cu, dtype=getattr(torch, case["cu"]), device=dev)
        st["workspace"] = (prefill.alloc_workspace(cu[-1], len(lens), dev, (case["hqk"], hv))
                           if case["workspace"] else None)
    elif case["graph"]:
        for x in layers:
            _call_decode(x)  # everything is loaded before the capture
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            for x in layers:
                _call_decode(x)
    return st


def run(st):
    if st["graph"] is not None:
        st["graph"].replay()
    elif st["op"] == "decode":
        for x in st["layers"]:
            _call_decode(x)
    else:
        x = st["layers"][0]
        prefill.kernel(x["q"], x["k"], x["v"], x["state"], x["A_log"], x["a"], x["dt_bias"],
                       x["b"], st["cu"], x["scale"], x["output"], x["new_state"],
                       workspace=st["workspace"])
    return [(x["output"], x["new_state"]) for x in st["layers"]]


def work(case):
    """Each input read once, each output written once; the operations of the
    recurrence itself (S k, the decay, the rank-one update and S q: 7 per state
    element and token)."""
    hqk, hv = case["hqk"], case["hv"]
    if case["op"] == "decode":
        tokens, n, reads = case["batch"] * case["tokens"], case["batch"], 1
    else:
        lens = _lens(case)
        tokens, n, reads = sum(lens), len(lens), int(case["state"])
    per_token = 2 * (2 * hqk * D + 2 * hv * D + 2 * hv)
    state = n * hv * D * D * 4
    layers = case.get("layers", 1)
    return {"bytes": layers * (tokens * per_token + (1 + reads) * state + 8 * hv),
            "flops": layers * tokens * hv * 7 * D * D}


def tolerance(case):
    """Against the float64 recurrence the bf16 outputs measure 1.7e-3 (decode:
    their own rounding) and 2.9e-3 (prefill: bf16 operands of the output
    products as well), the f32 states at most 2e-5; four times that.  One
    value may flip by a bf16 unit (2^-7 of it) in each."""
    if case["op"] == "decode":
        return {"rel": 7e-3, "max": 3e-2}
    return {"rel": 1.2e-2, "max": 5e-2}


def exact(case, seed):
    """The recurrence token by token in float64, over all sequences at once."""
    out = []
    for x in _inputs(case, seed):
        hv, ratio = case["hv"], case["hv"] // case["hqk"]
        f64 = {n: None if t is None else t.double() for n, t in x.items()}
        if case["op"] == "decode":
            lens = [case["tokens"]] * case["batch"]
        else:
            lens = _lens(case)
        dev = x["q"].device
        length = torch.tensor(lens, device=dev)
        first = torch.cumsum(length, 0) - length
        flat = {n: f64[n].reshape(-1, *f64[n].shape[-2:]) for n in ("q", "k", "v")}
        a, b = f64["a"].reshape(-1, hv), f64["b"].reshape(-1, hv)
        g = torch.exp(-torch.exp(f64["A_log"]) * torch.nn.functional.softplus(a + f64["dt_bias"]))
        beta = torch.sigmoid(b)
        S = (torch.zeros((len(lens), hv, D, D), dtype=torch.float64, device=dev)
             if f64["state"] is None else f64["state"].clone())
        o = torch.zeros_like(flat["v"])
        for t in range(max(lens)):
            live = torch.nonzero(length > t).flatten() if t >= min(lens) else None
            at = (first if live is None else first[live]) + t
            cur = S if live is None else S[live]
            kt = flat["k"][at].repeat_interleave(ratio, 1)
            qt = flat["q"][at].repeat_interleave(ratio, 1)
            cur = cur * g[at][..., None, None]
            pred = torch.matmul(cur, kt[..., None])[..., 0]
            v_new = beta[at][..., None] * (flat["v"][at] - pred)
            cur = cur + v_new[..., None] * kt[..., None, :]
            o[at] = torch.matmul(cur, qt[..., None])[..., 0] / math.sqrt(D)
            if live is None:
                S = cur
            else:
                S[live] = cur
        out.append((o.reshape(x["v"].shape), S))
    return out
