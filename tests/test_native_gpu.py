"""The native entry of ordinary calls (csrc/gdn_torch.cpp): the same bits as
the Python path, which takes every other call, errors included."""

import sys

import numpy as np
import pytest
import torch

from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu

from gdn_amd import _lib, decode, prefill  # noqa: E402


def _dev(inp, dev):
    d = {n: torch.from_numpy(np.ascontiguousarray(inp[n])).to(dev) for n in inp
         if isinstance(inp[n], np.ndarray)}
    return {n: t.to(torch.bfloat16) if n in ("q", "k", "v", "a", "b") else t for n, t in d.items()}


def _decode(d, scale, B, T, hv=8):
    dev = d["q"].device
    o = torch.empty((B, T, hv, 128), dtype=torch.bfloat16, device=dev)
    s = torch.empty((B, hv, 128, 128), device=dev)
    decode.kernel(d["q"], d["k"], d["v"], d.get("state"), d["A_log"], d["a"], d["dt_bias"], d["b"],
                  scale, o, s)
    return o, s


def _prefill(d, scale, workspace=None, hv=8):
    dev, T, N = d["q"].device, d["q"].shape[0], d["cu_seqlens"].numel() - 1
    o = torch.empty((T, hv, 128), dtype=torch.bfloat16, device=dev)
    s = torch.empty((N, hv, 128, 128), device=dev)
    prefill.kernel(d["q"], d["k"], d["v"], d.get("state"), d["A_log"], d["a"], d["dt_bias"], d["b"],
                   d["cu_seqlens"], scale, o, s, workspace=workspace)
    return o, s


def _both(monkeypatch, call):
    taken = call()
    monkeypatch.setattr(_lib, "native", lambda: None)
    python = call()
    monkeypatch.undo()
    return taken, python


@pytest.mark.parametrize("heads, B, T", [((4, 8), 3, 1), ((4, 8), 2, 5), ((2, 4), 3, 1)])
@pytest.mark.parametrize("with_state", [True, False])
def test_decode_same_bits(cuda_device, monkeypatch, heads, B, T, with_state):
    inp = O.make_prefill_inputs([T] * B, seed=5, heads=heads, with_state=with_state)
    d = _dev(inp, cuda_device)
    for n, h in (("q", heads[0]), ("k", heads[0]), ("v", heads[1])):
        d[n] = d[n].reshape(B, T, h, 128)
    for n in ("a", "b"):
        d[n] = d[n].reshape(B, T, heads[1])
    assert _lib.native() is not None
    for scale in (0.25, None, 0.0):
        x, y = _both(monkeypatch, lambda: _decode(d, scale, B, T, heads[1]))
        assert torch.equal(x[0], y[0]) and torch.equal(x[1], y[1])


@pytest.mark.parametrize("lens, heads, own", [([60], (4, 8), True), ([200, 0, 33], (4, 8), False),
                                              ([130], (2, 4), False)])
def test_prefill_same_bits(cuda_device, monkeypatch, lens, heads, own):
    d = _dev(O.make_prefill_inputs(lens, seed=6, heads=heads), cuda_device)
    ws = prefill.alloc_workspace(sum(lens), len(lens), cuda_device, heads) if own else None
    for cu in (torch.int32, torch.int64):
        d["cu_seqlens"] = d["cu_seqlens"].to(cu)
        x, y = _both(monkeypatch, lambda: _prefill(d, None, ws, heads[1]))
        assert torch.equal(x[0], y[0]) and torch.equal(x[1], y[1])


def test_other_calls_take_the_python_path(cuda_device):
    # strided inputs, a tensor scale, an empty batch: as they are there;
    # what it refuses stays refused, with its messages
    inp = O.make_prefill_inputs([1] * 4, seed=7)
    d = _dev(inp, cuda_device)
    for n in ("q", "k", "v"):
        d[n] = d[n][:, None]
    for n in ("a", "b"):
        d[n] = d[n][:, None]
    ref = _decode(d, 0.5, 4, 1)
    wide = dict(d, q=torch.cat([d["q"], d["q"]], -1)[..., :128])
    got = _decode(wide, torch.tensor(0.5), 4, 1)
    assert torch.equal(ref[0], got[0]) and torch.equal(ref[1], got[1])
    none = {n: t if n in ("A_log", "dt_bias") else t[:0] for n, t in d.items()}
    with pytest.raises(ValueError, match="null pointer"):  # empty tensors have no address
        _decode(none, 0.5, 0, 1)
    for bad, what in ((dict(d, q=d["q"].float()), "q must be"), (dict(d, k=d["k"][:3]), "k must have"),
                      (dict(d, v=d["v"].cpu()), "v is on")):
        with pytest.raises(ValueError, match=what):
            _decode(bad, 0.5, 4, 1)
    with pytest.raises(ValueError, match="scale"):
        _decode(d, -1.0, 4, 1)
    p = _dev(O.make_prefill_inputs([100], seed=8), cuda_device)
    with pytest.raises(_lib.GdnWorkspaceError):
        _prefill(p, None, torch.empty(256, dtype=torch.uint8, device=cuda_device))
    with pytest.raises(ValueError, match="overlaps"):
        decode.kernel(d["q"], d["k"], d["v"], d["state"], d["A_log"], d["a"], d["dt_bias"], d["b"], 0.5,
                      d["v"], torch.empty_like(d["state"]))


def test_cached_workspace_is_given_back(cuda_device):
    # a workspace without an address of its own (vmapped): the call is left to
    # the Python path, and the tensor is not held
    d = _dev(O.make_prefill_inputs([100], seed=9), cuda_device)
    o = torch.empty((100, 8, 128), dtype=torch.bfloat16, device=cuda_device)
    s = torch.empty((1, 8, 128, 128), device=cuda_device)

    def call(w):
        held = sys.getrefcount(w)
        rc = _lib.native().prefill(d["q"], d["k"], d["v"], d["state"], d["A_log"], d["a"], d["dt_bias"],
                                   d["b"], d["cu_seqlens"], None, o, s, None, lambda *_: w)
        assert rc == 1
        assert sys.getrefcount(w) == held
        return w

    torch.vmap(call)(torch.empty((2, prefill.workspace_bytes(100, 1)), dtype=torch.uint8, device=cuda_device))
