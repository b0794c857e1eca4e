"""The fused scan (csrc/gdn_scan.hip), which the built-in prefill takes for
most batches: lengths at the edges of its tiles, segments and launches, head
layouts, states, and batches it must split or leave whole, against the CPU
oracle at the operator tolerance; and the matrix-instruction chains of its
object file on the CPU.
"""

import os

import numpy as np
import pytest
import torch

from conftest import assert_output_close, assert_state_close
from oracle import gdn_oracle as O
from test_mfma_chains import BUILD, _disassemble, _functions, _need_tools, _violations

from gdn_amd import prefill  # noqa: E402

# lens -> what the batch exercises.  One sequence of 97..704 tokens (at most
# 11 chunks) and of 2049 on runs the scan at 8 v-heads; from about 24 chunks a
# lone sequence is cut into segments of at least 4 chunks.
BATCHES = {
    "one_partial": [97],
    "one_full": [128],
    "one_odd_chunks": [641],
    "one_11_chunks": [704],
    "cut_33_chunks": [2049],            # the last segment holds one token
    "cut_exact": [2560],                # 40 chunks: eight segments of 5
    "cut_many": [8191],
    "two_cut": [4100, 2111],
    "four_cut": [4096, 4033, 64, 2950],
    "ragged_cut": [6, 49, 294, 1800, 2040, 61],
    "long_among_ones": [3000] + [1] * 63,   # 64 sequences, the most that are cut
    "65_sequences": [100] * 64 + [1500],    # more than the segment lookup takes
    "empty_between": [0, 640, 0, 0, 65, 700, 0],
    "index_kernel": [200, 0, 63] * 90,      # more than 256 sequences
}


def _words(ws, T, N):
    """(chunks, path flag, segment length or operand form) that a batch of N > 1
    sequences left in its workspace, after the offsets of its sequences."""
    at = (O.max_chunks(T, N) * 16 + 255) // 256 * 256 + N * 4
    return ws[at:at + 12].cpu().numpy().view(np.int32).tolist()


def _run(inp, dev, heads=(4, 8), in_place=False, workspace=None):
    d = {n: torch.from_numpy(np.ascontiguousarray(inp[n])).to(dev).to(torch.bfloat16)
         for n in ("q", "k", "v", "a", "b")}
    for n in ("A_log", "dt_bias", "cu_seqlens"):
        d[n] = torch.from_numpy(inp[n]).to(dev)
    d["state"] = None if inp["state"] is None else torch.from_numpy(inp["state"]).to(dev)
    T, N = d["q"].shape[0], d["cu_seqlens"].numel() - 1
    out = torch.full((T, heads[1], 128), 7.0, dtype=torch.bfloat16, device=dev)
    ns = d["state"] if in_place else torch.full((N, heads[1], 128, 128), 7.0, device=dev)
    prefill.kernel(d["q"], d["k"], d["v"], d["state"], d["A_log"], d["a"], d["dt_bias"], d["b"],
                   d["cu_seqlens"], inp["scale"], out, ns, workspace=workspace)
    torch.cuda.synchronize()
    return out.float().cpu().numpy(), ns.cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(BATCHES))
def test_scan_matches_oracle(cuda_device, name):
    lens = BATCHES[name]
    print(f"scan {name}: {len(lens)} sequences, {sum(lens)} tokens", flush=True)
    inp = O.make_prefill_inputs(lens, seed=300 + len(name), with_state=len(name) % 2 == 0,
                                slow_decay_heads=(0, 7) if "cut" in name else ())
    o_ref, s_ref = O.prefill_seq_c(**inp)
    o, s = _run(inp, cuda_device)
    assert_output_close(o, o_ref)
    assert_state_close(s, s_ref)


@pytest.mark.gpu
@pytest.mark.parametrize("heads, lens", [((1, 1), [5200]), ((2, 8), [700, 33]), ((8, 8), [2500]),
                                         ((16, 32), [130, 2100]), ((3, 6), [2700, 10])])
def test_scan_heads_in_place(cuda_device, heads, lens):
    print(f"scan heads={heads} lens={lens}", flush=True)
    inp = O.make_prefill_inputs(lens, seed=331, heads=heads)
    o_ref, s_ref = O.prefill_seq_c(**inp)
    o, s = _run(inp, cuda_device, heads, in_place=True)
    assert_output_close(o, o_ref)
    assert_state_close(s, s_ref)


@pytest.mark.gpu
@pytest.mark.parametrize("T, cu", [(3200, [64, 3001]), (4500, [0, 100, 4100, 4100])])
def test_scan_cut_partial_batch(cuda_device, T, cu):
    # a cut sequence in a buffer that the batch does not span: the rows outside
    # are zeros (the idle map workgroups take no share of them)
    print(f"scan partial T={T} cu={cu}", flush=True)
    inp = O.make_prefill_inputs([T], seed=341, with_state=False)
    inp["cu_seqlens"] = np.asarray(cu, dtype=np.int64)
    o_ref, s_ref = O.prefill_seq_c(**inp)
    o, s = _run(inp, cuda_device)
    assert not o[:cu[0]].any() and not o[cu[-1]:].any()
    assert_output_close(o, o_ref)
    assert_state_close(s, s_ref)


# Batches whose path the device picks (the chunks, here) in more units than the
# capped grid has workgroups: (lengths, heads, tokens beyond the sequences).
LOOPED = {
    "300": ([200, 0, 500, 37, 1, 129] * 50, (4, 8), 0),
    "2100": ([3, 40, 0, 17, 130] * 420, (1, 1), 77),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(LOOPED))
def test_scan_looped_grid(cuda_device, name):
    lens, heads, extra = LOOPED[name]
    T, N = sum(lens) + extra, len(lens)
    print(f"scan looped N={N} T={T} heads={heads}", flush=True)
    inp = O.make_prefill_inputs(lens[:-1] + [lens[-1] + extra], seed=351, heads=heads)
    inp["cu_seqlens"][-1] -= extra  # the last rows belong to no sequence: zeros
    o_ref, s_ref = O.prefill_seq_c(**inp)
    ws = prefill.alloc_workspace(T, N, cuda_device, heads)
    o, s = _run(inp, cuda_device, heads, workspace=ws)
    assert _words(ws, T, N)[1] == 0  # the chunks, not the sequential kernel
    assert not o[T - extra:].any()
    assert_output_close(o, o_ref)
    assert_state_close(s, s_ref)


def test_scan_object_keeps_one_mfma_shape_per_chain(tmp_path):
    _need_tools()
    path = os.path.join(BUILD, "gdn_scan.o")
    if not os.path.exists(path):
        pytest.skip("gdn_scan.o is not built (run __graft_entry__.build() first)")
    funcs = _functions(_disassemble(path, str(tmp_path)))
    assert sum(mn.startswith("v_mfma") for _, body in funcs for mn, _ in body) > 0
    assert not _violations(funcs)
