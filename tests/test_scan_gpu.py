"""The fused scan (csrc/gdn_scan.hip), which the built-in prefill takes for
most batches: lengths at the edges of its tiles, segments and launches, head
layouts, states, extreme inputs, and batches it must cut or leave whole, against
the CPU oracle at the operator tolerance; that these batches take it, from the
host's plan (tests/test_host_sanitize.py) and from what the device left in the
workspace; and the matrix-instruction chains of its object file on the CPU.
"""

import os

import numpy as np
import pytest
import torch

from conftest import assert_output_close, assert_output_close_to_row_max, assert_state_close
from oracle import gdn_oracle as O
from test_mfma_chains import BUILD, _disassemble, _functions, _need_tools, _violations

from gdn_amd import prefill  # noqa: E402

# lens -> what the batch exercises.  One sequence of 97..704 tokens (at most
# 11 chunks) and of 2049 on runs the scan at 8 v-heads, the latter cut into
# segments of at least 4 chunks; the batches with "cut" or "long" in their name
# are cut.
BATCHES = {
    "one_partial": [97],
    "one_full": [128],
    "one_odd_chunks": [641],
    "one_11_chunks": [704],
    "cut_33_chunks": [2049],            # the last segment holds one token
    "cut_exact": [2560],                # 40 chunks: eight segments of 5
    "cut_many": [8191],
    "two_cut": [4100, 2111],
    "three_cut": [1280] * 3,            # a workgroup a compute unit: segments of 7
    "four_cut_long": [8191] * 4,        # two workgroups a compute unit
    "four_cut": [4096, 4033, 64, 2950],
    "ragged_cut": [6, 49, 294, 1800, 2040, 61],
    "long_among_ones": [3000] + [1] * 63,   # 64 sequences, the most that are cut
    "65_sequences": [100] * 64 + [1500],    # more than the segment lookup takes
    "empty_between": [0, 640, 0, 0, 65, 700, 0],
    "index_kernel": [200, 0, 63] * 90,      # more than 256 sequences
}


def is_cut(name):
    return "cut" in name or "long" in name


def _words(ws, T, N):
    """(chunks, path flag, segment length) that a batch left in its workspace,
    after the offsets of its sequences (one sequence: the length alone)."""
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
    T, N = sum(lens), len(lens)
    ws = prefill.alloc_workspace(T, N, cuda_device)
    ws.fill_(0xFF)  # nothing in it needs to hold anything
    o, s = _run(inp, cuda_device, workspace=ws)
    assert_output_close(o, o_ref)
    assert_state_close(s, s_ref)
    _, sequential, length = _words(ws, T, N)
    if N > 1:
        assert sequential == 0
    if is_cut(name):
        assert 4 <= length < max(lens) // 64, length
    # a second pass gives the same bits
    o2, s2 = _run(inp, cuda_device)
    assert np.array_equal(o, o2) and np.array_equal(s, s2)


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


# The stress inputs of the operand forms' tests (tests/test_prefill_gpu.py) through
# the scan: whole, cut, and cut beside a short sequence.
STRESS = [[200, 64, 130], [2600], [2600, 700], [1300, 1290, 40]]


@pytest.mark.gpu
@pytest.mark.parametrize("lens", STRESS, ids=lambda x: "_".join(map(str, x)))
def test_scan_extreme_gates(cuda_device, lens):
    # Per-head gates around softplus' threshold (x > 20), beta saturated at 0
    # and 1, decays ~1 (segment maps near the identity) and so fast that exp(G)
    # underflows inside a chunk.
    print(f"scan extreme gates lens={lens}", flush=True)
    T = sum(lens)
    inp = O.make_prefill_inputs(lens, seed=361)
    rng = np.random.default_rng(361)
    a_h = np.array([30.0, -30.0, 20.0, 0.0, 19.5, -5.0, 5.0, 1.0], np.float32)
    b_h = np.array([-40.0, 40.0, 0.0, 8.0, -8.0, 1.0, -1.0, 0.0], np.float32)
    inp["a"][:] = O.bf16_round(a_h[None, :] + rng.normal(0, 0.5, (T, 8)).astype(np.float32))
    inp["b"][:] = O.bf16_round(b_h[None, :] + rng.normal(0, 0.5, (T, 8)).astype(np.float32))
    inp["A_log"][:] = np.array([-10.0, 2.7, 0.0, -20.0, 1.0, 0.5, 0.1, 2.0], np.float32)
    o_ref, s_ref = O.prefill_seq_c(**inp)
    o, s = _run(inp, cuda_device)
    assert_output_close(o, o_ref)
    assert_state_close(s, s_ref)


@pytest.mark.gpu
@pytest.mark.parametrize("lens", STRESS, ids=lambda x: "_".join(map(str, x)))
def test_scan_operand_magnitudes(cuda_device, lens):
    # Keys and values far from unit size, per head (q/k head 0 keys x 1e-3, head 1
    # x 0.05; v-heads 0-1 values x 1e4, 2-3 x 1e-4), each head against its own
    # magnitude.
    print(f"scan operand magnitudes lens={lens}", flush=True)
    inp = O.make_prefill_inputs(lens, seed=362, slow_decay_heads=(7,))
    inp["k"] = O.bf16_round(inp["k"] * np.array([1e-3, 0.05, 1.0, 1.0], np.float32)[None, :, None])
    vs = np.array([1e4, 1e4, 1e-4, 1e-4, 1.0, 1.0, 1.0, 1.0], np.float32)
    inp["v"] = O.bf16_round(inp["v"] * vs[None, :, None])
    inp["state"] = (inp["state"] * vs[None, :, None, None]).astype(np.float32)
    o_ref, s_ref = O.prefill_seq_c(**inp)
    o, s = _run(inp, cuda_device)
    for h in range(8):
        m = max(float(np.abs(o_ref[:, h]).max()), 1e-30)
        assert_output_close(o[:, h] / m, o_ref[:, h] / m, what=f"output head {h}")
        assert_state_close(s[:, h], s_ref[:, h], what=f"state head {h}")


@pytest.mark.gpu
@pytest.mark.parametrize("noise", [0.0, 0.1])
def test_scan_all_same(cuda_device, noise):
    # The reference's adversarial family: equal keys, the state growing to ~1e27
    # within two chunks.  Single bf16 operands of the output products: the row
    # bound of conftest.py where the growth is uneven.
    lens = [100] if noise == 0.0 else [70, 48, 64]
    print(f"scan all_same lens={lens} noise={noise}", flush=True)
    inp = O.make_all_same_inputs(lens, noise=noise, seed=3)
    o_ref, s_ref = O.prefill_seq_c(**inp)
    o, s = _run(inp, cuda_device)
    if noise == 0.0:
        assert_output_close(o, o_ref)
    else:
        assert_output_close_to_row_max(o, o_ref)
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
