"""GPU parity of the tree gated-delta-rule scan in the reference's own
semantics (tt_gdn_problem.reference_truncated = 1: each whole node one chunk,
within-node correction I + R + R^2 from the uncorrected rows,
tree_dfs_ssm.py:100-150) against the float64 oracles of that mode, through
the C ABI: ``oracle.gdn.gdn_tree(mode="reference")`` (the literal row-by-row
restatement) for the forward, autograd through
``oracle.gdn.gdn_tree_reference_torch`` for the backward.

Bars: float32 outputs, node states and gradients (dq, dk, dv, dg, dbeta)
max_rel < 1e-5; bf16 < 2e-2 (max |error| over max |reference|). Nodes of 1 to
512 tokens (1 to 16 correction blocks, ragged last blocks), the c1 forest at
the Qwen3.5 head layout (16 q/k heads, 32 v heads), and the full 16K agent
tree (2 v heads against the oracle; 32 v heads through the per-path property).
"""
import numpy as np
import pytest
import torch

from oracle import gdn as ogdn
from tree_training_amd.gdn import GdnTree, gdn_tree_backward, gdn_tree_forward
from tree_training_amd.workloads import agent_tree, random_forest

pytestmark = pytest.mark.gpu
D = 128
BWD_NAMES = ("dq", "dk", "dv", "dg", "dbeta")


def _inputs(T, Hk, Hv, seed, realistic_gates=False):
    rng = np.random.default_rng(seed)
    q = rng.standard_normal((T, Hk, D)).astype(np.float32)
    k = rng.standard_normal((T, Hk, D)).astype(np.float32)
    v = rng.standard_normal((T, Hv, D)).astype(np.float32)
    if realistic_gates:
        a, b = rng.standard_normal((T, Hv)), rng.standard_normal((T, Hv))
        g, beta = ogdn.gdn_gates(a, b, np.log(rng.uniform(1e-3, 16, Hv)), np.ones(Hv))
    else:
        g = -np.abs(rng.standard_normal((T, Hv))) * 0.05
        beta = 1.0 / (1.0 + np.exp(-rng.standard_normal((T, Hv))))
    return q, k, v, g.astype(np.float32), beta.astype(np.float32)


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


def _t(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to(torch.device("cuda", 0))


def _run(q, k, v, g, beta, lens, par, dtype):
    tree = GdnTree(lens, par, torch.device("cuda", 0))
    o, st = gdn_tree_forward(_t(q).to(dtype), _t(k).to(dtype), _t(v).to(dtype), _t(g), _t(beta), tree,
                             reference_truncated=True)
    torch.cuda.synchronize()
    return o.float().cpu().numpy(), st.cpu().numpy()


def _run_bwd(q, k, v, g, beta, d_o, lens, par, dtype, saved=None):
    tree = GdnTree(lens, par, torch.device("cuda", 0))
    outs = gdn_tree_backward(_t(q).to(dtype), _t(k).to(dtype), _t(v).to(dtype), _t(g), _t(beta),
                             _t(d_o).to(dtype), tree, saved=saved, reference_truncated=True)
    torch.cuda.synchronize()
    return [x.float().cpu().numpy() for x in outs]


def _oracle_grads(q, k, v, g, beta, d_o, lens, par):
    tt = [torch.from_numpy(np.asarray(x, np.float64)).requires_grad_(True) for x in (q, k, v, g, beta)]
    o = ogdn.gdn_tree_reference_torch(*tt, lens, par)
    return [x.numpy() for x in torch.autograd.grad((o * torch.from_numpy(np.asarray(d_o, np.float64))).sum(), tt)]


CASES = {
    "forest_small_nodes": dict(topo=lambda: random_forest(3, node_len=(1, 12)), Hk=2, Hv=4),
    "forest_multi_block": dict(topo=lambda: random_forest(8, node_len=(20, 90)), Hk=2, Hv=2),
    "chain_ragged": dict(topo=lambda: ([33, 64, 95, 1], [-1, 0, 1, 2]), Hk=1, Hv=2),
    "single_tokens": dict(topo=lambda: ([1] * 9, [-1, 0, 1, 1, 3, -1, 5, 5, 0]), Hk=1, Hv=1),
    "long_nodes": dict(topo=lambda: ([512, 300, 130, 497, 64, 1], [-1, 0, 0, 1, 1, -1]), Hk=1, Hv=2),
    "c1_heads": dict(topo=lambda: ([3, 4, 3, 4, 5, 3, 3, 4, 4, 3, 4, 3, 4],
                                   [-1, 0, 1, 2, 3, 3, 2, 6, -1, 8, 9, 8, 11]), Hk=16, Hv=32),
}


@pytest.mark.parametrize("case", list(CASES))
def test_reference_mode_fp32_matches_oracle(case):
    c = CASES[case]
    lens, par = c["topo"]()
    T = sum(lens)
    q, k, v, g, beta = _inputs(T, c["Hk"], c["Hv"], sum(map(ord, case)))
    print(f"gdn reference fwd fp32 {case}: T={T} nodes={len(lens)}", flush=True)
    o, st = _run(q, k, v, g, beta, lens, par, torch.float32)
    o_ref, st_ref = ogdn.gdn_tree(q, k, v, g, beta, lens, par, mode="reference")
    assert _rel(o, o_ref) < 1e-5, (case, _rel(o, o_ref))
    assert _rel(st, st_ref) < 1e-5, (case, _rel(st, st_ref))
    o_ex, _ = ogdn.gdn_tree(q, k, v, g, beta, lens, par, mode="exact")
    d_ex = _rel(o_ref, o_ex)   # the reference's truncation vs the exact rule (0 when no node exceeds 3 tokens)
    if d_ex > 1e-4:
        assert _rel(o, o_ref) < d_ex / 10, (case, d_ex)


@pytest.mark.parametrize("case", ["forest_multi_block", "long_nodes", "c1_heads"])
def test_reference_mode_bf16_matches_oracle(case):
    c = CASES[case]
    lens, par = c["topo"]()
    T = sum(lens)
    q, k, v, g, beta = _inputs(T, c["Hk"], c["Hv"], 7 + sum(map(ord, case)), realistic_gates=True)
    rb = lambda x: torch.from_numpy(x).bfloat16().float().numpy()
    q, k, v = rb(q), rb(k), rb(v)                 # the oracle sees the same bf16 inputs
    print(f"gdn reference fwd bf16 {case}: T={T}", flush=True)
    o, _ = _run(q, k, v, g, beta, lens, par, torch.bfloat16)
    o_ref, _ = ogdn.gdn_tree(q, k, v, g, beta, lens, par, mode="reference")
    assert _rel(o, o_ref) < 2e-2, (case, _rel(o, o_ref))


@pytest.mark.parametrize("case", list(CASES))
def test_reference_mode_bwd_fp32_matches_autograd_oracle(case):
    c = CASES[case]
    lens, par = c["topo"]()
    T = sum(lens)
    q, k, v, g, beta = _inputs(T, c["Hk"], c["Hv"], 3 + sum(map(ord, case)))
    d_o = np.random.default_rng(11).standard_normal((T, c["Hv"], D)).astype(np.float32)
    print(f"gdn reference bwd fp32 {case}: T={T} nodes={len(lens)}", flush=True)
    got = _run_bwd(q, k, v, g, beta, d_o, lens, par, torch.float32)
    ref = _oracle_grads(q, k, v, g, beta, d_o, lens, par)
    for name, a, b in zip(BWD_NAMES, got, ref):
        assert _rel(a, b) < 1e-5, (case, name, _rel(a, b))


@pytest.mark.parametrize("case", ["forest_multi_block", "long_nodes", "c1_heads"])
def test_reference_mode_bwd_bf16_matches_autograd_oracle(case):
    c = CASES[case]
    lens, par = c["topo"]()
    T = sum(lens)
    q, k, v, g, beta = _inputs(T, c["Hk"], c["Hv"], 5 + sum(map(ord, case)), realistic_gates=True)
    rb = lambda x: torch.from_numpy(x).bfloat16().float().numpy()
    d_o = rb(np.random.default_rng(12).standard_normal((T, c["Hv"], D)).astype(np.float32))
    q, k, v = rb(q), rb(k), rb(v)
    print(f"gdn reference bwd bf16 {case}: T={T}", flush=True)
    got = _run_bwd(q, k, v, g, beta, d_o, lens, par, torch.bfloat16)
    ref = _oracle_grads(q, k, v, g, beta, d_o, lens, par)
    for name, a, b in zip(BWD_NAMES, got, ref):
        assert _rel(a, b) < 2e-2, (case, name, _rel(a, b))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_reference_mode_saved_forward_equals_recompute(dtype):
    """tt_gdn_tree_fwd_save + tt_gdn_tree_bwd_saved give bitwise the outputs,
    node states and gradients of tt_gdn_tree_fwd + the recomputing
    tt_gdn_tree_bwd in the reference mode too (its node-level terms are kept)."""
    from tree_training_amd import gdn as tgdn
    c = CASES["long_nodes"]
    lens, par = c["topo"]()
    T = sum(lens)
    q, k, v, g, beta = _inputs(T, c["Hk"], c["Hv"], 31, realistic_gates=True)
    d_o = np.random.default_rng(13).standard_normal((T, c["Hv"], D)).astype(np.float32)
    tree = GdnTree(lens, par, torch.device("cuda", 0))
    args = (_t(q).to(dtype), _t(k).to(dtype), _t(v).to(dtype), _t(g), _t(beta))
    print(f"gdn reference saved vs recompute {dtype}: T={T}", flush=True)
    o0, st0 = gdn_tree_forward(*args, tree, reference_truncated=True)
    o1, st1, saved = tgdn._gdn_forward(*args, tree, None, True, True, True)
    g0 = gdn_tree_backward(*args, _t(d_o).to(dtype), tree, reference_truncated=True)
    g1 = gdn_tree_backward(*args, _t(d_o).to(dtype), tree, saved=saved, reference_truncated=True)
    torch.cuda.synchronize()
    assert torch.equal(o0, o1) and torch.equal(st0, st1)
    for name, a, b in zip(BWD_NAMES, g0, g1):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("Hk,Hv", [(1, 2), (16, 32)])
def test_reference_mode_block_edges(Hk, Hv, dtype):
    """Nodes of 1, 31, 32, 33, 64, 65 and 97 tokens on one level (and a root of
    33): whole, ragged and single-token correction blocks, in the row layout of
    the level scans (14 pairs) and the column layout (224 pairs), with operands
    of three planes (fp32) and as they come (bf16): outputs, states and gradients
    against the float64 oracle, at each dtype's bar (the states are fp32 from
    exact inputs in both)."""
    lens, par = [33, 1, 31, 32, 33, 64, 65, 97], [-1] + [0] * 7
    T = sum(lens)
    q, k, v, g, beta = _inputs(T, Hk, Hv, 43 + Hv, realistic_gates=True)
    d_o = np.random.default_rng(14).standard_normal((T, Hv, D)).astype(np.float32)
    tol = 1e-5
    if dtype == torch.bfloat16:
        tol = 2e-2
        q, k, v, d_o = (torch.from_numpy(x).bfloat16().float().numpy() for x in (q, k, v, d_o))
    print(f"gdn reference block edges: T={T} heads {Hk}/{Hv} {dtype}", flush=True)
    o, st = _run(q, k, v, g, beta, lens, par, dtype)
    o_ref, st_ref = ogdn.gdn_tree(q, k, v, g, beta, lens, par, mode="reference")
    assert _rel(o, o_ref) < tol and _rel(st, st_ref) < 1e-5
    got = _run_bwd(q, k, v, g, beta, d_o, lens, par, dtype)
    for name, a, b in zip(BWD_NAMES, got, _oracle_grads(q, k, v, g, beta, d_o, lens, par)):
        assert _rel(a, b) < (1e-5 if name in ("dg", "dbeta") else tol), (name, _rel(a, b))


def test_reference_mode_agent16k_two_heads_matches_oracle():
    """Full c5 topology (agent tree, 16,318 tokens, 54 nodes of 64-512 tokens,
    realistic gates), fp32, one q/k head shared by two v heads, against the
    literal float64 oracle. Outputs and node states: < 1e-5 — tighter than
    the reference's own float32 evaluation of the same rule, which the test
    measures too (about 3e-5 on the states after 512-token nodes: its
    cumulative decays lose ~|G| 2^-24 in one float; the kernels carry them in
    two)."""
    lens, par = agent_tree(0)
    T = sum(lens)
    q, k, v, g, beta = _inputs(T, 1, 2, 17, realistic_gates=True)
    print(f"gdn reference fwd 16k: T={T} nodes={len(lens)}", flush=True)
    o, st = _run(q, k, v, g, beta, lens, par, torch.float32)
    o_ref, st_ref = ogdn.gdn_tree(q, k, v, g, beta, lens, par, mode="reference")
    with torch.no_grad():
        _, st32 = ogdn.gdn_tree_reference_torch(*[torch.from_numpy(x) for x in (q, k, v, g, beta)], lens, par,
                                                return_states=True)
    print(f"  o {_rel(o, o_ref):.2e}  states {_rel(st, st_ref):.2e} (the reference's own float32: "
          f"{_rel(st32.double().numpy(), st_ref):.2e})", flush=True)
    assert _rel(o, o_ref) < 1e-5, _rel(o, o_ref)
    assert _rel(st, st_ref) < 1e-5, _rel(st, st_ref)


def test_reference_mode_16k_tree_per_path_equivalence():
    """Full size (agent tree, 16,318 tokens, 16 q/k heads, 32 v heads, bf16):
    the reference's per-node rule depends only on a node's tokens and its
    parent's state, so each sampled root-to-leaf path run alone as a chain of
    the same nodes gives bitwise the tree's outputs and final state there; and
    with d_o only on that path the gradients equal the chain's bitwise and
    vanish elsewhere."""
    lens, par = agent_tree(0)
    T = sum(lens)
    q, k, v, g, beta = _inputs(T, 16, 32, 5, realistic_gates=True)
    print(f"gdn reference 16k per-path: T={T}", flush=True)
    o, st = _run(q, k, v, g, beta, lens, par, torch.bfloat16)
    assert np.isfinite(o).all() and np.isfinite(st).all()
    starts = np.concatenate([[0], np.cumsum(lens)[:-1]])
    leaves = [i for i in range(len(lens)) if i not in set(par)]
    paths = []
    for leaf in (leaves[0], leaves[len(leaves) // 2], leaves[-1]):
        path, j = [], leaf
        while j >= 0:
            path.append(j)
            j = par[j]
        paths.append((leaf, path[::-1]))
    for leaf, path in paths:
        idx = np.concatenate([np.arange(starts[i], starts[i] + lens[i]) for i in path])
        o_p, st_p = _run(q[idx], k[idx], v[idx], g[idx], beta[idx], [lens[i] for i in path],
                         list(range(-1, len(path) - 1)), torch.bfloat16)
        assert np.array_equal(o_p, o[idx])
        assert np.array_equal(st_p[-1], st[leaf])
    leaf, path = paths[1]
    idx = np.concatenate([np.arange(starts[i], starts[i] + lens[i]) for i in path])
    d_o = np.zeros((T, 32, D), np.float32)
    d_o[idx] = np.random.default_rng(4).standard_normal((len(idx), 32, D))
    full = _run_bwd(q, k, v, g, beta, d_o, lens, par, torch.bfloat16)
    chain = _run_bwd(q[idx], k[idx], v[idx], g[idx], beta[idx], d_o[idx], [lens[i] for i in path],
                     list(range(-1, len(path) - 1)), torch.bfloat16)
    off = np.setdiff1d(np.arange(T), idx)
    for name, a, b in zip(BWD_NAMES, full, chain):
        assert np.isfinite(a).all(), name
        assert np.array_equal(a[idx], b), name
        assert not np.any(a[off]), name
