"""Pruning of long rows (from 20480 logits) over several workgroups a row, bit for bit
against the CPU oracle, at the edges of its range and of its chunks (1024 logits), slices and
72-chunk panels; and the same bits from the base workspace (one workgroup a row)."""

import numpy as np
import pytest
import torch

from oracle import prune as op
from vllm_gr_amd import _C, ops, workloads
from vllm_gr_amd.entrypoints.catalog import Catalog

pytestmark = pytest.mark.gpu


def _bits(t):
    a = t.cpu().numpy()
    return a.view({4: np.int32, 8: np.int64}[a.itemsize])


def _run(wl, device, eos=-1, base=False):
    d = wl.to(device)
    R, W, V = wl.logits.shape
    n = (_C.lib().gr_beam_prune_workspace_size if base else _C.lib().gr_beam_prune_workspace_size_split)(R, W, V, wl.k)
    # garbage in the workspace: nothing may be taken from it before it is written
    ws = torch.full((n,), 0xA5, dtype=torch.uint8, device=device)
    out = ops.beam_prune_topk(d.logits, d.cum, wl.k, eos, workspace=ws)
    torch.cuda.synchronize()
    return out


def _check(wl, device, eos=-1):
    want = op.prune_topk(wl.logits.numpy(), wl.cum.numpy(), wl.k, eos)
    got = _run(wl, device, eos)
    for g, name in zip(got, ("parent", "token", "score", "eos_score")):
        assert np.array_equal(_bits(g), want[name].view(np.int32)), name
    for g, b in zip(got, _run(wl, device, eos, base=True)):
        assert np.array_equal(_bits(g), _bits(b))


@pytest.mark.parametrize("R,W,V,k", [(1, 1, 20476, 9), (1, 1, 20480, 1), (2, 3, 20484, 256), (1, 5, 21504, 100), (2, 2, 65536, 32),
                                     (1, 2, 73728, 17), (1, 3, 73732, 64), (1, 4, 151936, 32), (3, 4, 22528, 300), (2, 300, 32768, 8)])
def test_split_rows(device, R, W, V, k):
    _check(workloads.make_prune(R=R, W=W, V=V, k=k, seed=V + k), device)


@pytest.mark.parametrize("kind", ["ties", "equal", "masked", "tail", "eos"])
def test_split_rows_hard_inputs(device, kind):
    """Many ties at the bound, one value throughout (more survivors than the
    list holds), masked tokens and a masked beam, the best at the row's end, EOS."""
    wl = workloads.make_prune(R=2, W=4, V=20488, k=32, seed=3)
    lg = wl.logits
    if kind == "ties":
        lg.copy_(torch.round(lg))
    elif kind == "equal":
        lg.fill_(1.5)
        lg[0, 0] = -0.0
    elif kind == "masked":
        lg[0, :, 10:] = float("-inf")
        lg[1, 2] = float("-inf")
    elif kind == "tail":
        lg[:, :, -40:] += 50.0
    _check(wl, device, eos=int(lg[0, 0].argmax()) if kind == "eos" else -1)


def test_split_rows_f64_lists(device):
    """float64 scores and the candidate lists: the same bits from either workspace."""
    wl = workloads.make_prune(R=2, W=8, V=40004, k=48, seed=9)
    lg, cum = wl.logits.to(device), wl.cum.to(device).double()
    res = []
    for size in (_C.lib().gr_beam_prune_workspace_size, _C.lib().gr_beam_prune_workspace_size_split):
        ws = torch.empty(size(2, 8, 40004, 48), dtype=torch.uint8, device=device)
        res.append(ops.beam_prune_topk(lg, cum, 48, 5, workspace=ws, candidates=True))
    torch.cuda.synchronize()
    for x, y in zip(*res):
        assert np.array_equal(_bits(x), _bits(y))


@pytest.mark.parametrize("W,k,V", [(1, 1, 64), (32, 128, 1024), (33, 124, 1024), (200, 20, 256), (600, 6, 128)])
@pytest.mark.parametrize("kind", ["plain", "dead", "collapse", "empty"])
def test_one_group_merge(device, W, k, V, kind):
    """Requests whose candidates fit one merge group (W k <= 4096): dead rows
    (-inf scores), scores that round to one value, and too few candidates."""
    wl = workloads.make_prune(R=3, W=W, V=V, k=k, seed=W + k)
    eos = -1
    if kind == "dead":
        wl.cum[0, W // 2:] = float("-inf")
        wl.cum[1] = float("-inf")
    elif kind == "collapse":
        wl.cum.fill_(-1e15)
    elif kind == "empty":
        eos = 5
        wl.logits[:, :, eos] += 30.0  # with k = 1 no candidate is left
    _check(wl, device, eos)


@pytest.mark.parametrize("f64", [False, True])
def test_split_rows_catalog(device, f64):
    """Long rows under a catalog: beams at the root, inside the trie, dead, complete,
    and with EOS among their children; bit for bit against the masked oracle, from
    either workspace."""
    rng = np.random.default_rng(21)
    R, W, V, k, eos = 2, 10, 20484, 32, 7
    cat = Catalog()
    seqs = [rng.integers(0, V, size=3).tolist() for _ in range(1500)]
    for s in seqs + [[s[0], eos] for s in seqs[:30]]:
        cat.add(s)
    pick = lambda n, top: seqs[int(rng.integers(0, top))][:n]
    prefixes = [[([], pick(1, 30), pick(2, 1500), [V - 1, V - 2], pick(3, 1500))[b % 5] for b in range(W)]
                for _ in range(R)]
    node = torch.tensor([[cat.node_of(p) for p in row] for row in prefixes], dtype=torch.int32)
    allowed = np.zeros((R, W, V), bool)
    for r in range(R):
        for b in range(W):
            allowed[r, b, list(cat.valid(prefixes[r][b]))] = True
    logits = torch.from_numpy((rng.standard_normal((R, W, V)) * 3 + allowed * 9.0).astype(np.float32))
    cum = torch.from_numpy(rng.uniform(-20, 0, (R, W)))
    cum = cum if f64 else cum.float()
    want = op.prune_topk(logits.numpy(), cum.numpy(), k, eos, allowed=allowed)
    assert (want["parent"] >= 0).sum() > R * k // 2 and np.isfinite(want["eos_score64"]).any()
    for size in (_C.lib().gr_beam_prune_workspace_size_split, _C.lib().gr_beam_prune_workspace_size):
        ws = torch.full((size(R, W, V, k),), 0xA5, dtype=torch.uint8, device=device)
        status = ops.new_status(device)
        parent, token, score, eos_score, nodes = ops.beam_prune_topk(
            logits.to(device), cum.to(device), k, eos, catalog=cat.to_device(device), beam_node=node.to(device),
            workspace=ws, status=status)
        torch.cuda.synchronize()
        ops.check_status(status)
        names = ("parent", "token") + (("score64", "eos_score64") if f64 else ("score", "eos_score"))
        for g, name in zip((parent, token, score, eos_score), names):
            w = want[name].reshape(g.shape)
            assert np.array_equal(_bits(g), w.view({4: np.int32, 8: np.int64}[w.itemsize])), name
        assert nodes.cpu().tolist() == [[cat.node_of(prefixes[r][p] + [t]) if p >= 0 else -1
                                         for p, t in zip(want["parent"][r], want["token"][r])] for r in range(R)]


@pytest.mark.parametrize("kind", ["nan", "inf"])
def test_split_rows_nan_and_infinity(device, kind):
    """A few NaN logits count as -inf ones do (never selected, 2^-126 in the sum);
    an infinite one leaves its beam without a finite score: from either workspace."""
    wl = workloads.make_prune(R=2, W=4, V=20492, k=24, seed=13)
    at = torch.randint(0, 20492, (2, 4, 9), generator=torch.Generator().manual_seed(5))
    wl.logits[1].scatter_(1, at[1], float("nan" if kind == "nan" else "-inf"))
    if kind == "inf":
        wl.logits[0, 2, 777] = float("inf")
    want_in = torch.where(wl.logits.isnan(), -torch.inf, wl.logits)
    want = op.prune_topk(want_in.numpy(), wl.cum.numpy(), wl.k)
    for base in (False, True):
        got = _run(wl, device, base=base)
        for g, name in zip(got, ("parent", "token", "score", "eos_score")):
            assert np.array_equal(_bits(g), want[name].view(np.int32)), (name, base)
