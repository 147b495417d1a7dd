"""The decode kernel for 512-byte K / V rows (float32 at head_dim 128, bf16 /
fp16 at head_dim 256) at the edges of its tiles, against the float64 oracle.

Bounds.  The kernel works in float32 and rounds once, to the output type: at
most half a unit in the last place of the result (of 8 significant bits in
bf16: 2^-8 of it; 11 in fp16: 2^-11; 24 in float32: 2^-24), plus the float32
path's own error, taken as 2^-15 of the largest |v| for 16-bit inputs
(probabilities carried to 16 bits, float32 sums) and 1e-5 for float32 (the
path's stated bound).
"""

import numpy as np
import pytest
import torch

from oracle import attention as oa
from vllm_gr_amd import ops, workloads

pytestmark = pytest.mark.gpu

DTYPES = [(torch.float32, 128), (torch.bfloat16, 256), (torch.float16, 256)]
HALF_ULP = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _run(wl, device, kernel="auto", sinks=None, split=True, status=None):
    d = wl.to(device)
    lse = torch.empty(d.q.shape[:2], dtype=torch.float32, device=device)
    ops.set_decode_kernel(kernel)
    try:
        out = ops.beam_attn_decode(d.q, d.k_cache, d.v_cache, d.prefix_bt, d.prefix_len, d.beam_start, d.suffix_bt,
                                   d.suffix_len, q_per_beam=d.q_per_beam, scale=d.scale, softcap=d.softcap,
                                   max_beams_per_req=d.max_beams, lse=lse, sinks=sinks, split=split, status=status)
        torch.cuda.synchronize()
    finally:
        ops.set_decode_kernel("auto")
    return out.cpu().to(torch.float64).numpy(), lse.cpu().to(torch.float64).numpy()


def _bound(ref, wl, dtype):
    own = 1e-5 if dtype == torch.float32 else 2.0 ** -15 * float(wl.kv_cache[1].abs().max())
    return 1.01 * HALF_ULP[dtype] * np.abs(ref) + own


# (R, W, P, L, Hq, Hkv, T, block size, soft cap): a single key; one tile short,
# full and one over; eight wave tiles and one over; several rounds of tiles;
# chunks with one row, with beams across a chunk's edge, with sixteen beams
CASES = [
    (1, 1, 1, 0, 1, 1, 1, 16, 0.0), (1, 3, 31, 1, 4, 4, 1, 16, 0.0), (2, 5, 32, 2, 4, 2, 1, 16, 30.0),
    (1, 17, 33, 3, 2, 2, 1, 32, 0.0), (3, 16, 256, (1, 9), 8, 8, 1, 16, 0.0), (2, 9, 257, (3, 20), 6, 2, 3, 16, 0.0),
    (9, 4, 700, (1, 40), 16, 2, 1, 8, 50.0), (2, 7, 0, (1, 5), 8, 2, 2, 16, 0.0),
]


@pytest.mark.parametrize("dtype,D", DTYPES)
@pytest.mark.parametrize("case", CASES)
def test_row512_edges(device, dtype, D, case):
    R, W, P, L, Hq, Hkv, T, bs, cap = case
    L = (max(L[0], T), L[1]) if isinstance(L, tuple) else L
    wl = workloads.make_decode(R=R, W=W, P=P, L=L, Hq=Hq, Hkv=Hkv, D=D, dtype=dtype, block_size=bs,
                               input_scale=1.0, seed=R + W + P, q_per_beam=T, softcap=cap)
    out, lse = _run(wl, device)
    kv = wl.kv_cache.to(torch.float64).numpy()
    ref, ref_lse = oa.beam_attention_cascade(
        wl.q.to(torch.float64).numpy(), kv[0], kv[1], wl.prefix_bt.numpy(), wl.prefix_len.numpy(),
        wl.beam_start.numpy(), wl.suffix_bt.numpy(), wl.suffix_len.numpy(), q_per_beam=T, scale=wl.scale,
        softcap=cap, block_size=bs)
    assert (np.abs(out - ref) <= _bound(ref, wl, dtype)).all(), np.abs(out - ref).max()
    fin = np.isfinite(ref_lse)
    assert (np.isfinite(lse) == fin).all() and np.abs(lse[fin] - ref_lse[fin]).max(initial=0.0) <= 1e-4


@pytest.mark.parametrize("dtype,D", DTYPES)
def test_row512_sinks_and_bad_blocks_as_generic(device, dtype, D):
    """Sinks, and table entries out of range (left out and flagged), as the
    generic kernel treats them."""
    wl = workloads.make_decode(R=2, W=6, P=90, L=(2, 9), Hq=8, Hkv=2, D=D, dtype=dtype, input_scale=1.0, seed=5)
    wl.prefix_bt[1, 2] = -1
    wl.suffix_bt[3, 0] = 1 << 20
    sinks = torch.randn(8, device=device)
    res = []
    for kernel in ("auto", "generic"):
        status = ops.new_status(device)
        out, lse = _run(wl, device, kernel, sinks, status=status)
        res.append((out, lse, int(status.item())))
    (a, la, sa), (b, lb, sb) = res
    assert sa == sb != 0
    assert (np.abs(a - b) <= 2 * _bound(b, wl, dtype)).all()
    assert np.abs(la - lb).max() <= 1e-4


@pytest.mark.parametrize("dtype,D", DTYPES[1:])
def test_row512_infinite_value_row(device, dtype, D):
    """An infinite V row of a visible key gives that infinity, as a float32 weight does."""
    wl = workloads.make_decode(R=1, W=4, P=40, L=1, Hq=2, Hkv=2, D=D, dtype=dtype, input_scale=1.0, seed=8)
    blk = int(wl.prefix_bt[0, 1])
    wl.kv_cache[1, blk, 3, 0] = float("inf")
    wl.kv_cache[1, blk, 3, 1] = -float("inf")
    out, _ = _run(wl, device)
    assert (out[:, 0] == np.inf).all() and (out[:, 1] == -np.inf).all()


@pytest.mark.parametrize("dtype,D", DTYPES)
def test_row512_weights_keep_float32(device, dtype, D):
    """Two keys of nearly equal weight whose V rows cancel: the result is the
    difference of the weights, which terms of fewer bits than float32's show.

    Bound: the output's rounding, plus 2^-20 (of |v| = 1) for the float32 steps
    -- scores of at most 2 in size, rounded at 2^-23, and an exponential and sums
    of a few float32 units."""
    g = torch.Generator().manual_seed(D)
    wl = workloads.make_decode(R=1, W=64, P=2, L=0, Hq=16, Hkv=2, D=D, dtype=dtype, input_scale=0.5, seed=4)
    b = int(wl.prefix_bt[0, 0])
    wl.kv_cache[0, b, 1] = wl.kv_cache[0, b, 0]
    wl.kv_cache[0, b, 1, :, :4] += 0.05 * torch.randn(2, 4, generator=g).to(dtype)
    wl.kv_cache[1, b, 0] = 1.0
    wl.kv_cache[1, b, 1] = -1.0
    out, _ = _run(wl, device)
    q, k = wl.q.double().view(64, 2, 8, D), wl.kv_cache[0, b, :2].double()
    ref = torch.tanh(torch.einsum("whgd,hd->whg", q, (k[0] - k[1])) * wl.scale / 2).reshape(64, 16, 1).numpy()
    assert (np.abs(out - ref) <= 1.01 * HALF_ULP[dtype] * np.abs(ref) + 2.0 ** -20).all(), np.abs(out - ref).max()


@pytest.mark.parametrize("dtype,D", DTYPES)
def test_row512_small_weight_of_a_large_value(device, dtype, D):
    """A weight near 2^-29 on a large V row beside a V row of zeros: the result
    is that weight.

    Bound: the output's rounding (half of fp16's subnormal step at least), plus
    the score's error as a share of the result: a float32 sum of D products of one
    sign, each addition rounded at 2^-24 of a running sum that is half of the whole
    on average, and 2^-20 for the exponential and the quotient."""
    wl = workloads.make_decode(R=1, W=16, P=2, L=0, Hq=8, Hkv=1, D=D, dtype=dtype, input_scale=1.0, seed=6)
    b = int(wl.prefix_bt[0, 0])
    sign = torch.randn(D, generator=torch.Generator().manual_seed(7)).sign()
    amp = 18.0 / D ** 0.5 * (1.0 + torch.arange(128).view(16, 8, 1) / 1024.0)
    wl.q.copy_((amp * sign).to(dtype))
    wl.kv_cache[0, b, 0, 0] = sign.to(dtype)
    wl.kv_cache[0, b, 1, 0] = 0.0
    wl.kv_cache[1, b, 0, 0] = 0.0
    wl.kv_cache[1, b, 1, 0] = 60000.0
    out, _ = _run(wl, device)
    s = (wl.q.double() * sign.double()).sum(-1, keepdim=True) * wl.scale
    v = wl.kv_cache[1, b, 1, 0, 0].double()
    ref = (v / (1.0 + torch.exp(s))).numpy()
    sub = 2.0 ** -25 if dtype == torch.float16 else 0.0
    own = D * 2.0 ** -24 * s.numpy() / 2 + 2.0 ** -20
    assert (np.abs(out - ref) <= (1.01 * HALF_ULP[dtype] + own) * np.abs(ref) + sub).all(), (np.abs(out - ref) / ref).max()


def _padded(t, pad, dims):
    """t's values in a tensor whose given dims are `pad` longer, viewed at t's shape."""
    shape = [n + (pad if i in dims else 0) for i, n in enumerate(t.shape)]
    return torch.zeros(shape, dtype=t.dtype, device=t.device)[tuple(slice(n) for n in t.shape)].copy_(t)


@pytest.mark.parametrize("dtype,D", DTYPES)
def test_row512_layouts(device, dtype, D):
    """Caches padded per head or held head-major, strided q and out, suffixes
    that start inside their blocks: the same bits as the packed form, which is
    checked against the oracle.  Bases or strides off the 16-byte grid: the
    generic kernel's bits."""
    wl = workloads.make_decode(R=2, W=5, P=75, L=(3, 17), Hq=8, Hkv=2, D=D, dtype=dtype, input_scale=1.0, seed=11,
                               suffix_blocks=3)
    start = torch.randint(0, 16, (10,), dtype=torch.int32, generator=torch.Generator().manual_seed(1))
    kv = wl.kv_cache.double().numpy()
    ref, _ = oa.beam_attention_cascade(
        wl.q.double().numpy(), kv[0], kv[1], wl.prefix_bt.numpy(), wl.prefix_len.numpy(), wl.beam_start.numpy(),
        wl.suffix_bt.numpy(), wl.suffix_len.numpy(), start.numpy(), q_per_beam=1, scale=wl.scale, block_size=16)
    d, ch = wl.to(device), 16 // wl.q.element_size()
    start = start.to(device)

    def run(q, kvc, out, kernel="auto"):
        ops.set_decode_kernel(kernel)
        try:
            ops.beam_attn_decode(q, kvc[0], kvc[1], d.prefix_bt, d.prefix_len, d.beam_start, d.suffix_bt, d.suffix_len,
                                 start, scale=d.scale, max_beams_per_req=5, out=out)
            torch.cuda.synchronize()
        finally:
            ops.set_decode_kernel("auto")
        return out.contiguous()

    new = lambda: torch.empty_like(d.q)
    base = run(d.q, d.kv_cache, new())
    assert (np.abs(base.double().cpu().numpy() - ref) <= _bound(ref, wl, dtype)).all()
    wide = lambda t, pad: _padded(t.flatten(1), pad, (1,)).unflatten(1, t.shape[1:])  # token stride Hq D + pad
    for name, q, kvc, out in (
            ("padded heads", d.q, _padded(d.kv_cache, ch, (4,)), new()),
            ("padded tokens", d.q, _padded(d.kv_cache, 1, (2, 3)), new()),
            ("head-major", d.q, d.kv_cache.transpose(2, 3).contiguous().transpose(2, 3), new()),
            ("strided q, out", wide(d.q, ch), d.kv_cache, wide(new(), 3 * ch))):
        assert torch.equal(run(q, kvc, out), base), name
    gen = run(d.q, d.kv_cache, new(), "generic")
    off = torch.zeros(d.kv_cache.numel() + 1, dtype=dtype, device=device)[1:].view_as(d.kv_cache).copy_(d.kv_cache)
    for name, q, kvc, out in (
            ("unaligned heads", d.q, _padded(d.kv_cache, 1, (4,)), new()),
            ("unaligned base", d.q, off, new()),
            ("unaligned q", wide(d.q, 1), d.kv_cache, new()),
            ("unaligned out", d.q, d.kv_cache, wide(new(), 1))):
        assert torch.equal(run(q, kvc, out), gen), name


@pytest.mark.parametrize("dtype,D", DTYPES)
def test_row512_weights_of_every_size(device, dtype, D):
    """Scores spread over some 30: tiles with large weights only and tiles with
    weights far below 2^-12 of the row's largest, in one row.

    Bound: as above, plus the scores' float32 sums of D products (errors of both
    signs: 4 sqrt(D) 2^-24 of the largest score, 20) on the largest |v|."""
    wl = workloads.make_decode(R=2, W=11, P=500, L=(1, 6), Hq=8, Hkv=2, D=D, dtype=dtype, input_scale=2.0, seed=17)
    wl.kv_cache[0, wl.prefix_bt[:, ::2].long().flatten()] /= 8  # every other block: near ties
    out, lse = _run(wl, device)
    kv = wl.kv_cache.double().numpy()
    ref, ref_lse = oa.beam_attention_cascade(
        wl.q.double().numpy(), kv[0], kv[1], wl.prefix_bt.numpy(), wl.prefix_len.numpy(), wl.beam_start.numpy(),
        wl.suffix_bt.numpy(), wl.suffix_len.numpy(), q_per_beam=1, scale=wl.scale, block_size=16)
    own = 4 * D ** 0.5 * 2.0 ** -24 * 20 * float(wl.kv_cache[1].abs().max())
    assert (np.abs(out - ref) <= _bound(ref, wl, dtype) + own).all(), np.abs(out - ref).max()
    assert np.abs(lse - ref_lse).max() <= 1e-4
