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
