"""gr_linear against float64 at the edges of its tiles (64 x 64 to 128 x 192), of
its pipeline (8 stages of 64 features and more) and of its fragments (16
columns).

Bounds: float32 sums of K products differ from the exact sum by at most K 2^-24
of the sum of their magnitudes (here taken with a factor of 1/8: errors of both
signs); a 16-bit output adds half a unit in the last place (2^-8 bf16, 2^-11
fp16), and SwiGLU's exponential and quotient a few float32 units."""

import pytest
import torch

from vllm_gr_amd import _C, ops
from vllm_gr_amd.v1.sid_decoder import DecoderConfig, SidDecoder, init_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(1, 16, 512), (5, 48, 576), (64, 64, 640), (65, 80, 1024), (127, 208, 2048),
                                   (129, 400, 512), (200, 4096, 704), (512, 2048, 1536), (384, 6144, 512)])
def test_linear(device, dtype, M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g).to(dtype).to(device)[:, :K]  # strided rows
    w = (torch.randn(2 * N, K, generator=g) * 0.05).to(dtype).to(device)
    ref = x.double() @ w.double().t()
    mag = x.double().abs() @ w.double().abs().t()
    own = mag * K * 2.0 ** -24 / 8 + 1e-9
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    y32 = ops.linear(x, w[:N], out_f32=True)
    y = ops.linear(x, w[:N])
    z = ops.linear(x, w, swiglu=True)
    assert ((y32.double() - ref[:, :N]).abs() <= own[:, :N]).all()
    assert torch.equal(y, y32.to(dtype))
    gate, up = ref[:, :N], ref[:, N:]
    sw = gate * torch.sigmoid(gate) * up
    # gate and up are rounded once each, |d silu| <= 1.1 |d gate| and |silu| <= |gate|; the exponential's own
    # error 2^-21 of the result; fp16's subnormal step
    dg, du = own[:, :N] + half * gate.abs(), own[:, N:] + half * up.abs()
    tol = sw.abs() * (1.01 * half + 2.0 ** -21) + 1.01 * (1.1 * dg * up.abs() + gate.abs() * du) + 2.0 ** -24
    assert ((z.double() - sw).abs() <= tol).all()


# (rows, columns, SwiGLU, its tile): every tile of either form, with rows and columns left over
TILES = [(65, 80, 0, (64, 64)), (300, 4112, 0, (128, 64)), (301, 8144, 0, (128, 128)), (500, 8208, 0, (128, 192)),
         (65, 80, 1, (64, 64)), (301, 2064, 1, (128, 64)), (300, 4112, 1, (128, 128)), (500, 6128, 1, (128, 192))]


@pytest.mark.parametrize("K", [576, 640])  # an odd and an even number of stages past every pipeline's first
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,swiglu,tile", TILES)
def test_linear_every_tile(device, dtype, M, N, swiglu, tile, K):
    assert _C.lib().gr_linear_tile(M, N, K, swiglu) == 1000 * tile[0] + tile[1]
    assert M % tile[0] and (N * (1 + swiglu)) % tile[1]
    test_linear(device, dtype, M, N, K)


def test_linear_refuses(device):
    x = torch.zeros(4, 512, device=device, dtype=torch.bfloat16)
    w = torch.zeros(24, 512, device=device, dtype=torch.bfloat16)
    for a, b in ((x, w), (x.float(), w[:16].float()), (x[:, :448], w[:16, :448]), (x[:, 1:], w[:16, 1:])):
        assert not ops.linear_supported(a, b)
        with pytest.raises(ValueError):
            ops.linear(a, b)
    assert ops.linear(x[:0], w[:16]).shape == (0, 16)


def _decoder(device, dtype=torch.bfloat16, vocab=208):
    cfg = DecoderConfig(num_layers=1, hidden=512, num_heads=4, num_kv_heads=2, ffn=512, vocab=vocab, dtype=dtype)
    return SidDecoder(cfg, init_weights(cfg, 3, device), max_position=8)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_logits_are_rounded_alike_at_every_row_count(device, dtype):
    """Logits are the model type's values in float32, on either side of the row
    count from which the library computes them: a beam's score, and a tie of two
    of them, is not a matter of how many requests share the step."""
    dec = _decoder(device, dtype)
    hidden = torch.randn(513, 512, generator=torch.Generator().manual_seed(2)).to(dtype).to(device)
    want = (hidden.double() @ dec.w["lm_head"].double().t())
    mag = hidden.double().abs() @ dec.w["lm_head"].double().abs().t()
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for rows in (1, 8, 200, 512, 513):
        got = dec.compute_logits(hidden[:rows])
        assert got.dtype == torch.float32 and torch.equal(got, got.to(dtype).float()), rows
        tol = want[:rows].abs() * half * 1.01 + mag[:rows] * 512 * 2.0 ** -24 / 8 + 2.0 ** -25
        assert ((got.double() - want[:rows]).abs() <= tol).all(), rows


def test_logits_under_autograd_and_transforms(device):
    """compute_logits is differentiable in the hidden states and the weights, and
    works under vmap, forward mode and tracing, as the torch product it stands for."""
    import torch.autograd.forward_ad as fw
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    dec = _decoder(device)
    w = dec.w["lm_head"]
    h = torch.randn(6, 512, device=device, dtype=torch.bfloat16)
    plain = lambda x, w=w: torch.nn.functional.linear(x, w).float()
    up = torch.randn(6, 208, device=device)
    for hg, wg in ((True, False), (False, True), (True, True)):
        x, lm = h.clone().requires_grad_(hg), w.clone().requires_grad_(wg)
        x2, lm2 = h.clone().requires_grad_(hg), w.clone().requires_grad_(wg)
        dec.w["lm_head"] = lm
        (dec.compute_logits(x) * up).sum().backward()
        (plain(x2, lm2) * up).sum().backward()
        for a, b in ((x, x2), (lm, lm2)):
            assert (a.grad is None) == (b.grad is None)
            assert a.grad is None or torch.equal(a.grad, b.grad)
    dec.w["lm_head"] = w
    assert torch.equal(torch.func.vmap(dec.compute_logits)(h.view(2, 3, 512)), torch.func.vmap(plain)(h.view(2, 3, 512)))
    t = torch.randn_like(h)
    for a, b in zip(torch.func.jvp(dec.compute_logits, (h,), (t,)), torch.func.jvp(plain, (h,), (t,))):
        assert torch.equal(a, b)
    with fw.dual_level():
        assert torch.equal(fw.unpack_dual(dec.compute_logits(fw.make_dual(h, t))).tangent,
                           fw.unpack_dual(plain(fw.make_dual(h, t))).tangent)
    traced = make_fx(lambda x: dec.compute_logits(x))(h)
    assert torch.equal(traced(2 * h), plain(2 * h))  # not h's logits as a constant
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        assert dec.compute_logits(mode.from_tensor(h)).shape == (6, 208)
    with torch.no_grad():  # the usual call
        assert not dec.compute_logits(h.clone().requires_grad_()).requires_grad
