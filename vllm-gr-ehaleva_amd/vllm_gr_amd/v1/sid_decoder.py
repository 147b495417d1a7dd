"""Random-init Qwen-style decoder for end-to-end semantic-ID beam decode.

The reference serves a Qwen3 checkpoint through vLLM's model executor
(vllm==0.14, not vendored; the semantic-ID tasks use Qwen3 chat templates,
benchmarks/open_one_rec/tasks/recommendation/config.py:19).  This is the
same architecture, sized by a :class:`DecoderConfig`, with weights drawn
from N(0, std) -- there are no checkpoints here:

* token embedding, tied to the lm_head by default;
* per layer: RMSNorm, q/k/v projections (no bias), per-head RMSNorm of q and
  k, rotary embedding with rotate-half pairing (theta 1e6) at the positions
  the caller gives, attention through the BeamAttention backend, o
  projection, residual add; RMSNorm, SwiGLU MLP (silu(gate) * up, down),
  residual add;
* final RMSNorm; logits = lm_head products in ``cfg.dtype``, widened to float32.

The projections of a decode step's qkv, o, gate_up (with its SiLU gate) and
lm_head are gr_linear where that is the faster (up to 512 rows, from at most 2048
features: ``_own_sizes``); the others are ``torch.nn.functional.linear`` (hipBLASLt on ROCm).  The
elementwise stages are fused HIP kernels (include/gr_decoder.h): residual add
+ RMSNorm, per-head q/k RMSNorm + rotary + K/V cache write through the slot
mapping, and the SiLU-gated product.  Attention is
:class:`BeamAttentionImpl.forward`, the call vLLM's Attention layer makes
(beam_attn.py:703-755), with the K/V already written (key/value None).
Positions follow the reference's rule (a beam's j-th suffix token sits at prefix_len + j,
engine_core_patch.py:362-365); logits are taken for one row per beam, the
beam's newest token (:367-369).
"""

from __future__ import annotations

import math
from dataclasses import dataclass

import torch
import torch.nn.functional as F

from .. import ops
from .attention.backends.beam_attn import BeamAttentionImpl


@dataclass(frozen=True)
class DecoderConfig:
    num_layers: int = 28
    hidden: int = 2048
    num_heads: int = 16
    num_kv_heads: int = 8
    head_dim: int = 128
    ffn: int = 6144
    vocab: int = 8192
    rope_theta: float = 1.0e6
    rms_eps: float = 1.0e-6
    tie_embeddings: bool = True
    init_std: float = 0.02
    dtype: torch.dtype = torch.bfloat16

    @property
    def q_size(self) -> int:
        return self.num_heads * self.head_dim

    @property
    def kv_size(self) -> int:
        return self.num_kv_heads * self.head_dim

    def num_params(self) -> int:
        H, L = self.hidden, self.num_layers
        per_layer = (H * (self.q_size + 2 * self.kv_size) + self.q_size * H + 3 * H * self.ffn
                     + 2 * H + 2 * self.head_dim)
        emb = self.vocab * H * (1 if self.tie_embeddings else 2)
        return L * per_layer + emb + H


#: the 28-layer, 2048-hidden, 16/8-head, 6144-FFN, 8192-token decoder
SID_DECODER_1P7B = DecoderConfig()


def init_weights(cfg: DecoderConfig, seed: int, device="cpu") -> dict[str, torch.Tensor]:
    """Weights in nn.Linear layout ``[out, in]``, drawn from one generator on
    ``device`` in a fixed order (embedding, then per layer qkv, o, gate_up,
    down), N(0, init_std) in float32 rounded to ``cfg.dtype``; norm weights
    are ones.  The same seed and device give the same weights."""
    dev = torch.device(device)
    g = torch.Generator(device=dev)
    g.manual_seed(seed)

    def normal(*shape):
        w = torch.randn(*shape, generator=g, device=dev, dtype=torch.float32)
        return w.mul_(cfg.init_std).to(cfg.dtype)

    ones = lambda n: torch.ones(n, device=dev, dtype=cfg.dtype)
    H = cfg.hidden
    w = {"embed": normal(cfg.vocab, H)}
    for i in range(cfg.num_layers):
        p = f"layers.{i}."
        w[p + "qkv"] = normal(cfg.q_size + 2 * cfg.kv_size, H)
        w[p + "o"] = normal(H, cfg.q_size)
        w[p + "gate_up"] = normal(2 * cfg.ffn, H)
        w[p + "down"] = normal(H, cfg.ffn)
        w[p + "input_norm"] = ones(H)
        w[p + "post_norm"] = ones(H)
        w[p + "q_norm"] = ones(cfg.head_dim)
        w[p + "k_norm"] = ones(cfg.head_dim)
    w["final_norm"] = ones(H)
    w["lm_head"] = w["embed"] if cfg.tie_embeddings else normal(cfg.vocab, H)
    return w


class RotaryEmbedding:
    """Tables of the rotate-half rotary embedding: pair (i, i + D/2) turns by
    ``pos * theta^(-2i/D)``; cos/sin ``[max_pos, D/2]`` evaluated in float64
    and stored as float32 on the device (read by gr_qk_norm_rope_cache)."""

    def __init__(self, head_dim: int, theta: float, max_pos: int, device):
        half = head_dim // 2
        inv = 1.0 / (theta ** (torch.arange(0, half, dtype=torch.float64) * 2.0 / head_dim))
        ang = torch.arange(max_pos, dtype=torch.float64)[:, None] * inv[None]
        self.cos = ang.cos().float().to(device)
        self.sin = ang.sin().float().to(device)
        self.max_pos = max_pos


def _plain(*ts: torch.Tensor) -> bool:
    """Whether a kernel on the tensors' addresses can stand in for a torch
    operation: ordinary tensors, and nothing that follows torch operations --
    an autograd graph, forward mode, vmap and the other function transforms, a
    dispatch mode (fake tensors, tracing) or a compiler -- would miss it.  (The
    layers of ``forward`` run such kernels throughout; ``compute_logits`` is one
    product and keeps what the torch product does.)"""
    return (all(type(t) in (torch.Tensor, torch.nn.Parameter) for t in ts)
            and not (torch.is_grad_enabled() and any(t.requires_grad for t in ts))
            and torch.autograd.forward_ad._current_level < 0 and torch._C._functorch.peek_interpreter_stack() is None
            and torch._C._len_torch_dispatch_stack() == 0
            and not torch.jit.is_tracing() and not torch.compiler.is_compiling())


def _own_sizes(m: int, rows: int, k: int, swiglu: bool) -> bool:
    """Whether gr_linear takes a projection of ``m`` rows by ``rows`` weight rows
    of ``k`` features.

    Measured with cold weights over 1 to 512 rows, 512 to 151936 weight rows and
    512 to 2048 features, own time / the library's (SwiGLU: its product and the
    gate kernel's):

    * workgroups that fill the chip once (128 x 192 tiles, column tiles whole on
      one of the 8 XCDs of 32 CUs) and SwiGLU, 0.37 to 0.91, or at most 1024
      features, 0.44 to 1.00 (of random sizes 1 in 100 up to 1.17).  In more rounds
      0.75 to 1.60, SwiGLU 0.43 to 1.35;
    * one round and more features: 0.51 to 1.00, but not where few columns leave
      most CUs idle and the rows fill the library's tiles (33 to 128 rows: 512
      columns 0.97 to 1.04, 1024 0.85 to 1.09, 2048 at 64 and 128 rows 0.99 to
      1.03), and not around its best fits past 1536 features (337 to 384 rows, 3072
      and 4096 columns 1.01 to 1.08; 257 to 315 rows, 5664 to 6512 columns 1.04 to
      1.10, though 0.80 to 0.89 at 320 to 340);
    * up to 100 rows the weights' way from memory is the time, also in more
      rounds: 0.55 to 0.98 past 1024 features;
    * above the limits: 768 rows, SwiGLU 2048 in, 6144 out 53 us against 44; 6144
      in, 2048 out, 8 rows 21 against 12."""
    if m > 512 or k > 2048:
        return False
    one_round = -(-m // 128) * -(-rows // (8 * 192)) <= 32
    if swiglu or k <= 1024:
        return one_round
    if not one_round:
        return m <= 100
    if m <= 32:
        return True
    if m <= 128:
        return rows > 2048 or (rows > 1024 and m % 64 != 0)
    if k > 1536 and 256 < m <= 384 and 2560 < rows < 8192:
        return rows <= 5120 and m <= 336
    return rows > 512


def _own_linear(x: torch.Tensor, w: torch.Tensor, swiglu: bool = False) -> bool:
    return _own_sizes(x.shape[0], *w.shape, swiglu) and ops.linear_supported(x, w, swiglu)


def _linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return ops.linear(x, w) if _own_linear(x, w) else F.linear(x, w)


def _swiglu(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return ops.linear(x, w, swiglu=True) if _own_linear(x, w, True) else ops.silu_mul(F.linear(x, w))


class SidDecoder:
    """The decoder's forward over a flat batch of tokens.

    ``forward(input_ids, positions, attn_metadata, kv_caches)`` runs every
    layer; ``kv_caches[i]`` is layer i's ``[2, num_blocks, block_size, Hkv,
    D]`` cache and ``attn_metadata`` the backend metadata of the batch (its
    slot mapping says where each token's K/V is written).  Positions lie
    below ``max_position`` (the rotary table's length; the kernel flags and
    skips a token beyond it).  Returns the final normalised hidden states
    ``[T, hidden]``; :meth:`compute_logits` maps selected rows to float32
    logits."""

    def __init__(self, cfg: DecoderConfig, weights: dict[str, torch.Tensor], *, max_position: int = 32768):
        self.cfg = cfg
        self.w = weights
        dev = weights["embed"].device
        self.rope = RotaryEmbedding(cfg.head_dim, cfg.rope_theta, max_position, dev)
        self.layer_names = [f"model.layers.{i}.self_attn.attn" for i in range(cfg.num_layers)]
        self.attn = [BeamAttentionImpl(cfg.num_heads, cfg.head_dim, 1.0 / math.sqrt(cfg.head_dim),
                                       cfg.num_kv_heads, None, None, "auto")
                     for _ in range(cfg.num_layers)]

    @property
    def device(self) -> torch.device:
        return self.w["embed"].device

    def forward(self, input_ids: torch.Tensor, positions: torch.Tensor, attn_metadata,
                kv_caches) -> torch.Tensor:
        cfg, w, eps = self.cfg, self.w, self.cfg.rms_eps
        T = input_ids.shape[0]
        slots = attn_metadata.slot_mapping if attn_metadata is not None else None
        status = attn_metadata.status if attn_metadata is not None else None
        h = w["embed"][input_ids]  # the residual stream
        x = ops.rms_norm(h, w["layers.0.input_norm"], eps)
        mlp = None
        for i in range(cfg.num_layers):
            p = f"layers.{i}."
            if i:
                x = ops.rms_norm(mlp, w[p + "input_norm"], eps, residual=h, out=x)
            qkv = _linear(x, w[p + "qkv"])
            k_cache, v_cache = ops.split_kv_cache(kv_caches[i])
            q = ops.qk_norm_rope_cache(qkv, positions, self.rope.cos, self.rope.sin, w[p + "q_norm"],
                                       w[p + "k_norm"], k_cache, v_cache, slots, num_q_heads=cfg.num_heads,
                                       num_kv_heads=cfg.num_kv_heads, head_dim=cfg.head_dim, eps=eps,
                                       status=status)
            attn = torch.empty_like(q)
            self.attn[i].forward(None, q, None, None, kv_caches[i], attn_metadata, output=attn)
            x = ops.rms_norm(_linear(attn.view(T, cfg.q_size), w[p + "o"]), w[p + "post_norm"], eps,
                             residual=h, out=x)
            mlp = _linear(_swiglu(x, w[p + "gate_up"]), w[p + "down"])
        return ops.rms_norm(mlp, w["final_norm"], eps, residual=h)

    def compute_logits(self, hidden: torch.Tensor) -> torch.Tensor:
        # the model type's values on either path: scores and their ties do not
        # depend on how many rows share the step
        w = self.w["lm_head"]
        if _plain(hidden, w) and _own_linear(hidden, w):
            return ops.linear(hidden, w, out_f32=True, rounded=True)
        return F.linear(hidden, w).float()
