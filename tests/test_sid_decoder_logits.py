"""SidDecoder.compute_logits on host weights gives what the torch product gives."""

import pytest
import torch

from vllm_gr_amd.v1.sid_decoder import DecoderConfig, SidDecoder, init_weights


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_logits_on_the_host(dtype):
    cfg = DecoderConfig(num_layers=1, hidden=512, num_heads=4, num_kv_heads=2, ffn=512, vocab=64, dtype=dtype)
    dec = SidDecoder(cfg, init_weights(cfg, 0), max_position=8)
    hidden = torch.randn(5, 512, generator=torch.Generator().manual_seed(0)).to(dtype)
    assert torch.equal(dec.compute_logits(hidden), torch.nn.functional.linear(hidden, dec.w["lm_head"]).float())
