"""How a mixed step's attention goes: in two launches, or in one with 2, 4 or 8 waves per (row, kv head, key partition) item (host code only)."""
import pytest
import torch

from distributed_sse_for_llm_response_amd import ops


@pytest.mark.parametrize("rows,hq,hkv,nparts,tiles,waves", [
    (64, 32, 8, 1, 5, 4), (48, 32, 8, 1, 5, 8), (49, 32, 8, 1, 1, 4), (80, 32, 8, 1, 5, 4), (81, 32, 8, 1, 5, 2), (16, 32, 8, 4, 5, 4), (385, 4, 1, 1, 1, 4),
    (64, 16, 8, 1, 5, 0), (64, 8, 8, 1, 5, 0), (0, 32, 8, 1, 5, 0), (64, 32, 8, 1, 0, 0)])
def test_waves(rows, hq, hkv, nparts, tiles, waves):
    ops.load_library(required=True)
    assert torch.ops.dsse.mixed_attention_waves(rows, hq, hkv, nparts, tiles) == waves


@pytest.mark.parametrize("key,value,waves", [("attn_mixed", 0, 0), ("flash_hg", 2, 0), ("attn_kwv", 8, 8), ("attn_kwv", 1, 2)])
def test_keys(monkeypatch, key, value, waves):
    ops.load_library(required=True)
    monkeypatch.setenv("DSSE_KERNEL_CFG", ops.kernel_cfg_env(**{key: value}))
    ops.refresh_env()
    try:
        assert torch.ops.dsse.mixed_attention_waves(64, 32, 8, 1, 5) == waves
    finally:
        monkeypatch.undo()
        ops.refresh_env()
