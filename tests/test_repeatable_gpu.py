"""The same inputs give the same bits: kernels whose waits or order were wrong
show as rounding that changes from run to run."""
import pytest
import torch

from llm_mcp_amd import ops
from llm_mcp_amd.engine.engine import EngineConfig, LLMEngine
from llm_mcp_amd.models import config as mc

pytestmark = pytest.mark.gpu


def _bits(model, dtype="bfloat16"):
    cfg = mc.resolve(model)
    g = torch.Generator().manual_seed(1)
    toks = [torch.randint(0, 1000, (n,), generator=g).tolist() for n in (70, 33, 150)]
    first = None
    for _ in range(4):
        e = LLMEngine(EngineConfig(model=model, max_num_seqs=3, max_batched_tokens=512,
                                   mixed_prefill_tokens=0, max_model_len=256, kv_cache_tokens=512,
                                   use_graphs=False, prefix_cache=False, dtype=dtype), device="cuda",
                      model_cfg=cfg)
        out = [e.feed([(i + 1, t[:-8], [0, len(t) - 9]) for i, t in enumerate(toks)])]
        out += [e.feed([(i + 1, [t[k]], [0]) for i, t in enumerate(toks)]) for k in range(-8, 0)]
        out = torch.cat(out)
        assert bool(torch.isfinite(out).all())
        first = out if first is None else first
        assert torch.equal(out, first)


@pytest.mark.parametrize("model", ["llama-3-8b@L2", "zegopel-8b@L3", "zovozen-8b@L2"])
def test_steps_repeat_to_the_bit(model):
    """Prompts and decoded tokens through fresh engines, the kernels of the full widths."""
    ops.native()
    _bits(model)
