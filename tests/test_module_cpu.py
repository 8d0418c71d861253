"""Host-side pieces of the attention module and model that run without a
GPU: the fused q/k/v projection and the checkpoint name map."""

import pytest
import torch

from hayate_amd import linear
from hayate_amd.attention import GroupedQueryAttention, _norm_eps
from hayate_amd.model import (FeedForward, Qwen3Config, Qwen3Model, TransformerBlock,
                              qwen_weight_map)


def test_fused_qkv_projection_views_one_gemm():
    torch.manual_seed(0)
    mod = GroupedQueryAttention(64, 4, 2, 16, dtype=torch.float32)
    x = torch.randn(3, 5, 64)
    q, k, v = mod.project_qkv(x)
    torch.testing.assert_close(q, mod.q_proj(x).view(3, 5, 4, 16))
    torch.testing.assert_close(k, mod.k_proj(x).view(3, 5, 2, 16))
    torch.testing.assert_close(v, mod.v_proj(x).view(3, 5, 2, 16))
    # views of one buffer: no split copies, rows 16-byte aligned
    base = q.untyped_storage().data_ptr()
    assert k.untyped_storage().data_ptr() == base == v.untyped_storage().data_ptr()
    assert q.stride() == (5 * 128, 128, 16, 1) and k.stride(1) == 128
    # the fused weight follows in-place updates of the parameters
    with torch.no_grad():
        mod.k_proj.weight.mul_(2)
    _, k2, _ = mod.project_qkv(x)
    torch.testing.assert_close(k2, 2 * k)


def test_fused_qkv_weight_is_the_only_copy():
    """q/k/v_proj.weight are views of the one fused buffer (no second copy of
    the projection weights); in-place loads write through; the buffer is
    rebuilt, and the rebuild counter advances, only when a parameter is
    replaced rather than updated, and the first build under inference_mode
    still leaves trainable parameters."""
    import hayate_amd.attention as A

    torch.manual_seed(1)
    mod = GroupedQueryAttention(64, 4, 2, 16, dtype=torch.float32)
    x = torch.randn(2, 3, 64)
    ref = [lin.weight.detach().clone() for lin in (mod.q_proj, mod.k_proj, mod.v_proj)]
    n0 = A.qkv_rebuilds
    with torch.inference_mode():
        f = mod.fused_qkv_weight()
    assert A.qkv_rebuilds == n0 + 1
    assert torch.equal(f, torch.cat(ref))
    base = f.untyped_storage().data_ptr()
    for lin in (mod.q_proj, mod.k_proj, mod.v_proj):
        assert lin.weight.untyped_storage().data_ptr() == base
        assert isinstance(lin.weight, torch.nn.Parameter) and lin.weight.requires_grad
        assert not lin.weight.is_inference()
    assert mod.q_proj(x).requires_grad
    # a state-dict load copies into the views: same buffer, new values
    sd = {k: (2 * v if k.endswith("proj.weight") else v) for k, v in mod.state_dict().items()}
    mod.load_state_dict(sd)
    assert mod.fused_qkv_weight() is f and A.qkv_rebuilds == n0 + 1
    assert torch.equal(f, 2 * torch.cat(ref))
    # replacing a parameter rebuilds the buffer from the current weights
    mod.v_proj.weight = torch.nn.Parameter(torch.zeros_like(mod.v_proj.weight))
    f2 = mod.fused_qkv_weight()
    assert f2 is not f and A.qkv_rebuilds == n0 + 2
    assert torch.equal(f2[-32:], torch.zeros(32, 64)) and torch.equal(f2[:64], 2 * ref[0])


def test_checkpoint_name_map_covers_every_parameter():
    cfg = Qwen3Config(vocab_size=64, hidden_size=32, num_layers=2, num_heads=4,
                      num_kv_groups=2, head_dim=8, intermediate_size=48)
    with torch.device("meta"):
        model = Qwen3Model(cfg)
    names = qwen_weight_map(model)
    params = {id(p) for p in model.parameters()}
    assert {id(p) for p in names.values()} == params
    assert "model.layers.1.self_attn.q_norm.weight" in names
    assert len(names) == 3 + 11 * 2


def test_stop_ids_from_generation_config_and_tokenizer(tmp_path):
    """End-of-generation ids (engine.py:112-129 of the reference): the
    checkpoint's generation_config.json eos id or list, plus the
    tokenizer's eos id; a missing or broken config leaves the tokenizer's."""
    import json
    from types import SimpleNamespace

    from hayate_amd.engine import _stop_token_ids

    tok = SimpleNamespace(eos_token_id=7)
    (tmp_path / "generation_config.json").write_text(json.dumps({"eos_token_id": [1, 2]}))
    assert _stop_token_ids(str(tmp_path), tok) == {1, 2, 7}
    (tmp_path / "generation_config.json").write_text(json.dumps({"eos_token_id": 3}))
    assert _stop_token_ids(str(tmp_path), None) == {3}
    (tmp_path / "generation_config.json").write_text("{not json")
    assert _stop_token_ids(str(tmp_path), tok) == {7}
    assert _stop_token_ids(None, tok) == {7}
    assert _stop_token_ids(str(tmp_path / "missing"), None) == set()


@pytest.mark.parametrize("eps", [None, 0.0, 1e-6, 0.25])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32, torch.float64])
def test_norm_epsilon_is_the_modules(dtype, eps):
    """Rows small enough for the epsilon to decide the result."""
    g = torch.Generator().manual_seed(0)
    norm = torch.nn.RMSNorm(256, eps=eps, dtype=dtype)
    x = (torch.randn(8, 256, generator=g) * 1e-3).to(dtype)
    e = _norm_eps(norm, dtype)
    want = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + e)
    # one rounding of the result; fp32 sums add far less
    tol = torch.finfo(dtype).eps if dtype is not torch.float64 else 1e-12
    assert ((norm(x).double() - want).norm() / want.norm()) < max(tol, 1e-6 * (tol > 1e-12))


@pytest.fixture
def plain_block(monkeypatch):
    """A block whose weights the fused paths would take if they were on the GPU."""
    monkeypatch.setattr(linear, "_plain_weight", lambda w, index, dim: True)
    cfg = Qwen3Config(hidden_size=64, num_heads=4, num_kv_groups=2, head_dim=16,
                      intermediate_size=96, vocab_size=50, num_layers=1)
    block = TransformerBlock(cfg)
    x = torch.zeros(1, 3, 64, dtype=torch.bfloat16)
    assert block._plain_weights(x) is not None
    return block, x


def _keep(f):
    return lambda *a, **k: f(*a, **k)


@pytest.mark.parametrize("owner,name", [
    (torch.nn.Linear, "forward"), (torch.nn.Linear, "__call__"), (torch.nn.RMSNorm, "forward"),
    (torch.nn.RMSNorm, "__call__"), (torch.nn.Module, "__call__"),
    (torch.nn.functional, "linear"), (torch.nn.functional, "rms_norm"),
    (torch.nn.functional, "silu"), (FeedForward, "forward"), (GroupedQueryAttention, "forward"),
    (GroupedQueryAttention, "project_qkv")])
def test_replaced_functions_stay_in_charge(plain_block, monkeypatch, owner, name):
    block, x = plain_block
    with monkeypatch.context() as m:
        m.setattr(owner, name, _keep(getattr(owner, name)), raising=True)
        assert block._plain_weights(x) is None
    assert block._plain_weights(x) is not None


@pytest.mark.parametrize("path,name", [
    ("self_attn", "forward"), ("self_attn", "project_qkv"), ("mlp", "forward"),
    ("mlp.up_proj", "forward"), ("self_attn.o_proj", "forward"), ("input_layernorm", "forward"),
    ("post_attention_layernorm", "forward")])
def test_an_instances_own_method_stays_in_charge(plain_block, path, name):
    block, x = plain_block
    m = block.get_submodule(path)
    setattr(m, name, _keep(getattr(m, name)))
    assert block._plain_weights(x) is None
    delattr(m, name)
    assert block._plain_weights(x) is not None
    m.compile(backend="eager")
    assert block._plain_weights(x) is None


def test_functions_replaced_before_the_import_stay_in_charge():
    code = """
import torch
F = torch.nn.functional
real, torch.nn.Linear.forward = torch.nn.Linear.forward, lambda self, x: real(self, x)
from hayate_amd import linear
assert not linear._unpatched()
torch.nn.Linear.forward = real
"""
    import os
    import subprocess
    import sys

    env = dict(os.environ, PYTHONPATH=os.pathsep.join(sys.path))
    subprocess.run([sys.executable, "-c", code], check=True, env=env, timeout=300)


def test_a_default_device_watches_nothing():
    from torch.overrides import TorchFunctionMode

    class Watcher(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert linear.unwatched()
    for device in ("cpu", "meta", "cuda"):
        with torch.device(device):
            assert linear.unwatched()
            with Watcher():
                assert not linear.unwatched()
            with torch.device("cpu"):
                assert linear.unwatched()
        with Watcher(), torch.device(device):
            assert not linear.unwatched()
        try:
            torch.set_default_device(device)
            assert linear.unwatched()
        finally:
            torch.set_default_device(None)
    assert linear.unwatched()
