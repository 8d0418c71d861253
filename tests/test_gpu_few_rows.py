"""The few-row products (csrc/skinny.hip) and the block that uses them.

The products against float64 at the sizes where the kernels change shape:
row counts around the 16-row tiles, column counts that leave a workgroup a
partial tile or nothing, and K around the waves' step counts. The result is
rounded to bf16 once (at most 2^-8 of each value) and, with the norm, each
x * weight before the sums: those errors are independent, so a sum of them
is below 2^-8 of the root of its terms' sum of squares (three standard
deviations), of which a sum that cancels is only a part.
"""

import pytest
import torch

from gpu_util import say

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from hayate_amd import PagedKVCacheManager, linear
    from hayate_amd.model import Qwen3Config, Qwen3Model, TransformerBlock, init_synthetic_weights

DEV = "cuda"


def bf16(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(torch.bfloat16)


def rel(a, b):
    return float((a.double() - b).norm() / b.norm())


def off(y, h, w):
    """Error of y = h w^T over its bound's unit (see the top)."""
    exact = h.double() @ w.double().T
    terms = h.double().square() @ w.double().T.square()
    return float((y.double() - exact).norm() / (exact.norm() + terms.sqrt().norm()))


def norm64(x, w, eps):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


@pytest.mark.parametrize("k", [512, 576, 1024, 2048, 2560, 2624, 3072, 3136, 4096])
@pytest.mark.parametrize("m,n", [(1, 1), (1, 6144), (15, 300), (16, 9728), (17, 40), (32, 4111)])
def test_norm_linear(k, m, n):
    if not linear.norm_fits(k, m):
        pytest.skip("refused: 32 rows of more than 3072")
    g = torch.Generator(device=DEV).manual_seed(k + m + n)
    wide = bf16(g, m, k + 8, std=3.0)  # rows with a stride of their own
    x, w, u = wide[:, :k], bf16(g, n, k, std=k**-0.5), bf16(g, n, k, std=k**-0.5)
    nw = 1 + bf16(g, k, std=0.2)
    h = norm64(x, nw, 1e-3)
    plain = linear.norm_linear(x, None, 0.0, w)
    normed = linear.norm_linear(x, nw, 1e-3, w)
    gated = linear.norm_linear(x, nw, 1e-3, w, u)
    gate = h @ w.double().T
    assert off(plain, x, w) < 2**-8
    assert off(normed, h, w) < 2**-8
    # silu' is at most 1.1 and the two sums' errors meet in a product
    up = h @ u.double().T
    unit = (h.square() @ w.double().T.square()).sqrt()
    err = (gated.double() - gate * torch.sigmoid(gate) * up).norm()
    assert err < 2**-8 * 1.1 * ((unit + gate.abs()) * (unit + up.abs())).norm()
    # rows do not depend on how many others there are
    if m in (15, 17):
        tile = slice(0, 16) if m > 16 else slice(0, m)
        again = linear.norm_linear(x[tile], nw, 1e-3, w)
        assert off(again, h[tile], w) < 2**-8


@pytest.mark.parametrize("k", [128, 1024, 1152, 4096, 9728])
@pytest.mark.parametrize("m,n", [(1, 1), (1, 2560), (16, 2049), (17, 4100), (32, 2560)])
def test_linear_add(k, m, n):
    g = torch.Generator(device=DEV).manual_seed(k + m + n)
    x, w = bf16(g, m, k), bf16(g, n, k, std=k**-0.5)
    r = bf16(g, m, n + 5)[:, :n]
    exact = x.double() @ w.double().T
    assert rel(linear.linear_add(x, w), exact) < 2**-8  # one rounding of fp32 sums
    assert rel(linear.linear_add(x, w, r), exact + r.double()) < 2**-8


def test_infinite_weights_stay_in_their_columns():
    """An infinite weight makes its own column infinite or NaN, no other,
    also where a wave's window overlaps its neighbour's (K = 576)."""
    g = torch.Generator(device=DEV).manual_seed(1)
    x, w = bf16(g, 5, 576), bf16(g, 64, 576)
    w[7, 570] = float("inf")
    y = linear.norm_linear(x, None, 0.0, w)
    want = x.float() @ w.float().T
    assert torch.equal(torch.isinf(y), torch.isinf(want))
    assert not torch.isnan(y).any()


@pytest.mark.parametrize("at", [0, 447, 448, 470, 575])
def test_infinite_norm_weights(at):
    """An infinite norm weight gives the infinities it gives torch's norm and
    product, no NaN, also where the waves' windows overlap (from 448 on)."""
    g = torch.Generator(device=DEV).manual_seed(2)
    x, w, nw = bf16(g, 5, 576), bf16(g, 64, 576), 1 + bf16(g, 576, std=0.1)
    nw[at] = float("inf")
    x[:, at], w[:, at] = x[:, at].abs() + 0.1, w[:, at].abs() + 0.1
    y = linear.norm_linear(x, nw, 1e-6, w)
    assert (y == float("inf")).all()


def tick(cfg, q_lens, layers=1):
    m = PagedKVCacheManager(layers, cfg.num_kv_groups, cfg.head_dim, 32_768, 128, len(q_lens),
                            torch.bfloat16, DEV, num_q_heads=cfg.num_heads)
    g = torch.Generator(device=DEV).manual_seed(5)
    m.k_cache.normal_(generator=g)
    m.v_cache.normal_(generator=g)
    handles = []
    for i in range(len(q_lens)):
        h = m.allocate()
        m.reserve(h, 100 + 37 * i)
        h.length = 100 + 37 * i
        handles.append(h)
    return m, m.begin_tick(handles, q_lens)


@pytest.mark.parametrize("q_lens", [[1], [1] * 20, [5, 1, 1], [1] * 32, [33]])
def test_block_equals_its_modules(q_lens, monkeypatch):
    """The fused block against the same block with a hook on its MLP (which
    puts the modules back in charge): both within the block's rounding of
    each other; 33 rows take the tile products instead of the few-row ones."""
    say(f"[block, q_lens {q_lens}]")
    cfg = Qwen3Config()
    torch.manual_seed(3)
    with torch.device(DEV):
        block = TransformerBlock(cfg)
    with torch.no_grad():
        for p in block.parameters():
            if p.dim() == 2:
                p.normal_(std=p.shape[1] ** -0.5)
    x = torch.randn(1, sum(q_lens), cfg.hidden_size, device=DEV).to(torch.bfloat16)
    from hayate_amd.rope import compute_rope_params

    cos, sin = compute_rope_params(128, 1_000_000, 4096, device=DEV)
    used = []
    real = linear.linear_add
    monkeypatch.setattr(linear, "linear_add", lambda *a: (used.append(1), real(*a))[1])
    tiles = []
    tile = linear.tile_linear
    monkeypatch.setattr(linear, "tile_linear", lambda *a, **k: (tiles.append(1), tile(*a, **k))[1])
    m, batch = tick(cfg, q_lens)
    with torch.inference_mode():
        fused = block(x, cos, sin, None, None, None, None, batch, 0)[0]
        assert len(used) == (2 if sum(q_lens) <= 32 else 0)
        k1 = m.k_cache.clone()
        hook = block.mlp.register_forward_hook(lambda *a: None)
        plain = block(x, cos, sin, None, None, None, None, batch, 0)[0]
        hook.remove()
        assert len(used) == (2 if sum(q_lens) <= 32 else 0)
        assert len(tiles) == (0 if sum(q_lens) <= 32 else 3)
    e = rel(fused, plain.double())
    say(f"  relative difference {e:.2e}")
    # five rounded products on either side, each 2^-8 of a part of the sum
    assert e < 2**-7
    assert rel(k1, m.k_cache.double()) < 2**-8


def test_gradients_and_hooks_keep_the_modules():
    """Nothing fused where it could be seen: gradients enabled, a hook, a bias,
    other types, autocast, a dispatch mode."""
    x = torch.randn(2, 1, 2560, device=DEV).to(torch.bfloat16)
    lin = torch.nn.Linear(2560, 64, bias=False, dtype=torch.bfloat16, device=DEV)
    norm = torch.nn.RMSNorm(2560, dtype=torch.bfloat16, device=DEV)
    assert not linear.few_rows(x)  # gradients enabled
    with torch.no_grad():
        assert linear.few_rows(x) and linear.plain(x, norms=(norm,), linears=(lin,))
        assert not linear.few_rows(x.float()) and not linear.few_rows(x.cpu())
        assert not linear.few_rows(x.expand(2, 17, 2560))
        with torch.autocast("cuda", dtype=torch.float16):
            assert not linear.few_rows(x)
        from torch.utils.flop_counter import FlopCounterMode

        with FlopCounterMode(display=False):
            assert not linear.few_rows(x)
        assert not torch.func.vmap(lambda r: torch.tensor(linear.few_rows(r)), out_dims=None)(x)
        h = lin.register_forward_pre_hook(lambda *a: None)
        assert not linear.plain(x, linears=(lin,))
        h.remove()
        assert not linear.plain(x, linears=(torch.nn.Linear(2560, 8, dtype=torch.bfloat16,
                                                            device=DEV),))
        assert not linear.plain(x, norms=(torch.nn.RMSNorm(2560, device=DEV),))


def test_head_of_a_tick():
    """The final norm and head against the modules' own calls."""
    cfg = Qwen3Config(vocab_size=1000, num_layers=1)
    with torch.device(DEV):
        model = Qwen3Model(cfg)
    init_synthetic_weights(model, 2)
    ids = torch.arange(40, device=DEV).view(1, 40)
    _, batch = tick(cfg, [38, 1, 1])
    with torch.inference_mode():
        logits = model(ids, paged_cache=batch)[0]
        hook = model.norm.register_forward_hook(lambda *a: None)
        plain = model(ids, paged_cache=batch)[0]
        hook.remove()
    assert logits.shape == plain.shape == (3, 1, 1000)
    assert rel(logits, plain.double()) < 2**-7


@pytest.mark.parametrize("tokens", [3, 40])
def test_norms_without_an_epsilon(tokens):
    """eps=None is the module's default also on the fused paths: rows of rms
    0.05, which another epsilon would change by more than the roundings."""
    cfg = Qwen3Config(hidden_size=1024, num_heads=8, num_kv_groups=2, intermediate_size=2048,
                      vocab_size=1000, num_layers=1, rms_norm_eps=None)
    with torch.device(DEV):
        model = Qwen3Model(cfg)
    init_synthetic_weights(model, 4)
    with torch.no_grad():
        model.embed_tokens.weight.normal_(std=0.05)
        for w in (model.layers[0].self_attn.o_proj, model.layers[0].mlp.down_proj):
            w.weight.mul_(0.01)  # the rows stay small up to the head
    ids = torch.arange(tokens, device=DEV).view(1, tokens)
    _, batch = tick(cfg, [tokens - 2, 1, 1])
    with torch.inference_mode():
        logits = model(ids, paged_cache=batch)[0]
        hooks = [m.register_forward_hook(lambda *a: None)
                 for m in (model.norm, model.layers[0].mlp)]
        plain = model(ids, paged_cache=batch)[0]
        for h in hooks:
            h.remove()
    assert rel(logits, plain.double()) < 2**-7


@pytest.mark.parametrize("device", ["cpu", "cuda", "meta"])
@pytest.mark.parametrize("tokens", [4, 70])
def test_a_default_device_keeps_the_kernels(device, tokens, monkeypatch):
    """Logits and tokens under torch.device(...): the same bits by the same
    kernels."""
    from hayate_amd import _native
    from hayate_amd.sampler import sample_batch

    cfg = Qwen3Config(hidden_size=512, num_heads=8, num_kv_groups=2, intermediate_size=1024,
                      vocab_size=1000, num_layers=1)
    with torch.device(DEV):
        model = Qwen3Model(cfg)
    init_synthetic_weights(model, 6)
    model.initialize_rope(DEV)
    ids = torch.arange(tokens, device=DEV).view(1, tokens)

    def call():
        _, batch = tick(cfg, [tokens - 2, 1, 1])
        batch.plan(cfg.num_heads)
        used = []
        for name in ("norm_linear", "linear_add", "row_norm", "tile_linear"):
            real = getattr(linear, name)
            monkeypatch.setattr(linear, name,
                                lambda *a, f=real, n=name, **k: (used.append(n), f(*a, **k))[1])
        with torch.inference_mode():
            logits = model(ids, paged_cache=batch)[0]
            tokens_ = sample_batch(logits[:, 0], [0.0, 0.7, 1.0], [None, 20, None],
                                   [None, None, 0.9], torch.Generator(device=DEV).manual_seed(3))
        monkeypatch.undo()
        return logits, tokens_, used

    want = call()
    assert set(want[2]) == ({"norm_linear", "linear_add"} if tokens < 32 else
                            {"row_norm", "tile_linear", "norm_linear"})
    with torch.device(device):
        got = call()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and got[2] == want[2]
