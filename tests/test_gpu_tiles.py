"""The prompt-row products (csrc/tiles.hip) and the block that uses them.

Against float64: row and column counts that leave the last tile one row, all but
one, or a fraction of a fragment, and K of one step, of fewer steps than the
ring has stages and of many, on the small tiles; and every tile shape, split and
whole, at sizes that test_tile_plan.py holds the plan to. The result is rounded
to bf16 once (at most 2^-8 of each value); the fp32 sums add far less.
"""

import pytest
import torch

from gpu_util import say
from test_tile_plan import SIZES

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from hayate_amd import PagedKVCacheManager, _native, linear
    from hayate_amd.model import Qwen3Config, TransformerBlock

DEV = "cuda"


def bf16(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(torch.bfloat16)


def rel(y, exact):
    return float((y.double() - exact).norm() / exact.norm())


ROWS = [1, 33, 64, 65, 127, 129, 256, 300, 513, 2064]


@pytest.mark.parametrize("k", [64, 192, 256, 1024, 2560, 9728])
@pytest.mark.parametrize("n", [4, 100, 160, 2560])
@pytest.mark.parametrize("m", ROWS)
def test_linear_add(m, n, k):
    say(f"tiles add {m} x {n} x {k}")
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    wide = bf16(g, m, k + 8)  # rows with strides of their own
    x, w = wide[:, :k], bf16(g, n, k + 16, std=k**-0.5)[:, :k]
    r = bf16(g, m, n + 4)[:, :n]
    exact = x.double() @ w.double().T
    assert rel(linear.tile_linear(x, w), exact) < 2**-8
    assert rel(linear.tile_linear(x, w, residual=r), exact + r.double()) < 2**-8


@pytest.mark.parametrize("n,k", [(4, 64), (76, 256), (80, 128), (3072, 1024), (9728, 2560)])
@pytest.mark.parametrize("m", ROWS)
def test_gated_linear(m, n, k):
    say(f"tiles gated {m} x {n} x {k}")
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x, w, u = bf16(g, m, k), bf16(g, n, k, std=k**-0.5), bf16(g, n, k, std=k**-0.5)
    gate = x.double() @ w.double().T
    exact = gate * torch.sigmoid(gate) * (x.double() @ u.double().T)
    assert rel(linear.tile_linear(x, w, u), exact) < 2**-8


@pytest.mark.parametrize("gated,m,n,k", SIZES)
def test_every_plan(gated, m, n, k):
    say(f"tiles plan {m} x {n} x {k}, gated {gated}")
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x, w = bf16(g, m, k), bf16(g, n, k, std=k**-0.5)
    if gated:
        u = bf16(g, n, k, std=k**-0.5)
        gate = x.double() @ w.double().T
        exact = gate * torch.sigmoid(gate) * (x.double() @ u.double().T)
        assert rel(linear.tile_linear(x, w, u), exact) < 2**-8
    else:
        r = bf16(g, m, n)
        exact = x.double() @ w.double().T + r.double()
        y = linear.tile_linear(x, w, residual=r)
        assert rel(y, exact) < 2**-8
        # no single output is far off, which the norm would not show: the rounding,
        # and fp32 sums of up to 5,824 terms (k 2^-24 sum|x w| < 2^-6 of them)
        assert ((y.double() - exact).abs() <= 2**-8 * exact.abs() + 2**-6).all()


@pytest.mark.parametrize("k", [8, 504, 512, 520, 2560, 3592, 4096])
@pytest.mark.parametrize("m", [1, 33, 4096, 4099])
def test_row_norm(m, k):
    """fp32 sums of k squares, one rounding to bf16 (8 significant bits)."""
    g = torch.Generator(device=DEV).manual_seed(m + k)
    wide = bf16(g, m, k + 8, std=3.0)
    x, w = wide[:, :k], 1 + bf16(g, k, std=0.2)
    exact = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-3) * w.double()
    y = linear.row_norm(x, w, 1e-3).double()
    assert ((y - exact).abs() <= (2**-8 + 1e-5) * exact.abs() + 1e-30).all()


def test_nothing_outside_the_result_is_written():
    g = torch.Generator(device=DEV).manual_seed(3)
    for m, n, k, gated in ((300, 2560, 9728, 0), (65, 100, 256, 0), (129, 76, 256, 1)):
        x, w, u = bf16(g, m, k), bf16(g, n, k), bf16(g, n, k)
        lib = _native.lib()
        size = lib.hy_linear_tiles_workspace_bytes(m, n, k, gated)
        work = torch.full((size + 64,), 7, dtype=torch.uint8, device=DEV)
        y = torch.full((m + 2, n + 8), 5.0, dtype=torch.bfloat16, device=DEV)
        inner = y[1:-1, 4:-4]
        _native.check(lib.hy_linear_tiles(
            x.data_ptr(), k, m, k, w.data_ptr(), u.data_ptr() if gated else None, k, n, None, 0,
            inner.data_ptr(), n + 8, work.data_ptr(), size,
            torch.cuda.current_stream().cuda_stream), "hy_linear_tiles")
        assert (work[size:] == 7).all()
        y[1:-1, 4:-4] = 5.0
        assert (y == 5.0).all()


def test_infinities_and_nans_stay_in_their_rows():
    g = torch.Generator(device=DEV).manual_seed(4)
    x, w, u = bf16(g, 70, 256), bf16(g, 160, 256), bf16(g, 160, 256)
    x[3, 5], x[69, 255] = float("inf"), float("nan")
    want = torch.nn.functional.silu(x.float() @ w.float().T) * (x.float() @ u.float().T)
    got = linear.tile_linear(x, w, u).float()
    rows = [i for i in range(70) if i not in (3, 69)]
    assert rel(got[rows], want[rows].double()) < 2**-8
    assert got[69].isnan().all() and torch.equal(got[3].isnan(), want[3].isnan())


@pytest.mark.parametrize("lens", [(40,), (256, 1, 44), (600,)])
def test_block_equals_its_modules(lens, monkeypatch):
    """The fused block against the modules' own calls (taken when a hook is
    there), both bf16: each output is within the roundings of the fused one's
    fewer intermediates."""
    used = []
    for name in ("tile_linear", "row_norm"):
        monkeypatch.setattr(linear, name, lambda *a, f=getattr(linear, name), n=name, **k:
                            (used.append(n), f(*a, **k))[1])
    cfg = Qwen3Config(hidden_size=1024, num_heads=16, num_kv_groups=8, intermediate_size=3072)
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    with torch.device(DEV):
        block = TransformerBlock(cfg).eval()
    with torch.no_grad():
        for p in block.parameters():
            p.copy_(bf16(g, *p.shape, std=p.shape[-1] ** -0.5) if p.dim() == 2 else 1 + bf16(g, *p.shape, std=0.1))
    n = sum(lens)
    x = bf16(g, 1, n, 1024)
    cos = torch.randn(4096, 128, generator=g, device=DEV)
    sin = torch.randn(4096, 128, generator=g, device=DEV)
    outs = []
    for hooked in (False, True):
        mgr = PagedKVCacheManager(1, 8, 128, 8192, 128, 8, torch.bfloat16, DEV, num_q_heads=16)
        handles = [mgr.allocate() for _ in lens]
        batch = mgr.begin_tick(handles, list(lens))
        hook = block.mlp.register_forward_hook(lambda *a: None) if hooked else None
        with torch.no_grad():
            outs.append(block(x, cos, sin, None, None, None, None, batch, 0)[0])
        if hook:
            hook.remove()
        # by the fused block only
        assert used.count("tile_linear") == 3 and used.count("row_norm") == 2
    # five roundings of 2^-8 in a chain of products at most
    assert rel(outs[0], outs[1].double()) < 5 * 2**-8


@pytest.mark.parametrize("rows,tiles", [(33, 3), (11_264, 3), (11_265, 1), (13_000, 1)])
def test_many_outputs_leave_the_residual_products_to_the_library(rows, tiles, monkeypatch):
    """On both sides of the line (rows x 512 outputs): how many products take the
    tiles, and the block against its modules."""
    cfg = Qwen3Config(hidden_size=512, num_heads=8, num_kv_groups=8, intermediate_size=512)
    g = torch.Generator(device=DEV).manual_seed(rows)
    with torch.device(DEV):
        block = TransformerBlock(cfg).eval()
    with torch.no_grad():
        for p in block.parameters():
            p.copy_(bf16(g, *p.shape, std=p.shape[-1] ** -0.5) if p.dim() == 2 else 1 + bf16(g, *p.shape, std=0.1))
    lens = [512] * (rows // 512) + [rows % 512] * (rows % 512 > 0)
    x = bf16(g, 1, rows, 512)
    cos = torch.randn(1024, 128, generator=g, device=DEV)
    sin = torch.randn(1024, 128, generator=g, device=DEV)
    used = []
    real = linear.tile_linear
    monkeypatch.setattr(linear, "tile_linear", lambda *a, **k: (used.append(1), real(*a, **k))[1])
    outs = []
    for hooked in (False, True):
        mgr = PagedKVCacheManager(1, 8, 128, 32_768, 128, len(lens), torch.bfloat16, DEV, num_q_heads=8)
        batch = mgr.begin_tick([mgr.allocate() for _ in lens], lens)
        hook = block.mlp.register_forward_hook(lambda *a: None) if hooked else None
        before = x.clone()
        with torch.no_grad():
            outs.append(block(x, cos, sin, None, None, None, None, batch, 0)[0])
        if hook:
            hook.remove()
        assert torch.equal(x, before)
    assert len(used) == tiles
    assert rel(outs[0], outs[1].double()) < 5 * 2**-8  # five roundings in a chain at most
