"""hy_paged_prefill through the C ABI with query and output rows off 16-byte
boundaries: the same bits as with aligned rows, for whole tiles, a chunk that
ends inside a tile, split key ranges, and GQA groups 1, 4 and 16."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from hayate_amd import PagedKVCacheManager, _native


def rows(n, heads, shift):
    """(n, heads, 128) bf16 whose rows start `shift` elements into 16 bytes."""
    flat = torch.zeros(n * heads * 130 + 16, dtype=torch.bfloat16, device="cuda")
    if not shift:
        return flat[: n * heads * 128].view(n, heads, 128)
    return flat[shift : shift + n * heads * 130].view(n, heads, 130)[..., :128]


@pytest.mark.parametrize("hq,hkv", [(32, 8), (8, 8), (16, 1)])
@pytest.mark.parametrize("cache,q_len", [(0, 2), (100, 65), (6000, 300)])
@pytest.mark.parametrize("shift", [2, 4])
def test_rows_off_sixteen_bytes(hq, hkv, cache, q_len, shift):
    g = torch.Generator(device="cuda").manual_seed(hq + cache + q_len)
    m = PagedKVCacheManager(1, hkv, 128, 8192, 128, 1, torch.bfloat16, "cuda", num_q_heads=hq)
    m.k_cache.normal_(generator=g)
    m.v_cache.normal_(generator=g)
    h = m.allocate()
    m.reserve(h, cache)
    h.length = cache
    batch = m.begin_tick([h], [q_len])
    plan = batch.plan(hq)
    values = torch.randn(q_len, hq, 128, generator=g, device="cuda").to(torch.bfloat16)
    outs = []
    for s in (0, shift):
        q, out = rows(q_len, hq, s), rows(q_len, hq, s)
        q.copy_(values)
        args = (0, out.stride(0), out.stride(1))
        k_ptr, v_ptr, hs = batch._layer_pools(0)
        stream = torch.cuda.current_stream().cuda_stream
        lib = _native.lib()
        _native.check(lib.hy_paged_prefill(
            q.data_ptr(), 0, q.stride(0), q.stride(1), out.data_ptr(), *args, k_ptr, v_ptr, hs,
            batch._pt_ptr, batch._pt_stride, batch._q_start_ptr, batch._kv_lens_ptr,
            plan.prefill_ptr, plan.n_prefill, plan.n_prefill_slots, plan.prefill_workspace_ptr,
            plan.prefill_workspace_bytes, 1, hq, hkv, 128, 128, 1 / math.sqrt(128), stream),
            "hy_paged_prefill")
        if plan.n_prefill_merge:
            _native.check(lib.hy_paged_prefill_merge(
                out.data_ptr(), *args, batch._q_start_ptr, plan.prefill_merge_ptr,
                plan.n_prefill_merge, plan.n_prefill_slots, plan.prefill_workspace_ptr,
                plan.prefill_workspace_bytes, hq, hkv, 128, stream), "hy_paged_prefill_merge")
        outs.append(out.clone())
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    # against plain fp32 attention of the same pages
    t = torch.arange(cache + q_len, device="cuda")
    pages = torch.tensor(h.pages, device="cuda")
    where = pages[t // 128] * 128 + t % 128
    k, v = m.k_cache[0, 0][:, where].float(), m.v_cache[0, 0][:, where].float()
    mask = t[None] > (cache + torch.arange(q_len, device="cuda"))[:, None]
    grp = hq // hkv
    for head in (0, hq - 1):
        s = (values[:, head].float() @ k[head // grp].T) / math.sqrt(128)
        want = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[head // grp]
        err = (outs[0][:, head].float() - want).norm() / want.norm()
        assert err < 1e-2, float(err)  # bf16 probabilities and output
