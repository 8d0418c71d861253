"""hy_paged_prefill through the C ABI with query and output rows off 16-byte
boundaries: the same bits as with aligned rows, for whole tiles, a chunk that
ends inside a tile, split key ranges, and GQA groups 1, 4 and 16. And ticks of
GQA groups 1 and 2 whose waves end far apart."""

import math

import pytest
import torch

from test_prefill_ring import FAR

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


@pytest.mark.parametrize("group,cache,q_lens", FAR)
def test_waves_that_end_tiles_apart(group, cache, q_lens):
    """Few heads a group: a workgroup's waves span up to 256 tokens, and an early
    one's last V block must not be gone when it multiplies it."""
    hkv = 8
    g = torch.Generator(device="cuda").manual_seed(group + sum(q_lens))
    m = PagedKVCacheManager(1, hkv, 128, 16_384, 128, len(cache), torch.bfloat16, "cuda",
                            num_q_heads=hkv * group)
    m.k_cache.normal_(generator=g)
    m.v_cache.normal_(generator=g)
    handles = []
    for c in cache:
        h = m.allocate()
        m.reserve(h, c)
        h.length = c
        handles.append(h)
    batch = m.begin_tick(handles, q_lens)
    q = torch.randn(sum(q_lens), hkv * group, 128, generator=g, device="cuda").to(torch.bfloat16)
    outs = [batch.attend_layer(q, 0).clone() for _ in range(3)]
    row = 0
    for h, c, n in zip(handles, cache, q_lens):
        t = torch.arange(c + n, device="cuda")
        where = torch.tensor(h.pages, device="cuda")[t // 128] * 128 + t % 128
        k = m.k_cache[0, 0][:, where].float().repeat_interleave(group, 0)
        v = m.v_cache[0, 0][:, where].float().repeat_interleave(group, 0)
        late = t[None] > (c + torch.arange(n, device="cuda"))[:, None]
        s = (q[row : row + n].float().transpose(0, 1) @ k.transpose(1, 2).contiguous()) / math.sqrt(128)
        want = (torch.softmax(s.masked_fill(late, -math.inf), -1) @ v).transpose(0, 1)
        for out in outs:
            got = out[row : row + n].float()
            # row by row: a wave holds 32 of them
            err = (got - want).norm(dim=-1) / want.norm(dim=-1)
            assert err.max() < 3e-2, float(err.max())  # bf16 probabilities and output
        row += n
    assert all(torch.equal(o.view(torch.int16), outs[0].view(torch.int16)) for o in outs)
