"""The store fused into a packed prefill (nva_store_prefill, Attention.forward without a cached
prefix): caches bit-identical to store_kvcache and outputs equal to flash_attn_varlen_func on
the same inputs, over the grids and head shapes that fuse, those that do not, and rows that no
work item carries (past cu_seqlens_q's end, past max_seqlen_q)."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    from nanovllm_amd import _capi
    _capi.load()
    return torch.device("cuda:0")


def _case(dev, lens, nh, nkv, d, seed):
    from nanovllm_amd import workloads as W
    return W.make_prefill_case(lens, nh, nkv, sum(-(-n // 256) for n in lens) + 2, head_dim=d, seed=seed, bulk_device=dev)


def _forward(c, k, v, max_q=None):
    import nanovllm_amd as nva
    layer = nva.Attention(c.num_heads, c.head_dim, c.scale, c.num_kv_heads)
    layer.k_cache, layer.v_cache = c.k_cache.clone(), c.v_cache.clone()
    nva.set_context(True, c.cu_seqlens_q, c.cu_seqlens_k, max_q or c.max_seqlen_q, c.max_seqlen_k, c.slot_mapping)
    try:
        o = layer(c.q, k, v)
    finally:
        nva.reset_context()
    return o.view(-1, c.num_heads, c.head_dim), layer.k_cache, layer.v_cache


def _two_calls(c, k, v):
    import nanovllm_amd as nva
    kc, vc = c.k_cache.clone(), c.v_cache.clone()
    nva.store_kvcache(k, v, kc, vc, c.slot_mapping)
    o = nva.flash_attn_varlen_func(c.q, k, v, c.max_seqlen_q, c.cu_seqlens_q, c.max_seqlen_k, c.cu_seqlens_k, c.scale)
    return o, kc, vc


RAGGED = [37, 1, 300, 129, 64, 513, 2, 255]


@pytest.mark.parametrize("nh,nkv,d", [(16, 8, 128), (32, 8, 128), (64, 8, 128), (8, 8, 128), (14, 2, 64), (4, 4, 64),
                                      (4, 1, 128), (48, 3, 128)])
@pytest.mark.parametrize("lens", [[1], [927], RAGGED, RAGGED * 9], ids=["one", "long", "ragged", "persistent"])
def test_matches_the_two_calls(dev, nh, nkv, d, lens):
    from _helpers import assert_attn_close, f32
    c = _case(dev, lens, nh, nkv, d, seed=len(lens) + nh)
    c.slot_mapping[::5] = -1  # skipped rows
    c.slot_mapping[-1] = c.k_cache.shape[0] * c.k_cache.shape[1]  # one past the pool
    for _ in range(2):  # the workspace as the first call left it
        o, kc, vc = _forward(c, c.k, c.v)
        ro, rk, rv = _two_calls(c, c.k, c.v)
        torch.cuda.synchronize()
        assert torch.equal(kc, rk) and torch.equal(vc, rv)
        # bit-identical but for key halves, whose merge takes the halves in order of arrival
        assert_attn_close(f32(o), f32(ro), what="output")


@pytest.mark.parametrize("lens", [RAGGED, RAGGED * 9], ids=["direct", "persistent"])
def test_rows_that_no_item_carries(dev, lens):
    c = _case(dev, lens, 16, 8, 128, seed=4)
    _, rk, rv = _two_calls(c, c.k, c.v)
    # the last sequence's tokens and the first's outside cu_seqlens: padding rows of the batch
    c.cu_seqlens_q = c.cu_seqlens_q[1:-1].contiguous()
    c.cu_seqlens_k = c.cu_seqlens_k[1:-1].contiguous()
    _, kc, vc = _forward(c, c.k, c.v)
    torch.cuda.synchronize()
    assert torch.equal(kc, rk) and torch.equal(vc, rv)
    # positions past max_seqlen_q get no output, but their rows are stored
    c = _case(dev, lens, 16, 8, 128, seed=4)
    _, kc, vc = _forward(c, c.k, c.v, max_q=130)
    torch.cuda.synchronize()
    assert torch.equal(kc, rk) and torch.equal(vc, rv)


def test_keys_inside_the_cache_store_first(dev):
    """Keys that lie inside the cache they are stored to: the attention reads them after the
    store, as with the two calls."""
    import nanovllm_amd as nva
    c = _case(dev, RAGGED, 16, 8, 128, seed=8)
    T = c.k.shape[0]
    layer = nva.Attention(16, 128, c.scale, 8)
    outs = []
    for fused in (True, False):
        pool = torch.zeros_like(c.k_cache)
        pool.view(-1, 8, 128)[:T] = c.k
        vc = c.v_cache.clone()
        k = pool.view(-1, 8, 128)[:T]
        slots = (torch.arange(T, dtype=torch.int32, device=dev) + 7) % T  # rows of the pool that hold other keys
        slots[torch.arange(T, device=dev) % 3 != 0] = -1
        if fused:
            layer.k_cache, layer.v_cache = pool, vc
            nva.set_context(True, c.cu_seqlens_q, c.cu_seqlens_k, c.max_seqlen_q, c.max_seqlen_k, slots[:T])
            o = layer(c.q, k, c.v).view(T, 16, 128)
            nva.reset_context()
        else:
            nva.store_kvcache(k, c.v, pool, vc, slots)
            o = nva.flash_attn_varlen_func(c.q, k, c.v, c.max_seqlen_q, c.cu_seqlens_q, c.max_seqlen_k, c.cu_seqlens_k,
                                           c.scale)
        torch.cuda.synchronize()
        outs.append((o, vc))
    assert torch.equal(outs[0][1], outs[1][1])
    assert float((outs[0][0].float() - outs[1][0].float()).abs().max()) < 2e-2


@pytest.mark.parametrize("cells", ["one per CU", "above one", "four per CU", "above four"])
@pytest.mark.parametrize("prefix", [0, 128])
def test_head_dim_64_grids(dev, cells, prefix):
    """Head dim 64 at the limits of its three grids (one workgroup per CU, two, the persistent
    one): every output row against the oracle, packed and paged."""
    from _helpers import assert_attn_close, f32, prefill_reference
    from nanovllm_amd import workloads as W
    import nanovllm_amd as nva
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    per_seq = 2 * 2  # 2 kv heads x 2 query tiles of 36 positions
    seqs = {"one per CU": cus // per_seq, "above one": cus // per_seq + 1, "four per CU": 4 * cus // per_seq,
            "above four": 4 * cus // per_seq + 1}[cells]
    lens = [72 - (i % 3) * 35 for i in range(seqs)]
    c = W.make_prefill_case(lens, 14, 2, 4 * seqs, prefix_len=prefix, block_size=64, head_dim=64, seed=seqs,
                            bulk_device=dev, shared_prefix=False)
    k, v = (c.k_cache, c.v_cache) if prefix else (c.k, c.v)
    if prefix:
        nva.store_kvcache(c.k, c.v, c.k_cache, c.v_cache, c.slot_mapping)
    o = nva.flash_attn_varlen_func(c.q, k, v, c.max_seqlen_q, c.cu_seqlens_q, c.max_seqlen_k, c.cu_seqlens_k, c.scale,
                                   block_table=c.block_tables)
    torch.cuda.synchronize()
    assert_attn_close(f32(o), prefill_reference(c), what=cells)


@pytest.mark.parametrize("nh,nkv,d", [(16, 8, 128), (32, 8, 128), (24, 8, 128), (7, 1, 128), (8, 8, 128), (14, 2, 64)])
@pytest.mark.parametrize("prefix", [0, 512])
@pytest.mark.parametrize("over", [0, 1], ids=["half rows", "full rows"])
def test_half_row_items(dev, nh, nkv, d, prefix, over):
    """Small launches run items of half the rows: the last size that does and the first that does
    not, with keys enough for key halves (a long first sequence), every row against the oracle."""
    from _helpers import assert_attn_close, f32, prefill_reference
    from nanovllm_amd import workloads as W
    import nanovllm_amd as nva
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    bp = 256 // (nh // nkv)
    items = (3 if d == 128 else 1) * cus // 8  # of full rows, at most
    tiles = 2 if prefix or bp >= 256 else -(-512 // bp)  # of the longest sequence
    seqs = max(1, items // (nkv * tiles)) + over
    if not over and seqs * nkv * tiles * 8 > (3 if d == 128 else 1) * cus:
        pytest.skip("one sequence is above the limit")
    lens = [tiles * bp - 3] + [max(1, (37 * i) % (tiles * bp)) for i in range(1, seqs)]
    c = W.make_prefill_case(lens, nh, nkv, sum(-(-(n + prefix) // 128) for n in lens) + 2, prefix_len=prefix, block_size=128,
                            head_dim=d, seed=seqs, bulk_device=dev, shared_prefix=False)
    layer = nva.Attention(nh, d, c.scale, nkv)
    layer.k_cache, layer.v_cache = c.k_cache, c.v_cache
    for _ in range(2):
        nva.set_context(True, c.cu_seqlens_q, c.cu_seqlens_k, c.max_seqlen_q, c.max_seqlen_k, c.slot_mapping, None,
                        c.block_tables)
        o = layer(c.q, c.k, c.v).view(-1, nh, d)
        nva.reset_context()
        torch.cuda.synchronize()
        assert_attn_close(f32(o), prefill_reference(c), what=f"{seqs} sequences")
    rows = c.k_cache.view(-1, nkv, d)[c.slot_mapping.long()]
    assert torch.equal(rows, c.k)
