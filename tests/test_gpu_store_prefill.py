"""The store fused into a packed prefill (nva_store_prefill, Attention.forward without a cached
prefix): caches bit-identical to store_kvcache and outputs equal to flash_attn_varlen_func on
the same inputs, over the grids and head shapes that fuse, those that do not, and rows that no
work item carries (past cu_seqlens_q's end, past max_seqlen_q)."""
from __future__ import annotations

from types import SimpleNamespace

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


SHORT_D64 = [1, 63, 64, 65, 300, 0, 777]  # 44 cells a sequence at heads 14/2, 13 key tiles


@pytest.mark.parametrize("times", [1, 2, 3], ids=["key halves", "up to four per CU", "four per CU"])
def test_two_workgroups_per_cu(dev, times):
    """Head dim 64 with two workgroups per CU and the store in the launch: caches bit-identical to
    store_kvcache and every output row against the oracle, with skipped slots, rows outside
    cu_seqlens and positions past max_seqlen_q."""
    from _helpers import assert_attn_close, f32, prefill_reference
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    lens = SHORT_D64 * times + [40] * (2 if times == 3 else 0)
    cells = 2 * len(lens) * -(-max(lens) // 36)
    lo, hi = ((cus, 2 * cus), (2 * cus, 3 * cus), (3 * cus, 4 * cus))[times - 1]
    assert lo < cells <= hi and -(-max(lens) // 64) <= 16, "another grid"
    c = _case(dev, lens, 14, 2, 64, seed=times)
    c.slot_mapping[::5] = -1
    c.slot_mapping[-1] = c.k_cache.shape[0] * c.k_cache.shape[1]
    ref = prefill_reference(c)
    _, rk, rv = _two_calls(c, c.k, c.v)
    for _ in range(2):  # the workspace as the first call left it
        o, kc, vc = _forward(c, c.k, c.v)
        torch.cuda.synchronize()
        assert torch.equal(kc, rk) and torch.equal(vc, rv)
        assert_attn_close(f32(o), ref, what=f"{cells} cells")
    _, kc, vc = _forward(c, c.k, c.v, max_q=max(lens) - 40)
    torch.cuda.synchronize()
    assert torch.equal(kc, rk) and torch.equal(vc, rv)
    c.cu_seqlens_q, c.cu_seqlens_k = (t[1:-1].contiguous() for t in (c.cu_seqlens_q, c.cu_seqlens_k))
    assert cus < 2 * (len(lens) - 2) * -(-max(lens) // 36) or times == 1
    _, kc, vc = _forward(c, c.k, c.v)
    torch.cuda.synchronize()
    assert torch.equal(kc, rk) and torch.equal(vc, rv)


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


@pytest.mark.parametrize("nh,nkv,d", [(16, 8, 128), (8, 1, 128), (14, 2, 64)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("keys", [16, 17, 24, 25], ids=lambda t: f"{t} tiles")
@pytest.mark.parametrize("seqs", [1, 3, 9])
def test_half_row_items_and_key_halves(dev, nh, nkv, d, fp8, keys, seqs):
    """Half-row items on both sides of the context lengths from which they are cut in key halves
    (one to nine sequences of 40 tokens behind a cached prefix, and the first alone long):
    every row against the oracle."""
    from _helpers import FP8_MAX_ABS, assert_attn_close, f32, prefill_reference
    from nanovllm_amd import workloads as W
    import nanovllm_amd as nva
    if fp8 and d == 64:
        pytest.skip("fp8 caches are read at head dim 128")
    prefix = 64 * keys - 64
    lens = [64] + [40] * (seqs - 1)
    c = W.make_prefill_case(lens, nh, nkv, seqs * -(-(prefix + 64) // 64) + 2, prefix_len=prefix, block_size=64, head_dim=d,
                            seed=keys + seqs, bulk_device=dev, shared_prefix=False)
    layer = nva.Attention(nh, d, c.scale, nkv)
    tol = {}
    if fp8:
        c.k_cache, layer.k_scale = W.quantize_cache_fp8(c.k_cache, extra=c.k)
        c.v_cache, layer.v_scale = W.quantize_cache_fp8(c.v_cache, extra=c.v)
        tol = dict(max_abs=FP8_MAX_ABS, mean_abs=FP8_MAX_ABS)
    layer.k_cache, layer.v_cache = c.k_cache, c.v_cache
    for _ in range(2):
        nva.set_context(True, c.cu_seqlens_q, c.cu_seqlens_k, c.max_seqlen_q, c.max_seqlen_k, c.slot_mapping, None,
                        c.block_tables)
        o = layer(c.q, c.k, c.v).view(-1, nh, d)
        nva.reset_context()
        torch.cuda.synchronize()
        ref = c
        if fp8:  # the oracle reads the dequantised values
            ref = SimpleNamespace(**{**vars(c), "k_cache": c.k_cache.float() * layer.k_scale[:, None],
                                     "v_cache": c.v_cache.float() * layer.v_scale[:, None]})
        assert_attn_close(f32(o), prefill_reference(ref), what=f"{keys} tiles", **tol)
