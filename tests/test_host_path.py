"""The native form of Attention.forward and qk_norm_rope (csrc/host/nva_host.cpp): bit-identical
to the general Python path over the forms it takes, None (and so the general path) for the
others, and the store inside a small batch's decode launch equal to store-then-decode for any
slots."""
from __future__ import annotations

import pytest
import torch


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    from nanovllm_amd import _capi
    _capi.load()
    return torch.device("cuda:0")


class _Off:
    """A host module that takes nothing."""

    @staticmethod
    def attention(*args):
        return None

    @staticmethod
    def qk_norm_rope(*args):
        return None


class _Spy:
    def __init__(self, real):
        self.real, self.taken = real, 0

    def attention(self, *args):
        o = self.real.attention(*args)
        self.taken += o is not None
        return o

    def qk_norm_rope(self, *args):
        o = self.real.qk_norm_rope(*args)
        self.taken += o is not None
        return o


def test_host_module_missing(monkeypatch, tmp_path):
    """Without the host module, and with one built for another torch, the calls run in Python."""
    from nanovllm_amd import _capi
    assert _capi.host().torch_version == torch.__version__.split("+")[0]
    for path, version in ((tmp_path / "_nva_host.so", torch.__version__), (_capi.HOST_PATH, "1.0.0")):
        with monkeypatch.context() as m:
            m.setattr(_capi, "_host", None)
            m.setattr(_capi, "HOST_PATH", path)
            m.setattr(torch, "__version__", version)
            with pytest.warns(RuntimeWarning, match="is not used"):
                host = _capi.host()
            assert host.attention(1, 2) is None and host.qk_norm_rope(1) is None
            assert _capi.host() is host


def _layer(c, k_cache, v_cache, scales=(None, None)):
    import nanovllm_amd as nva
    layer = nva.Attention(c.num_heads, c.head_dim, c.scale, c.num_kv_heads)
    layer.k_cache, layer.v_cache = k_cache, v_cache
    layer.k_scale, layer.v_scale = scales
    return layer


def _both(monkeypatch, run):
    """run() through the general path and through the native one; each returns its tensors."""
    from nanovllm_amd import _capi
    real = _capi.host()
    with monkeypatch.context() as m:
        m.setattr(_capi, "_host", _Off)
        want = run()
    spy = _Spy(real)
    with monkeypatch.context() as m:
        m.setattr(_capi, "_host", spy)
        got = run()
    torch.cuda.synchronize()
    return want, got, spy.taken


def _same(want, got):
    for a, b in zip(want, got):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["2d", "3d", "strided"])
@pytest.mark.parametrize("prefix", [0, 256])
@pytest.mark.parametrize("fp8", [False, True])
def test_prefill_equals_the_general_path(dev, monkeypatch, form, prefix, fp8):
    import nanovllm_amd as nva
    from nanovllm_amd import workloads as W
    c = W.make_prefill_case([30, 1, 100], 16, 8, 12, prefix_len=prefix, seed=3, bulk_device=dev)
    scales = (None, None)
    if fp8:
        c.k_cache, ks = W.quantize_cache_fp8(c.k_cache, extra=c.k)
        c.v_cache, vs = W.quantize_cache_fp8(c.v_cache, extra=c.v)
        scales = (ks, vs)
    q, k, v = c.q, c.k, c.v
    if form == "2d":
        q, k = q.view(-1, 2048), k.view(-1, 1024)
    elif form == "strided":
        qkv = torch.cat([t.reshape(t.shape[0], -1) for t in (q, k, v)], dim=1)
        q, k, v = qkv[:, :2048], qkv[:, 2048:3072], qkv[:, 3072:]

    def run():
        layer = _layer(c, c.k_cache.clone(), c.v_cache.clone(), scales)
        nva.set_context(True, c.cu_seqlens_q, c.cu_seqlens_k, c.max_seqlen_q, c.max_seqlen_k, c.slot_mapping, None,
                        c.block_tables)
        o = layer(q, k, v)
        nva.reset_context()
        return o, layer.k_cache, layer.v_cache
    run()  # the stream's workspace
    want, got, taken = _both(monkeypatch, run)
    _same(want, got)
    assert taken == 1


def _decode_inputs(dev, B, nh, nkv, d, fp8, seed):
    from nanovllm_amd import workloads as W
    base = [1, 33, 0, 256, 257, 700, 31, 32, 64, 900]
    lens = [base[i % len(base)] for i in range(B)]
    return W.make_decode_case(B, nh, nkv, 0, 0, 5 * B + 2, head_dim=d, fp8=fp8, seed=seed, bulk_device=dev, lengths=lens,
                              table_width=4)


@pytest.mark.gpu
@pytest.mark.parametrize("slots", ["own", "rolled", "inside", "foreign", "padding", "out of range"])
@pytest.mark.parametrize("B,nh,nkv,d,fp8", [(1, 16, 8, 128, False), (10, 16, 8, 128, False), (10, 64, 8, 128, True),
                                            (32, 16, 8, 128, False), (100, 14, 2, 64, False), (200, 4, 1, 128, False),
                                            (64, 16, 8, 128, False)])
def test_decode_equals_store_then_decode(dev, monkeypatch, slots, B, nh, nkv, d, fp8):
    """Spread mode (batch x kv heads up to 256) and, last, the balanced mode."""
    import nanovllm_amd as nva
    c = _decode_inputs(dev, B, nh, nkv, d, fp8, seed=B)
    s = c.slot_mapping
    live = [b for b, n in enumerate(c.lengths) if n > 0]
    if slots == "padding" and B == 1:
        pytest.skip("one live row")
    if slots == "rolled":  # row b goes to another sequence's last key
        s[live] = s[live].roll(1)
    elif slots == "inside":  # row b goes to the middle of its own context
        for b in live:
            n = c.lengths[b] // 2
            s[b] = int(c.block_tables[b, n // 256]) * 256 + n % 256
    elif slots == "foreign":  # row b goes to the first key of the sequence after it
        s[live] = (c.block_tables[live, 0] * 256).roll(-1)
    elif slots == "padding":  # rows without keys go to slots that live sequences read
        # (of more than one key: the row of a one-key sequence goes to that very slot, and which
        # of two rows a slot keeps is not defined by the store; test_rows_that_share_a_slot)
        empty = [b for b, n in enumerate(c.lengths) if n == 0]
        longer = [b for b in live if c.lengths[b] > 1]
        for i, b in enumerate(empty):
            s[b] = int(c.block_tables[longer[i % len(longer)], 0]) * 256
    elif slots == "out of range":
        s[::2] = -1
        s[1::2] = c.k_cache.shape[0] * 256

    def run():
        layer = _layer(c, c.k_cache.clone(), c.v_cache.clone(), (c.k_scale, c.v_scale))
        nva.set_context(False, slot_mapping=s, context_lens=c.context_lens, block_tables=c.block_tables)
        o = layer(c.q, c.k_new, c.v_new)
        nva.reset_context()
        return o, layer.k_cache, layer.v_cache
    want, got, taken = _both(monkeypatch, run)
    assert taken == 1
    _same(want, got)


@pytest.mark.gpu
@pytest.mark.parametrize("width", [1, 4])  # one block: the short-table kernel
@pytest.mark.parametrize("B,nh,nkv,d,fp8", [(3, 16, 8, 128, False), (10, 64, 8, 128, True), (32, 16, 8, 128, False),
                                            (100, 14, 2, 64, False), (200, 4, 1, 128, False)])
def test_rows_that_share_a_slot(dev, B, nh, nkv, d, fp8, width):
    """Of rows that share a slot the spread mode stores the first, and every sequence attends over
    what the caches then hold (bit-identical to the two calls with the later rows skipped)."""
    import nanovllm_amd as nva
    from nanovllm_amd import workloads as W
    base = [1, 33, 0, 256, 0, 1, 31, 200, 0, 64]
    lens = [base[i % len(base)] for i in range(B)]
    c = W.make_decode_case(B, nh, nkv, 0, 0, B * width + 2, head_dim=d, fp8=fp8, seed=B, bulk_device=dev, lengths=lens,
                           table_width=width)
    last = [int(c.block_tables[b, (n - 1) // 256]) * 256 + (n - 1) % 256 if n else -1 for b, n in enumerate(lens)]
    s = list(last)
    for b in range(1, B):
        if b % 3 == 2 or lens[b] == 0:  # an earlier or a later row's slot, or its sequence's first key
            o = (b * 7 + 1) % B
            s[b] = last[o] if b % 2 else int(c.block_tables[o, 0]) * 256
    if lens[0] == 1 and B > 2:
        s[2] = s[0]  # a row without keys against the only key of a sequence
    seen, first = set(), []
    for x in s:
        first.append(-1 if x in seen else x)
        seen.add(x)
    assert any(x != y for x, y in zip(s, first))

    def slots(x):
        return torch.tensor(x, dtype=torch.int32, device=dev)
    layer = _layer(c, c.k_cache.clone(), c.v_cache.clone(), (c.k_scale, c.v_scale))
    nva.set_context(False, slot_mapping=slots(s), context_lens=c.context_lens, block_tables=c.block_tables)
    o = layer(c.q, c.k_new, c.v_new).view(B, nh, d)
    nva.reset_context()
    nva.store_kvcache(c.k_new, c.v_new, c.k_cache, c.v_cache, slots(first), c.k_scale, c.v_scale)
    two = nva.flash_attn_with_kvcache(c.q.unsqueeze(1), c.k_cache, c.v_cache, c.context_lens, c.block_tables,
                                      softmax_scale=c.scale, k_scale=c.k_scale, v_scale=c.v_scale)
    torch.cuda.synchronize()
    _same((two[:, 0], c.k_cache, c.v_cache), (o, layer.k_cache, layer.v_cache))


@pytest.mark.gpu
@pytest.mark.parametrize("B,nh,nkv,d,fp8,bs,width", [
    (1, 16, 8, 128, False, 256, 1), (10, 16, 8, 128, False, 256, 1), (16, 64, 8, 128, True, 128, 2),
    (10, 128, 8, 128, False, 32, 8), (60, 14, 2, 64, False, 256, 1), (128, 4, 1, 128, True, 32, 5),
    (9, 16, 8, 128, False, 32, 2), (20, 5, 5, 64, False, 64, 3)])
@pytest.mark.parametrize("slots", ["own", "rolled", "empty rows"])
def test_short_tables_in_one_launch(dev, B, nh, nkv, d, fp8, bs, width, slots):
    """Tables of at most eight steps: one workgroup per (sequence, kv head), bit-identical to the
    spread kernel and its merge (store_and_decode keeps those), with and without the store,
    and equal to the oracle."""
    import nanovllm_amd as nva
    from _helpers import FP8_MAX_ABS, assert_attn_close, decode_reference, f32
    from nanovllm_amd import workloads as W
    cap = bs * width
    base = [1, 31, 0, 32, 33, cap, cap - 1, cap // 2, 2, min(cap, 64)]
    lens = [base[i % len(base)] for i in range(B)]
    c = W.make_decode_case(B, nh, nkv, 0, 0, B * width + 2, head_dim=d, fp8=fp8, seed=B + d, bulk_device=dev,
                           block_size=bs, lengths=lens, table_width=width)
    live = [b for b, n in enumerate(lens) if n > 0]
    s = c.slot_mapping
    if slots == "rolled":
        s[live] = s[live].roll(1)
    elif slots == "empty rows":  # to slots past the live keys: nobody reads them
        used = set(c.block_tables.flatten().tolist())
        free = [i for i in range(B * width + 2) if i not in used]
        for i, b in enumerate(b for b, n in enumerate(lens) if n == 0):
            s[b] = free[i // bs] * bs + i % bs
    tol = dict(max_abs=FP8_MAX_ABS, mean_abs=FP8_MAX_ABS) if fp8 else {}
    args = dict(softmax_scale=c.scale, k_scale=c.k_scale, v_scale=c.v_scale)
    layer = _layer(c, c.k_cache.clone(), c.v_cache.clone(), (c.k_scale, c.v_scale))
    nva.set_context(False, slot_mapping=s, context_lens=c.context_lens, block_tables=c.block_tables)
    one = layer(c.q, c.k_new, c.v_new).view(B, nh, d)
    nva.reset_context()
    if slots != "rolled":
        kc, vc = c.k_cache.clone(), c.v_cache.clone()
        spread = nva.store_and_decode(c.q.unsqueeze(1), c.k_new, c.v_new, kc, vc, s, c.context_lens, c.block_tables, **args)
        torch.cuda.synchronize()
        _same((spread[:, 0], kc, vc), (one, layer.k_cache, layer.v_cache))
    nva.store_kvcache(c.k_new, c.v_new, c.k_cache, c.v_cache, s, c.k_scale, c.v_scale)
    two = nva.flash_attn_with_kvcache(c.q.unsqueeze(1), c.k_cache, c.v_cache, c.context_lens, c.block_tables, **args)
    torch.cuda.synchronize()
    _same((two[:, 0], c.k_cache, c.v_cache), (one, layer.k_cache, layer.v_cache))
    assert_attn_close(f32(one), decode_reference(c), what=f"short {B} {nh}/{nkv} d={d}", **tol)


@pytest.mark.gpu
def test_producer_equals_the_general_path(dev, monkeypatch):
    from nanovllm_amd import workloads as W
    from nanovllm_amd.layers.qk_norm_rope import qk_norm_rope
    for nh, nkv, d, norm in ((16, 8, 128, True), (14, 2, 64, False)):
        c = W.make_producer_case(19, nh, nkv, head_dim=d, norm=norm, seed=2, device=dev)
        for q, k in ((c.q, c.k), (c.qkv[:, :nh * d], c.qkv[:, nh * d:(nh + nkv) * d])):
            want, got, taken = _both(monkeypatch, lambda: qk_norm_rope(
                c.positions, q, k, c.cos_sin_cache, nh, nkv, d, c.q_norm_weight, c.k_norm_weight))
            _same(want, got)
            assert taken == 1


@pytest.mark.gpu
def test_other_forms_are_left_to_the_general_path(dev):
    """Wrapped tensors, active modes and forms that the general path converts or refuses."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from nanovllm_amd import _capi
    c = _decode_inputs(dev, 10, 16, 8, 128, False, seed=1)

    def call(**kw):
        a = dict(q=c.q, k=c.k_new, v=c.v_new, kc=c.k_cache, vc=c.v_cache, ks=None, vs=None, nh=16, nkv=8, d=128,
                 scale=c.scale, fuse=False, pre=False, cq=None, ck=None, mq=0, mk=0, slots=c.slot_mapping,
                 lens=c.context_lens, bt=c.block_tables, ws={}, lim=4096)
        a.update(kw)
        return _capi.host().attention(*a.values())

    assert call() is not None

    class Sub(torch.Tensor):
        pass

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for kw in (dict(q=c.q.float()), dict(q=c.q.cpu()), dict(q=c.q.as_subclass(Sub)), dict(q=c.q[:, ::2]),
               dict(q=c.q[:9]), dict(slots=c.slot_mapping.long()), dict(slots=c.slot_mapping.cpu()),
               dict(lens=c.context_lens[:9]), dict(bt=c.block_tables.t()), dict(bt=None), dict(scale=1), dict(nh=True),
               dict(kc=c.k_cache.transpose(0, 1)), dict(kc=c.k_cache.half()), dict(nh=12), dict(pre=1),
               dict(pre=True, cq=c.context_lens, ck=c.context_lens), dict(kc=torch.tensor([]), vc=torch.tensor([]))):
        assert call(**kw) is None, kw.keys()
    with Mode():
        assert call() is None
    with torch.device("cpu"):  # a function mode (as torch.set_default_device installs)
        assert call() is None
    assert call() is not None
    assert torch.func.vmap(lambda x: (call(q=x) is None) * x.sum())(c.q.unsqueeze(0)) is not None
    seen = []
    torch.func.vmap(lambda x: (seen.append(call(q=x)), x)[1])(c.q.unsqueeze(0))
    assert seen == [None]


@pytest.mark.gpu
def test_streams_and_threads(dev):
    """Native decodes and prefills on streams of their own, from two threads at once, equal those
    on the default stream (each stream has its own prefill workspace)."""
    import threading

    import nanovllm_amd as nva
    from nanovllm_amd import _capi
    from nanovllm_amd import workloads as W
    from nanovllm_amd.layers import attention as A
    host = _capi.host()
    dec = [_decode_inputs(dev, 40, 16, 8, 128, False, seed=i) for i in range(2)]
    pre = [W.make_prefill_case([900, 300 + i, 40], 16, 8, 12, seed=i, bulk_device=dev) for i in range(2)]

    def both(i):
        c, p = dec[i], pre[i]
        kc, vc, pk, pv = c.k_cache.clone(), c.v_cache.clone(), p.k_cache.clone(), p.v_cache.clone()
        stream = torch.cuda.current_stream(dev)
        nva.flash_attn_varlen_func(p.q, p.k, p.v, p.max_seqlen_q, p.cu_seqlens_q, p.max_seqlen_k, p.cu_seqlens_k, p.scale)
        a = host.attention(c.q, c.k_new, c.v_new, kc, vc, None, None, 16, 8, 128, c.scale, False, False, None, None, 0, 0,
                           c.slot_mapping, c.context_lens, c.block_tables, {}, 4096)
        b = host.attention(p.q, p.k, p.v, pk, pv, None, None, 16, 8, 128, p.scale, False, True, p.cu_seqlens_q,
                           p.cu_seqlens_k, p.max_seqlen_q, p.max_seqlen_k, p.slot_mapping, None, None,
                           A._PREFILL_WORKSPACES, 4096)
        assert a is not None and b is not None
        stream.synchronize()
        return a, kc, vc, pk, pv, b

    want = [both(i) for i in range(2)]
    torch.cuda.synchronize()
    got, errors = [None, None], []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream(dev)):
                for _ in range(5):
                    got[i] = both(i)
        except Exception as e:  # a thread's exception would be lost
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for w, g in zip(want, got):
        _same(w[:5], g[:5])
        # key halves merge in order of arrival: the prefill's outputs to rounding
        assert float((w[5].float() - g[5].float()).abs().max()) < 2e-2


def test_host_tensors_are_left_to_the_general_path():
    from nanovllm_amd import _capi
    x = torch.zeros(2, 8, 128, dtype=torch.bfloat16)
    i = torch.zeros(2, dtype=torch.int32)
    kc = torch.zeros(2, 256, 8, 128, dtype=torch.bfloat16)
    host = _capi.host()
    assert host.attention(x, x, x, kc, kc, None, None, 8, 8, 128, 0.1, False, False, None, None, 0, 0, i, i,
                          torch.zeros(2, 1, dtype=torch.int32), {}, 4096) is None
    assert host.attention() is None and host.qk_norm_rope() is None
    assert host.qk_norm_rope(i.long(), x, x, torch.zeros(4, 128), 8, 8, 128, None, None, 1e-6) is None
