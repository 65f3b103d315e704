"""The attention call carried from its tensors to the library in one native step: the same bits as the Python methods give
on a second cache, and the same errors; what is not of the ordinary form is left to those methods with nothing done."""
import sys

import pytest
import torch

import kvhip
import kvhip._lib as L

B, HQ, HKV, D, CTX = 2, 8, 2, 64, 70


class OtherRoPE(kvhip.RoPE):
    def to_c(self):
        return kvhip.RoPE(self.dims, base=500.0).to_c()


def _rand(gen, *shape, dtype):
    return torch.randn(*shape, generator=gen, device="cuda").to(dtype)


def _pair(kind, dtype):
    """Two caches of the same rows, the second without the native step, and the list of the first one's native outcomes."""
    gen = torch.Generator(device="cuda").manual_seed(11)
    k, v = _rand(gen, B, HKV, CTX, D, dtype=dtype), _rand(gen, B, HKV, CTX, D, dtype=dtype)
    caches, outcomes = [], []
    for _ in range(2):
        c = {"simple": kvhip.KVCacheSimple, "ring": lambda: kvhip.RotatingKVCache(64, keep=4),
             "q4": lambda: kvhip.QuantizedKVCache(64, 4)}[kind]()
        c._update(k, v)
        caches.append(c)
    native = caches[0]._attend_natively
    caches[0]._attend_natively = lambda *a: outcomes.append(native(*a)) or outcomes[-1]
    caches[1]._attend_natively = lambda *a: None
    return caches, outcomes, gen


def _same(caches, call):
    got, want = call(caches[0]), call(caches[1])
    assert got.dtype == want.dtype and torch.equal(got, want)
    assert caches[0].offset == caches[1].offset
    for a, b in zip(caches[0].state, caches[1].state):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,dtype", [("simple", torch.float16), ("simple", torch.float32), ("ring", torch.bfloat16), ("q4", torch.float16)])
@pytest.mark.parametrize("n", [1, 3, 40])
def test_ordinary_calls_are_taken(kind, dtype, n):
    caches, outcomes, gen = _pair(kind, dtype)
    freqs = torch.linspace(1.0, 900.0, D // 2)
    for rope in (None, kvhip.RoPE(D), kvhip.RoPE(D // 2, traditional=True, base=500, scale=0.5), kvhip.RoPE(D, freqs=freqs)):
        for mask in (None, kvhip.MaskMode.none(), kvhip.MaskMode.causal()):
            q, k, v = (_rand(gen, B, h, n, D, dtype=dtype) for h in (HQ, HKV, HKV))
            if rope is None:
                _same(caches, lambda c: kvhip.attention_with_cache_update(q, k, v, c, 0.125, mask))
            else:
                _same(caches, lambda c: kvhip.attention_with_rope_and_cache_update(rope, q, k, v, c, 0.125, mask))
    assert len(outcomes) == 12 and all(o is not None for o in outcomes)


@pytest.mark.gpu
def test_other_forms_are_left_to_the_general_path():
    caches, outcomes, gen = _pair("simple", torch.float16)
    q, k, v = (_rand(gen, B, h, 2, D, dtype=torch.float16) for h in (HQ, HKV, HKV))
    rope, offset = kvhip.RoPE(D), CTX
    turned = q.transpose(1, 2).contiguous().transpose(1, 2)
    for call in (lambda c: kvhip.attention_with_cache_update(turned, k, v, c, 0.125),
                 lambda c: kvhip.attention_with_cache_update(q, k, v, c, 0.125, kvhip.MaskMode.window_mask(c.offset, 16)),
                 lambda c: kvhip.attention_with_rope_and_cache_update(OtherRoPE(D), q, k, v, c, 0.125),
                 lambda c: kvhip.attention_with_rope_and_cache_update(rope, q, k, v.transpose(0, 1).contiguous().transpose(0, 1),
                                                                              c, 0.125)):
        _same(caches, call)
    assert outcomes and all(o is None for o in outcomes)
    _same(caches, lambda c: kvhip.attention_with_rope_and_cache_update(
        rope, q, k, v, c, 0.125, batch_offsets=torch.tensor([3, 9], dtype=torch.int32)))
    assert caches[0].offset == offset + 10
    bad = [(q.float(), k, v), (q, k.float(), v.float()), (_rand(gen, B, 3, 2, D, dtype=torch.float16), k, v)]
    for args in bad:
        raised = []
        for c in caches:
            with pytest.raises(Exception) as e:
                kvhip.attention_with_cache_update(*args, c, 0.125)
            raised.append((e.type, str(e.value), c.offset))
        assert raised[0] == raised[1]


@pytest.mark.gpu
@pytest.mark.parametrize("rotary", [False, True])
def test_first_rows_and_captured_steps(rotary):
    gen = torch.Generator(device="cuda").manual_seed(5)
    caches = [kvhip.KVCacheSimple(), kvhip.KVCacheSimple()]
    caches[1]._attend_natively = lambda *a: None
    rope = kvhip.RoPE(D)

    def call(c, q, k, v):
        if rotary:
            return kvhip.attention_with_rope_and_cache_update(rope, q, k, v, c, 0.125)
        return kvhip.attention_with_cache_update(q, k, v, c, 0.125)

    for n in (300, 1):
        q, k, v = (_rand(gen, B, h, n, D, dtype=torch.float16) for h in (HQ, HKV, HKV))
        _same(caches, lambda c: call(c, q, k, v))
    want = call(caches[1], q, k, v)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = call(caches[0], q, k, v)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_host_tensors_and_wrong_arguments_are_not_taken():
    step = L.step()[0] if torch.cuda.is_available() else pytest.importorskip("kvhip._step")
    x = torch.zeros(1, 1, 1, 64)
    if not torch.cuda.is_available():
        step.bind(torch.Tensor, kvhip.RoPE, (torch.float16, torch.bfloat16, torch.float32), int, int)
    assert step.attend(1, 1, (1, 1, 64, 64, torch.float32), x, x, x, 1.0, 1, None, 0) is None
    assert step.attend(1, 1, None, None, x, x, 1.0, 1, None, 0) is None
    with pytest.raises(TypeError):
        step.attend(1, 1)


def test_the_package_does_without_the_extension(monkeypatch):
    monkeypatch.setitem(sys.modules, "kvhip._step", None)
    monkeypatch.setattr(L, "_step", None)
    assert L.step() == (None, None, None)


@pytest.mark.gpu
def test_caches_without_the_extension_give_the_same(monkeypatch):
    caches, outcomes, gen = _pair("q4", torch.float16)
    with monkeypatch.context() as m:
        m.setitem(sys.modules, "kvhip._step", None)
        m.setattr(L, "_step", None)
        other = kvhip.QuantizedKVCache(64, 4)
    other.state = caches[0].state
    other.offset = caches[0].offset
    rope = kvhip.RoPE(D)
    for n in (1, 3):
        q, k, v = (_rand(gen, B, h, n, D, dtype=torch.float16) for h in (HQ, HKV, HKV))
        _same([caches[0], other], lambda c: kvhip.attention_with_rope_and_cache_update(rope, q, k, v, c, 0.125))
        _same([caches[0], other], lambda c: kvhip.attention_with_cache_update(q, k, v, c, 0.125))
    assert outcomes and all(o is not None for o in outcomes)


@pytest.mark.gpu
def test_a_call_that_is_not_taken_is_tried_once():
    gen = torch.Generator(device="cuda").manual_seed(3)
    cache, tried = kvhip.KVCacheSimple(), []
    native = cache._attend_natively
    cache._attend_natively = lambda *a: tried.append(a) or native(*a)
    rope = kvhip.RoPE(D)
    for n, mask in ((CTX, None), (700, kvhip.MaskMode.causal()), (2, kvhip.MaskMode.window_mask(CTX + 700, 16))):
        q, k, v = (_rand(gen, B, h, n, D, dtype=torch.float16) for h in (HQ, HKV, HKV))
        kvhip.attention_with_rope_and_cache_update(rope, q, k, v, cache, 0.125, mask)
        assert len(tried) == 1, n
        tried.clear()


@pytest.mark.gpu
def test_an_interrupt_is_not_swallowed():
    class Scale:
        interrupted = False

        def __float__(self):
            if not self.interrupted:
                self.interrupted = True
                raise KeyboardInterrupt
            return 0.125

    gen = torch.Generator(device="cuda").manual_seed(4)
    cache = kvhip.KVCacheSimple()
    q, k, v = (_rand(gen, B, h, 4, D, dtype=torch.float16) for h in (HQ, HKV, HKV))
    kvhip.attention_with_cache_update(q, k, v, cache, 0.125)
    with pytest.raises(KeyboardInterrupt):
        kvhip.attention_with_cache_update(q, k, v, cache, Scale())
    assert cache.offset == 4
