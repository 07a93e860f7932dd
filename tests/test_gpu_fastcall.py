"""The native call paths (threadcut_amd._fast) against the general Python ones over the forms that reach them: the
same bits, the same refusals. Calls that the native code leaves (None) take the Python path as before."""
import pytest
import torch

from threadcut_amd import _lib, attention, kv, paged


def general(monkeypatch, f):
    """f() by the Python path; an exception's type and text instead of a result."""
    with monkeypatch.context() as m:
        m.setattr(_lib, "FAST", None)
        return outcome(f)


def outcome(f):
    try:
        return f()
    except Exception as e:  # noqa: BLE001
        return type(e), str(e)


def same(a, b):
    if isinstance(a, torch.Tensor):
        return isinstance(b, torch.Tensor) and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)
    return a == b


def test_host_tensors_are_left_to_python():
    _lib.load()
    f, x = _lib.FAST, torch.zeros(1, 1, 1, 128, dtype=torch.float16)
    assert f.decode(x, x, x, 1.0, 0) is None and f.decode_append(x, x, x, x, x, 1, 1.0, 0) is None
    assert f.paged_append(x, x, x, x, x, x, x, None, 1.0, 0) is None and f.append_rows(x, x, 0, x, x, 0) is False
    assert f.decode(None, 1, "k", 1.0, 0) is None and f.decode() is None


QUERIES = ["tokens first", "heads first", "heads apart", "one head more", "misaligned", "float32"]
CACHES = ["view", "whole", "tokens first", "wide rows", "dims apart", "other type", "too few heads"]


def query(form, b, hq, dtype, dev):
    g = torch.Generator(device=dev).manual_seed(1)
    r = lambda *s: torch.randn(s, generator=g, device=dev).to(dtype)
    return {"tokens first": lambda: r(b, 1, hq, 128).transpose(1, 2), "heads first": lambda: r(b, hq, 1, 128),
            "heads apart": lambda: r(b, 1, hq, 256)[..., :128].transpose(1, 2), "one head more": lambda: r(b, hq + 1, 1, 128),
            "misaligned": lambda: r(b, hq, 1, 129)[..., 1:], "float32": lambda: r(b, hq, 1, 128).float()}[form]()


def cache(form, b, hkv, n, dtype, dev):
    g = torch.Generator(device=dev).manual_seed(2)
    r = lambda *s: torch.randn(s, generator=g, device=dev).to(dtype)
    one = {"view": lambda: r(b, hkv, n + 9, 128)[:, :, :n], "whole": lambda: r(b, hkv, n, 128),
           "tokens first": lambda: r(b, n, hkv, 128).transpose(1, 2), "wide rows": lambda: r(b, hkv, n, 192)[..., 64:],
           "dims apart": lambda: r(b, hkv, n, 256)[..., ::2], "other type": lambda: r(b, hkv, n, 128).float(),
           "too few heads": lambda: r(b, max(1, hkv - 1), n, 128)}[form]
    return one(), one()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("qf,cf", [(q, "view") for q in QUERIES] + [("tokens first", c) for c in CACHES[1:]])
@pytest.mark.parametrize("b,hq,hkv,n", [(1, 8, 2, 1), (1, 32, 8, 300), (3, 4, 4, 77), (2, 16, 1, 20), (2, 8, 1, 2300)])
def test_decode(gpu, monkeypatch, qf, cf, b, hq, hkv, n, dtype):
    if cf == "too few heads" and hkv == 1:
        pytest.skip("one head")
    q, (k, v) = query(qf, b, hq, dtype, gpu), cache(cf, b, hkv, n, dtype, gpu)
    f = lambda: attention.attention(None, q, k, v, None, scaling=0.1)[0]
    assert same(outcome(f), general(monkeypatch, f))


@pytest.mark.gpu
@pytest.mark.parametrize("pos", [False, True])
@pytest.mark.parametrize("new", ["tokens first", "heads first", "misaligned", "float32"])
@pytest.mark.parametrize("b,hq,hkv,n", [(1, 8, 2, 1), (1, 32, 8, 300), (3, 4, 4, 77), (2, 8, 1, 2300)])
def test_append(gpu, monkeypatch, new, pos, b, hq, hkv, n):
    def step():
        layer = kv.GrowingLayer()
        layer.fused_append = True
        k, v = cache("whole", b, hkv, n + 1, torch.float16, gpu)
        layer.update(k, v)
        layer.n = n
        if pos:
            layer.device_pos = torch.full((b,), n, dtype=torch.int32, device=gpu)
            layer.in_graph_step = True
        kn = query(new, b, hkv, torch.float16, gpu)
        q = query("tokens first", b, hq, torch.float16, gpu)
        out = attention.attention(None, q, *layer.update(kn, kn + 1), None)[0]
        assert layer.pending is None
        return torch.cat((out.flatten(), layer.kbuf[:, :, :n + 1].flatten(), layer.vbuf[:, :, :n + 1].flatten()))

    assert same(outcome(step), general(monkeypatch, step))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "out", "small out", "float32 row", "wrong heads", "no step"])
@pytest.mark.parametrize("b", [1, 3])
def test_paged_append(gpu, monkeypatch, form, b):
    def step():
        c = paged.PagedKV(2, 4, 30, 16, batch=b, device=gpu)
        for i in range(b):
            k = cache("whole", 1, 4, 20 + 30 * i, torch.float16, gpu)[0]
            c.append(i, [k, k], [k, k])
        q = query("heads first", b, 16, torch.float16, gpu).reshape(b, 4, 4, 128)
        kn = query("tokens first", b, 4, torch.float32 if form == "float32 row" else torch.float16, gpu)
        if form == "wrong heads":
            q = q[:, :3]
        out = {"out": torch.zeros_like(q), "small out": torch.zeros_like(q)[:, :2]}.get(form)
        if form != "no step":
            c.reserve_step()
        got = c.decode_append(1, q, kn, kn, 0.1, out=out)
        assert out is None or got is out or got.data_ptr() == out.data_ptr()
        return torch.cat((got.flatten(), c.k_pools[1].flatten(), c.v_pools[1].flatten()))

    assert same(outcome(step), general(monkeypatch, step))


@pytest.mark.gpu
def test_native_calls_follow_the_current_stream(gpu):
    """A call inside a stream's context is enqueued there: it waits for the work before it."""
    q = query("tokens first", 1, 32, torch.float16, gpu)
    k, v = cache("whole", 1, 8, 300, torch.float16, gpu)
    want = attention.attention(None, q, k, v, None)[0]
    k2, s = torch.zeros_like(k), torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(20):
            k2.zero_()
        k2.copy_(k)
        got = attention.attention(None, q, k2, v, None)[0]
    s.synchronize()
    assert torch.equal(got, want)
