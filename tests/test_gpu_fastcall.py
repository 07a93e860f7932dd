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


def watch(monkeypatch):
    """Watches the native functions from here on; calling the result tells of each that was called whether it took
    its last call."""
    _lib.load()
    taken, fast = {}, _lib.FAST

    class Watched:
        def __getattr__(self, name):
            def call(*args):
                r = getattr(fast, name)(*args)
                taken[name] = r is not None and r is not False
                return r

            return call

    monkeypatch.setattr(_lib, "FAST", Watched())
    return lambda: taken


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
    taken = watch(monkeypatch)
    got, heads = outcome(f), k.shape[1]
    assert taken() == {"decode": qf in QUERIES[:3] and cf in (*CACHES[:4], "too few heads") and hq % heads == 0
                       and hq // heads <= 8}
    assert same(got, general(monkeypatch, f))


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

    taken = watch(monkeypatch)
    got = outcome(step)
    assert taken()["decode_append"] == (new in ("tokens first", "heads first"))
    assert same(got, general(monkeypatch, step))


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

    taken = watch(monkeypatch)
    got = outcome(step)
    assert taken().get("paged_append", False) == (form in ("plain", "out"))
    assert same(got, general(monkeypatch, step))


SPIN = 100_000_000  # cycles of torch.cuda._sleep's counter: tens of milliseconds or more


@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["decode", "decode_append", "paged_append", "append_rows"])
def test_native_calls_follow_the_current_stream(gpu, monkeypatch, entry):
    """A call inside a stream's context is enqueued there: behind a spin and the copies that fill its input, it finds
    the input filled."""
    b, hkv, n = 2, 8, 300
    src = query("tokens first", b, hkv if entry != "decode" else 32, torch.float16, gpu)
    k, v = cache("whole", b, hkv, n, torch.float16, gpu)
    q = query("heads first", b, 32, torch.float16, gpu)
    if entry == "append_rows":
        src = cache("tokens first", b, hkv, 70, torch.float16, gpu)[0]

    def prepared():
        """The call's input, empty, and the call."""
        x = torch.zeros_like(src)
        if entry == "decode":
            return x, lambda: attention.attention(None, x, k, v, None)[0]
        if entry == "paged_append":
            c = paged.PagedKV(1, hkv, 60, 16, batch=b, device=gpu)
            for i in range(b):
                c.append(i, [k[i]], [v[i]])
            c.reserve_step()
            return x, lambda: (c.decode_append(0, q.view(b, hkv, 4, 128), x, x, 0.1), c.k_pools[0])
        layer = kv.GrowingLayer()
        layer.update(k, v)
        if entry == "append_rows":
            return x, lambda: layer.update(x, x)
        layer.fused_append = True
        return x, lambda: (attention.attention(None, q, *layer.update(x, x), None)[0], layer.keys)

    x, call = prepared()
    x.copy_(src)
    want = [t.clone() for t in torch.utils._pytree.tree_leaves(call())]
    x, call = prepared()
    taken = watch(monkeypatch)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(SPIN)
        x.copy_(src)
        got = torch.utils._pytree.tree_leaves(call())
    assert not side.query(), "the spin ended before the call was enqueued"
    side.synchronize()
    assert taken() == {entry: True}
    assert len(got) == len(want) and all(torch.equal(a, w) for a, w in zip(got, want))
