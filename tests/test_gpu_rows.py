"""The cache appends as kernels (tc_append_rows, tc_paged_append_rows) against torch's own copies: every view a
caller may hand over lands in the same rows bit for bit, and nothing else of the buffer changes. Views that the
kernels do not take (misaligned, another type, a broadcast batch) go through torch and give the same."""
import types

import pytest
import torch

from threadcut_amd import _lib, kv, paged
from threadcut_amd.match import Split

pytestmark = pytest.mark.gpu


def rows(form, b, h, n, dtype, dev, seed):
    """[b, h, n, 128] new rows in one of the forms that reach an append."""
    g = torch.Generator(device=dev).manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g, device=dev).to(dtype)
    if form == "heads first":
        return r(b, h, n, 128)
    if form == "tokens first":  # a projection's transposed view
        return r(b, n, h, 128).transpose(1, 2)
    if form == "fused qkv":     # a slice of a wider projection
        return r(b, n, h + 3, 128)[:, :, 2:2 + h].transpose(1, 2)
    if form == "every other token":
        return r(b, h, 2 * n, 128)[:, :, ::2]
    if form == "one head's rows":
        return r(b, 1, n, 128).expand(b, h, n, 128)
    if form == "misaligned":
        return r(b, h, n, 132)[..., 3:131]
    if form == "float32":
        return torch.randn(b, h, n, 128, generator=g, device=dev)
    if form == "broadcast batch":
        return r(1, h, n, 128)
    raise ValueError(form)


KERNEL = ["heads first", "tokens first", "fused qkv", "every other token", "one head's rows"]
TORCH = ["misaligned", "float32", "broadcast batch"]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form", KERNEL + TORCH)
@pytest.mark.parametrize("b,h,n", [(1, 8, 1), (2, 3, 15), (1, 8, 64), (3, 2, 65), (1, 1, 300)])
def test_growing_layer_append(gpu, form, b, h, n, dtype):
    layer = kv.GrowingLayer()
    first = rows("heads first", b, h, 7, dtype, gpu, 1)
    layer.update(first, -first)
    layer.kbuf[:, :, 7:] = 5.0
    layer.vbuf[:, :, 7:] = 6.0
    k, v = rows(form, b, h, n, dtype, gpu, 2), rows("tokens first", b, h, n, dtype, gpu, 3)
    want_k, want_v = layer.kbuf.clone(), layer.vbuf.clone()
    want_k[:, :, 7:7 + n] = k
    want_v[:, :, 7:7 + n] = v
    assert kv.rows_ok(k, layer.kbuf, n) == (form in KERNEL or form == "broadcast batch")
    native = _lib.FAST.append_rows
    taken = []
    with pytest.MonkeyPatch.context() as m:
        m.setattr(_lib, "FAST", types.SimpleNamespace(append_rows=lambda *a: taken.append(native(*a)) or taken[-1]))
        layer.update(k, v)
    assert taken == [form in KERNEL or form == "broadcast batch" and b == 1]
    assert layer.n == 7 + n
    assert torch.equal(layer.kbuf, want_k) and torch.equal(layer.vbuf, want_v)


def test_append_under_autograd_stays_with_torch(gpu):
    layer = kv.GrowingLayer()
    k = torch.randn(1, 2, 5, 128, device=gpu, dtype=torch.float16, requires_grad=True)
    assert not kv.rows_ok(k, k.detach(), 5)
    layer.update(k, k)
    layer.keys.float().sum().backward()
    assert torch.equal(k.grad, torch.ones_like(k))


def watch_rows(monkeypatch):
    """What every later PagedKV._write_rows call returns: True where the kernel took the rows."""
    taken, write = [], paged.PagedKV._write_rows
    monkeypatch.setattr(paged.PagedKV, "_write_rows", lambda *a: taken.append(write(*a)) or taken[-1])
    return taken


class Config:
    num_hidden_layers = 2

    def get_text_config(self, decoder=True):
        return self


STORES = ["layer", "layer, Python path", "slab", "slab, Python path", "pools", "paged layer"]


class Store:
    """Two heads of one sequence behind one of the caches that appends reach: rows in, cut to n tokens, and the
    tensor the cache reads its K from."""

    def __init__(self, kind, gpu, monkeypatch):
        self.kind = kind
        if "Python path" in kind:
            _lib.load()
            monkeypatch.setattr(_lib, "FAST", None)
        if kind == "pools":
            self.kv = paged.PagedKV(1, 2, 4, 16, device=gpu)
        elif kind == "paged layer":
            self.cache = paged.new_paged_cache(Config(), 8, 16)
            self.layer = self.cache.layers[0]
        else:
            self.layer = kv.new_cache(Config(), slab=kind.startswith("slab")).layers[0]

    def append(self, k, v):
        if self.kind == "pools":
            self.kv.append(0, [k], [v])
        else:
            self.layer.update(k, v)

    def cut(self, n):
        if self.kind == "pools":
            self.kv.prune(0, Split(n, self.kv.length(), 0), None)
        elif self.kind == "paged layer":
            store = paged.state_of(self.cache).kv
            store.table.prune(0, n, store.length(), 0)
            self.layer.n = n
        else:
            self.layer.crop(n)

    def keys(self):
        if self.kind not in ("pools", "paged layer"):
            return self.layer.keys[0]
        store = self.kv if self.kind == "pools" else paged.state_of(self.cache).kv
        return store.k_pools[0][int(store.table.token_slots(0)[0, 0])]


@pytest.mark.parametrize("kind", STORES)
def test_append_over_rows_that_autograd_tracks(gpu, monkeypatch, kind):
    """Plain rows written over tracked ones cut those off: no gradient reaches the rows that are gone."""
    s = Store(kind, gpu, monkeypatch)
    k = torch.randn(1, 2, 5, 128, device=gpu, dtype=torch.float16, requires_grad=True)
    s.append(k, k.detach())
    s.cut(3)
    s.append(rows("heads first", 1, 2, 2, torch.float16, gpu, 1), rows("heads first", 1, 2, 2, torch.float16, gpu, 2))
    s.keys().float().sum().backward()
    want = torch.zeros_like(k)
    want[:, :, :3] = 1
    assert torch.equal(k.grad, want)


@pytest.mark.parametrize("kind", STORES)
def test_append_tells_autograd_of_the_write(gpu, monkeypatch, kind):
    """Rows that an operation saved for its backward and an append has overwritten: backward refuses them."""
    s = Store(kind, gpu, monkeypatch)
    s.append(rows("heads first", 1, 2, 5, torch.float16, gpu, 1), rows("heads first", 1, 2, 5, torch.float16, gpu, 2))
    w = torch.ones(128, device=gpu, dtype=torch.float16, requires_grad=True)
    y = (s.keys() * w).sum()
    s.cut(3)
    with torch.no_grad():
        s.append(rows("heads first", 1, 2, 2, torch.float16, gpu, 3), rows("heads first", 1, 2, 2, torch.float16, gpu, 4))
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()


@pytest.mark.parametrize("kind", STORES)
def test_append_outside_inference_mode_keeps_its_refusal(gpu, monkeypatch, kind):
    """A cache made in inference mode takes rows there and, like any inference tensor, nowhere else."""
    with torch.inference_mode():
        s = Store(kind, gpu, monkeypatch)
        x = rows("heads first", 1, 2, 5, torch.float16, gpu, 1)
        s.append(x, x)
        s.append(x, x)
    with pytest.raises(RuntimeError, match="inference tensor"):
        s.append(rows("heads first", 1, 2, 5, torch.float16, gpu, 2), rows("heads first", 1, 2, 5, torch.float16, gpu, 2))


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
@pytest.mark.parametrize("kind", STORES)
def test_append_is_recorded_by_tracing(gpu, monkeypatch, kind):
    """torch.jit.trace, make_fx and torch.compile record the write: what they return follows new inputs."""
    from torch.fx.experimental.proxy_tensor import make_fx

    def f(k):
        s = Store(kind, gpu, monkeypatch)
        s.append(k, k)
        return s.keys()[:, :5].clone()

    a, b = (rows("heads first", 1, 2, 5, torch.float16, gpu, i) for i in (1, 2))
    assert torch.equal(f(b), b[0])
    assert torch.equal(make_fx(f)(a)(b), b[0])
    with torch.no_grad():
        assert torch.equal(torch.jit.trace(f, (a,), check_trace=False)(b), b[0])
    if kind in ("layer", "slab"):  # (the page table is host code, which compilation does not enter)
        s = Store(kind, gpu, monkeypatch)
        s.append(a, a)

        def g(k):
            s.append(k, k)
            return s.layer.keys.clone()

        assert torch.equal(torch.compile(g, backend="eager", fullgraph=True)(b), torch.cat((a, b), 2))


@pytest.mark.parametrize("native", [True, False])
def test_append_of_more_rows_than_the_kernel_takes(gpu, monkeypatch, native):
    """65535 tiles of 64 rows fill the kernel's grid; one row more goes through torch."""
    if not native:
        _lib.load()
        monkeypatch.setattr(_lib, "FAST", None)
    for n in (64 * 65535, 64 * 65535 + 1):
        layer = kv.GrowingLayer()
        k, v = (rows("heads first", 1, 1, 1, torch.float16, gpu, i).expand(1, 1, n, 128) for i in (1, 2))
        layer.update(k, v)
        assert kv.rows_ok(k, layer.kbuf, n) == (n == 64 * 65535)
        assert torch.equal(layer.kbuf, k) and torch.equal(layer.vbuf, v)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form", [f for f in KERNEL + TORCH if f != "broadcast batch"])
@pytest.mark.parametrize("layers,P,n", [(1, 16, 1), (3, 64, 65), (70, 16, 37)])
def test_paged_append(gpu, monkeypatch, form, layers, P, n, dtype):
    """PagedKV.append (every layer in one launch; 70 layers take two) from a page that is partly full."""
    h = 3
    cache = paged.PagedKV(layers, h, 12, P, dtype=dtype, device=gpu)
    cache.table.free.reverse()
    start = [rows("heads first", 1, h, 5, dtype, gpu, i) for i in range(layers)]
    cache.append(0, start, start)
    taken = watch_rows(monkeypatch)
    ks = [rows(form, 1, h, n, dtype, gpu, 100 + i) for i in range(layers)]
    vs = [rows("tokens first", 1, h, n, dtype, gpu, 300 + i)[0] for i in range(layers)]
    cache.append(0, ks, vs)
    assert taken == [form in KERNEL]
    for i in range(layers):
        k, v = cache.gather(i)
        assert torch.equal(k, torch.cat((start[i], ks[i].to(dtype)), 2)[0])
        assert torch.equal(v, torch.cat((start[i][0], vs[i]), 1))
    used = cache.table.token_slots(0)
    held = torch.zeros(12, P, dtype=torch.bool)
    held[used[:, 0], used[:, 1]] = True
    for pool in cache.k_pools + cache.v_pools:  # nothing else was written
        assert not pool.transpose(1, 2)[~held.to(gpu)].any()


@pytest.mark.parametrize("form", KERNEL + ["misaligned", "float32"])
@pytest.mark.parametrize("b,n", [(1, 40), (3, 17)])
def test_paged_layer_update(gpu, monkeypatch, form, b, n):
    """A paged cache layer's update writes every sequence's rows with one launch."""
    cache = paged.new_paged_cache(Config(), 40, 16, batch=b)
    first = rows("heads first", b, 4, 9, torch.float16, gpu, 5)
    k, v = rows(form, b, 4, n, torch.float16, gpu, 6), rows("tokens first", b, 4, n, torch.float16, gpu, 7)
    for i in range(2):
        cache.update(first, first, i)
    taken = watch_rows(monkeypatch)
    for i in range(2):
        cache.update(k, v, i)
    assert taken == [form in KERNEL] * 2
    store = paged.state_of(cache).kv
    for i in range(2):
        for j in range(b):
            gk, gv = store.gather(i, j)
            assert torch.equal(gk, torch.cat((first[j], k[j].half()), 1)) and torch.equal(gv, torch.cat((first[j], v[j]), 1))
