"""Every entry point enqueues on the caller's current stream.

On a side stream (default priority, non-blocking), a spin kernel holds the
stream for milliseconds, the inputs are then written on that stream by
device-to-device copies from sources already on the GPU, and the call
follows. A launch on any other stream would run at once and read
the inputs as they were before the writes (zeros, or the cache before it was
filled), so a wrong stream shows as a wrong result, not as a flaky one. Each
result is checked against the oracle: decode and fused-append decode (float64
closed form, 2e-3), prefill (float64 closed form, 2e-3), the GrowingLayer
splice (bit-exact) and the paged prune + decode.
"""
import time

import numpy as np
import pytest
import torch

from oracle import decode as od
from oracle import prefill as opf
from oracle import splice as osp
from threadcut_amd import flash_decode, kv, prefill, workloads
from threadcut_amd.match import Split
from threadcut_amd.paged import PagedKV, new_paged_cache, state_of

pytestmark = pytest.mark.gpu

D = 128
SPIN = 100_000_000  # cycles of torch.cuda._sleep's counter: tens of milliseconds or more


def rnd(shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).half()


def on_side_stream(gpu, fn):
    """Run fn() on a fresh side stream after a spin kernel; return its result once done.
    The stream must still be spinning when fn() has enqueued everything, or a launch on a
    wrong stream could have found its inputs ready."""
    side = torch.cuda.Stream(device=gpu)
    side.wait_stream(torch.cuda.current_stream(gpu))
    with torch.cuda.stream(side):
        torch.cuda._sleep(SPIN)
        out = fn()
    assert not side.query(), "the spin ended before the calls were enqueued"
    side.synchronize()
    return out


def test_decode_and_fused_append_on_a_side_stream(gpu):
    b, hkv, g, n = 2, 8, 4, 3000
    qh, kh, vh = rnd((b, hkv, g, D), 1), rnd((b, hkv, n, D), 2), rnd((b, hkv, n, D), 3)
    qd, kd, vd = qh.to(gpu), kh.to(gpu), vh.to(gpu)
    q = torch.zeros_like(qd)
    kbuf = torch.zeros((b, hkv, n + 16, D), dtype=torch.float16, device=gpu)
    vbuf = torch.zeros_like(kbuf)

    def work():
        q.copy_(qd)
        kbuf[:, :, :n].copy_(kd)
        vbuf[:, :, :n].copy_(vd)
        plain = flash_decode.decode_attention_batched(q, kbuf[:, :, :n], vbuf[:, :, :n], D ** -0.5)
        out = torch.empty_like(q)
        # Append row n - 1 again from k_new / v_new (the same values) and attend n tokens.
        flash_decode.decode_append_into(q, kbuf, vbuf, kbuf[:, :, n - 1].clone(), vbuf[:, :, n - 1].clone(), n,
                                        D ** -0.5, out)
        return plain, out

    plain, fused = on_side_stream(gpu, work)
    want = od.attention_f64(qh.float().numpy(), kh.float().numpy(), vh.float().numpy(), D ** -0.5)
    assert np.abs(plain.float().cpu().numpy() - want).max() <= 2e-3
    assert np.abs(fused.float().cpu().numpy() - want).max() <= 2e-3


def test_prefill_on_a_side_stream(gpu):
    b, hq, hkv, ql, n = 1, 32, 8, 200, 900
    qh, kh, vh = rnd((b, hq, ql, D), 4), rnd((b, hkv, n, D), 5), rnd((b, hkv, n, D), 6)
    mh = (torch.arange(n)[None, :] <= torch.arange(ql)[:, None] + (n - ql))[None, None]
    srcs = [t.to(gpu) for t in (qh, kh, vh, mh)]
    q, k, v, m = (torch.zeros_like(t) for t in srcs)

    def work():
        for dst, src in zip((q, k, v, m), srcs):
            dst.copy_(src)
        return prefill.prefill_attention(q, k, v, m, D ** -0.5)

    out = on_side_stream(gpu, work)
    want = opf.prefill_f64(qh.float().numpy(), kh.float().numpy(), vh.float().numpy(), D ** -0.5, mh.numpy())
    assert np.abs(out.float().cpu().numpy() - want).max() <= 2e-3


def test_splice_on_a_side_stream(gpu):
    n, s = 600, Split(50, 80, 500)
    inv = workloads.inv_freq()
    kh, vh = rnd((1, 8, n, D), 7), rnd((1, 8, n, D), 8)
    kd, vd = kh.to(gpu), vh.to(gpu)
    layer = kv.GrowingLayer()
    layer.update(torch.zeros_like(kd), torch.zeros_like(vd))

    def work():
        layer.kbuf[:, :, :n].copy_(kd)
        layer.vbuf[:, :, :n].copy_(vd)
        layer.splice(s, inv)
        return layer.kbuf[:, :, :n].clone(), layer.vbuf[:, :, :n].clone()

    k_out, v_out = on_side_stream(gpu, work)
    cos, sin = osp.rope_table(-s.gap, inv)
    kw, vw, _ = osp.splice_growing(kh.numpy(), vh.numpy(), n, s.a, s.c0, s.c, cos, sin)
    assert np.array_equal(k_out.cpu().numpy().view(np.uint16), kw.view(np.uint16))
    assert np.array_equal(v_out.cpu().numpy().view(np.uint16), vw.view(np.uint16))


def test_paged_prune_and_decode_on_a_side_stream(gpu):
    n, s = 700, Split(100, 260, 440)
    inv = workloads.inv_freq()
    kh, vh, qh = rnd((8, n, D), 9), rnd((8, n, D), 10), rnd((1, 8, 4, D), 11)
    cache = PagedKV(1, 8, 64, 16, batch=1, device=gpu)
    srcs = [t.to(gpu) for t in (kh, vh, qh)]
    k, v, q = (torch.zeros_like(t) for t in srcs)

    def work():
        for dst, src in zip((k, v, q), srcs):
            dst.copy_(src)
        cache.append(0, [k], [v])
        cache.prune(0, s, inv)
        kg, vg = cache.gather(0)
        return cache.decode(0, q, D ** -0.5), kg, vg

    out, kg, vg = on_side_stream(gpu, work)
    cos, sin = osp.rope_table(-s.gap, inv)
    kw, vw = osp.splice_copy(kh.numpy(), vh.numpy(), s.a, s.c0, s.c, cos, sin)
    assert np.array_equal(kg.cpu().numpy().view(np.uint16), kw.view(np.uint16))
    assert np.array_equal(vg.cpu().numpy().view(np.uint16), vw.view(np.uint16))
    want = od.attention_f64(qh.float().numpy(), kw[None].astype(np.float32), vw[None].astype(np.float32), D ** -0.5)
    assert np.abs(out.float().cpu().numpy() - want).max() <= 2e-3


def running_stream(gpu):
    """A side stream whose work runs now: streams share a few hardware queues, and one behind a spinning stream's
    would wait for it whatever the code under test does."""
    for _ in range(8):
        side = torch.cuda.Stream(device=gpu)
        with torch.cuda.stream(side):
            torch.zeros(1, device=gpu)
        for _ in range(50):
            if side.query():
                return side
            time.sleep(0.001)
    raise AssertionError("every side stream waits for the spinning one")


def zeros_to_reuse(shape, dtype, gpu):
    """Zeroed device memory handed back to the current stream's pool: the next tensor of this size holds zeros until
    it is written."""
    torch.zeros(shape, dtype=dtype, device=gpu)


def test_a_mask_map_on_other_streams(gpu):
    """The tile map of a mask is built on the stream of its first call; a call on another stream that meets the same
    mask does not read it before it is there."""
    b, hq, hkv, ql, n = 1, 32, 8, 200, 900
    q, k, v = (rnd(s, i).to(gpu) for i, s in enumerate(((b, hq, ql, D), (b, hkv, n, D), (b, hkv, n, D))))
    m = (torch.arange(n, device=gpu)[None, :] <= torch.arange(ql, device=gpu)[:, None] + (n - ql))[None, None]
    m[..., 5:90] = False
    want = prefill.prefill_attention(q, k, v, m.clone(), D ** -0.5)
    map_bytes = prefill.mask_tiles(m.clone(), hq, hkv).numel()
    first = torch.cuda.Stream(device=gpu)
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        zeros_to_reuse(map_bytes, torch.uint8, gpu)  # every tile of such a map would be skipped
        torch.cuda._sleep(SPIN)
        a = prefill.prefill_attention(q, k, v, m, D ** -0.5)
    with torch.cuda.stream(running_stream(gpu)):
        got = prefill.prefill_attention(q, k, v, m, D ** -0.5)
        again = prefill.prefill_attention(q, k, v, m, D ** -0.5)
    assert not first.query(), "the spin ended before the calls were enqueued"
    torch.cuda.synchronize()
    assert torch.equal(a, want) and torch.equal(got, want) and torch.equal(again, want)


class TwoLayers:
    num_hidden_layers = 2

    def get_text_config(self, decoder=True):
        return self


def test_paged_slots_on_other_streams(gpu):
    """The slot list of a chunk is uploaded by the first layer's append; another layer's append on another stream
    does not read it before it is there."""
    n = 40
    k = [rnd((1, 8, n, D), i).to(gpu) for i in range(2)]
    cache = new_paged_cache(TwoLayers(), 8, 16)
    for i in range(2):
        cache.update(k[i][:, :, :16], k[i][:, :, :16], i)
    first = torch.cuda.Stream(device=gpu)
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        zeros_to_reuse((1, n, 2), torch.int64, gpu)  # every row of such a list would go to slot 0 of page 0
        torch.cuda._sleep(SPIN)
        cache.update(k[0], k[0], 0)
    with torch.cuda.stream(running_stream(gpu)):
        cache.update(k[1], k[1], 1)
    assert not first.query(), "the spin ended before the calls were enqueued"
    torch.cuda.synchronize()
    for i in range(2):
        gk, gv = state_of(cache).kv.gather(i)
        want = torch.cat((k[i][0, :, :16], k[i][0]), 1)
        assert torch.equal(gk, want) and torch.equal(gv, want)


def test_paged_tables_on_other_streams(gpu):
    """The tile table and the token offsets are uploaded by the first call that reads them; decode and prefill calls
    on another stream do not read them before they are there."""
    n = 300
    k, q, qp = rnd((8, n, D), 1).to(gpu), rnd((1, 8, 4, D), 2).to(gpu), rnd((1, 32, 20, D), 3).to(gpu)
    want = None
    for spin in (0, SPIN):
        cache = PagedKV(1, 8, 24, 16, device=gpu)
        cache.append(0, [k], [k])
        first = torch.cuda.Stream(device=gpu)
        torch.cuda.synchronize()
        with torch.cuda.stream(first):
            if spin:
                torch.cuda._sleep(spin)
            got = [cache.decode(0, q, D ** -0.5), cache.prefill(0, qp, D ** -0.5)]
        if spin:
            with torch.cuda.stream(running_stream(gpu)):
                got += [cache.decode(0, q, D ** -0.5), cache.prefill(0, qp, D ** -0.5)]
            assert not first.query(), "the spin ended before the calls were enqueued"
        torch.cuda.synchronize()
        want = want or got
        for i, x in enumerate(got):
            assert torch.equal(x, want[i % 2])
