"""The prefill kernel's work-group shapes (128 or 64 query rows, one, two or four key groups whose partial results
are merged in LDS) at the sizes where each is chosen and at the edges of their tiles, against plain attention in
float64 on the same device.

Tolerance: P and the output are rounded to the storage type, so an output of size |o| <= max|v| is off by at most
about two roundings, 2 * 2^-11 * |o| in fp16 (2 * 2^-8 in bf16); with N(0, 1) values |o| stays below 4 except
where a row sees a few keys, where it is one value of V and |v| < 6: 6e-3 and 4.7e-2 at worst, and 2e-3 of the
outputs' norm (1.6e-2 in bf16)."""
import pytest
import torch

from threadcut_amd import _lib, paged, prefill, workloads

pytestmark = pytest.mark.gpu
SCALE = 128 ** -0.5


def reference(q, k, v, vis, scale):
    b, hq, ql, _ = q.shape
    g = hq // k.shape[1]
    out = torch.zeros(b, ql, hq, 128, dtype=torch.float64, device=q.device)
    for i in range(b):
        for h in range(hq):
            s = q[i, h].double() @ k[i, h // g].double().t() * scale
            s = s.masked_fill(~vis[i if vis.shape[0] > 1 else 0], float("-inf"))
            out[i, :, h] = torch.softmax(s, -1).nan_to_num() @ v[i, h // g].double()
    return out


def masks(mode, ql, n, b, dev, seed):
    """(mask or None, visible [b|1, ql, n])."""
    g = torch.Generator(device=dev).manual_seed(seed)
    causal = workloads.causal_mask(ql, n, device=dev)
    if mode == "causal":
        return None, causal[0]
    if mode == "none":
        return None, torch.ones(1, ql, n, dtype=torch.bool, device=dev)
    if mode == "chunk":
        return causal.contiguous(), causal[0]
    if mode == "padded":  # hides whole tiles, and every key of some rows
        pads = torch.randint(0, max(1, n - ql // 2), (b,), generator=g, device=dev)
        m = causal & (torch.arange(n, device=dev)[None, :] >= pads[:, None])[:, None, None, :]
    else:  # holes: every tile tested key by key
        m = causal & (torch.rand(b, 1, ql, n, generator=g, device=dev) < 0.8)
    return m.contiguous(), m[:, 0]


def check(out, want, dtype):
    tol = (6e-3, 2e-3) if dtype == torch.float16 else (4.7e-2, 1.6e-2)
    d = out.double() - want
    assert torch.isfinite(out.float()).all()
    assert d.abs().max().item() <= tol[0] and d.norm().item() <= tol[1] * max(want.norm().item(), 1e-30)


# (q_heads, kv_heads, queries, keys): which shape 256 compute units give, at and around its tiles' edges.
SIZES = [
    (32, 8, 1, 1), (32, 8, 17, 33), (8, 2, 64, 64), (16, 8, 200, 257), (64, 8, 300, 639),    # 64 rows, two key groups
    (32, 8, 14, 43), (8, 8, 1, 64), (16, 2, 9, 65), (32, 4, 31, 320),                        # (chunks on a few keys)
    (16, 8, 700, 700), (8, 8, 127, 641), (32, 8, 5, 3000), (8, 2, 93, 4097), (64, 8, 8, 2111),  # 64 rows, four
    (32, 4, 31, 321),
    (32, 8, 1100, 1100), (32, 8, 100, 5000), (64, 8, 129, 4223), (8, 8, 1500, 7000),         # 128 rows, two
    (16, 8, 1300, 1300),                                                                     # (W64 = 1.3 C, W < C)
    (64, 8, 1030, 1030), (32, 8, 600, 5001),                                                 # 128 rows, one
]


@pytest.mark.parametrize("mode", ["causal", "none", "chunk", "padded", "holes"])
@pytest.mark.parametrize("hq,hkv,ql,n", SIZES)
def test_shapes(gpu, hq, hkv, ql, n, mode):
    dtype = torch.bfloat16 if (ql + n) % 3 == 0 else torch.float16
    b = 2 if mode == "padded" else 1
    if mode == "causal" and 2 * ql < n:
        mode = "chunk"
    print(f"case: {hq}/{hkv} q={ql} n={n} {mode} {dtype}", flush=True)
    q, k, v = workloads.prefill_inputs(ql + n, batch=b, q_len=ql, n=n, q_heads=hq, kv_heads=hkv, dtype=dtype, device=gpu)
    m, vis = masks(mode, ql, n, b, gpu, n)
    out = prefill.prefill_attention(q, k, v, m, SCALE, mode == "causal")
    check(out, reference(q, k, v, vis, SCALE), dtype)


@pytest.mark.parametrize("mode", ["causal", "padded"])
@pytest.mark.parametrize("hq,hkv,ql,n,b", [(8, 2, 300, 300, 5), (32, 8, 700, 900, 3), (64, 16, 290, 290, 9),
                                           (16, 16, 150, 1100, 7), (32, 32, 130, 650, 6)])
def test_batches(gpu, hq, hkv, ql, n, b, mode):
    """Several sequences, in both orders of their blocks: prompts of few and of many rounds, and chunks."""
    if mode == "causal" and 2 * ql < n:
        mode = "chunk"
    q, k, v = workloads.prefill_inputs(ql + b, batch=b, q_len=ql, n=n, q_heads=hq, kv_heads=hkv, dtype=torch.float16,
                                       device=gpu)
    m, vis = masks(mode, ql, n, b, gpu, n)
    out = prefill.prefill_attention(q, k, v, m, SCALE, mode == "causal")
    check(out, reference(q, k, v, vis, SCALE), torch.float16)


@pytest.mark.parametrize("splits", [2, 3, 5, 9, 17, 32, 40])
@pytest.mark.parametrize("hq,hkv,ql,n", [(32, 8, 5, 3000), (32, 8, 100, 5000), (16, 8, 200, 257), (32, 8, 600, 5001)])
def test_split_counts(gpu, hq, hkv, ql, n, splits):
    """Every combine (compiled for a few counts) with splits that end inside a tile, and empty ones."""
    q, k, v = workloads.prefill_inputs(splits, q_len=ql, n=n, q_heads=hq, kv_heads=hkv, device=gpu)
    for mode in ("chunk", "holes"):
        m, vis = masks(mode, ql, n, 1, gpu, splits)
        out = prefill.prefill_attention(q, k, v, m, SCALE, splits=splits)
        check(out, reference(q, k, v, vis, SCALE), torch.float16)


@pytest.mark.parametrize("hq,hkv", [(3, 3), (6, 3), (20, 5), (56, 7)])
@pytest.mark.parametrize("b,ql", [(1, 2), (2, 9), (1, 77)])
def test_combine_of_odd_heads_and_rows(gpu, hq, hkv, b, ql):
    """Eight rows of one KV head per combine work-group: the last group of a head is partly empty."""
    n = 2500
    q, k, v = workloads.prefill_inputs(ql, batch=b, q_len=ql, n=n, q_heads=hq, kv_heads=hkv, dtype=torch.float16, device=gpu)
    m, vis = masks("chunk", ql, n, b, gpu, n)
    assert prefill.num_splits(b, ql, n, hq, hkv) > 1
    check(prefill.prefill_attention(q, k, v, m, SCALE, False), reference(q, k, v, vis, SCALE), torch.float16)


@pytest.mark.parametrize("hq,hkv,ql,n", [(16, 8, 200, 257), (32, 8, 5, 3000), (32, 8, 100, 5000), (32, 8, 1100, 1100)])
@pytest.mark.parametrize("P", [16, 48, 64])
def test_paged_shapes(gpu, hq, hkv, ql, n, P):
    """Through the pools (pages out of order, from a partly filled one): the contiguous kernel's bits."""
    q, k, v = workloads.prefill_inputs(P + n, q_len=ql, n=n, q_heads=hq, kv_heads=hkv, device=gpu)
    cache = paged.PagedKV(1, hkv, -(-n // P) + 3, P, device=gpu)
    cache.table.free = cache.table.free[::2] + cache.table.free[1::2]
    for lo, hi in ((0, 3), (3, n // 3), (n // 3, n)):
        cache.append(0, [k[0, :, lo:hi]], [v[0, :, lo:hi]])
    for mode in ("chunk", "padded", "holes"):
        m, _ = masks(mode, ql, n, 1, gpu, n + P)
        assert torch.equal(cache.prefill(0, q, SCALE, m), prefill.prefill_attention(q, k, v, m, SCALE))


@pytest.mark.parametrize("scale", [0.0, -0.1, 0.5])
@pytest.mark.parametrize("hq,hkv,ql,n", [(16, 8, 200, 257), (32, 8, 5, 3000), (32, 8, 100, 5000), (64, 8, 1030, 1030)])
def test_scales(gpu, hq, hkv, ql, n, scale):
    """A scale of 0 averages the visible values; a negative one flips the order."""
    q, k, v = workloads.prefill_inputs(n, q_len=ql, n=n, q_heads=hq, kv_heads=hkv, device=gpu)
    for mode in ("chunk", "holes"):
        m, vis = masks(mode, ql, n, 1, gpu, 3)
        check(prefill.prefill_attention(q, k, v, m, scale), reference(q, k, v, vis, scale), torch.float16)


@pytest.mark.parametrize("hq,hkv,ql,n", [(16, 8, 200, 257), (32, 8, 5, 3000), (32, 8, 100, 5000), (64, 8, 1030, 1030)])
def test_nonfinite_keys_stay_hidden(gpu, hq, hkv, ql, n):
    """Infinite or NaN keys that no row sees change nothing; one that a row sees makes that row NaN."""
    q, k, v = workloads.prefill_inputs(n + 1, q_len=ql, n=n, q_heads=hq, kv_heads=hkv, device=gpu)
    m, _ = masks("chunk", ql, n, 1, gpu, 0)
    m[..., 7] = False
    want = prefill.prefill_attention(q, k, v, m, SCALE)
    k2 = k.clone()
    k2[:, :, 7] = float("nan")
    assert torch.equal(prefill.prefill_attention(q, k2, v, m, SCALE), want)
    k2[:, :, 7] = float("inf")
    assert torch.equal(prefill.prefill_attention(q, k2, v, m, SCALE), want)
    m[..., -1, 7] = True
    got = prefill.prefill_attention(q, k2, v, m, SCALE)
    assert torch.equal(got[:, :-1], want[:, :-1]) and torch.isnan(got[:, -1]).all()


@pytest.mark.parametrize("pad", [0, 1, 2])
def test_strided_rows_and_mask_views(gpu, pad):
    """Token strides wider than a row, K and V strides that differ, a mask view that is not word-aligned."""
    ql, n = 150, 700
    g = torch.Generator(device=gpu).manual_seed(pad)
    r = lambda *s: torch.randn(s, generator=g, device=gpu).half()
    k = r(1, n, 4, 128 + 64)[..., :128].transpose(1, 2)
    v = r(1, n, 4, 128 + 8 * pad)[..., :128].transpose(1, 2)
    q = r(1, ql, 16, 256)[..., 8:136].transpose(1, 2)
    m = (torch.rand(1, 1, ql, n + pad, generator=g, device=gpu) < 0.7)[..., pad:]
    out = torch.zeros(1, ql, 20, 128, device=gpu, dtype=torch.float16)
    prefill.prefill_attention(q, k, v, m, SCALE, out=out[:, :, 2:18])
    check(out[:, :, 2:18], reference(q, k, v, m[:, 0], SCALE), torch.float16)
    assert not out[:, :, :2].any() and not out[:, :, 18:].any()


@pytest.mark.parametrize("ql,n,b,off", [(1, 1, 1, 0), (7, 513, 2, 1), (33, 64, 1, 3), (130, 1500, 3, 2), (40, 511, 1, 0),
                                        (64, 1025, 2, 5)])
@pytest.mark.parametrize("hq", [8, 16, 32, 64])
def test_mask_map(gpu, ql, n, b, off, hq):
    """The tile map of masks at any alignment: full, empty, causal and mixed tiles, rows and keys past the ends."""
    tokens, T = 128 // (hq // 8), -(-n // 64)
    g = torch.Generator(device=gpu).manual_seed(n)
    m = torch.zeros(b, 1, ql, n + off, dtype=torch.bool, device=gpu)[..., off:]
    m[:] = workloads.causal_mask(ql, n, device=gpu)
    m[:, :, ql // 2:, : n // 2] = True
    m[-1, :, :, : n // 3] = False
    m[0, :, :, -1] |= torch.rand(1, ql, generator=g, device=gpu) < 0.5
    got = prefill.mask_tiles(m, hq, 8).cpu()
    pitch = -(-T // 8) * 8
    got = got.reshape(b, -1, pitch)
    causal = workloads.causal_mask(ql, n)[0, 0]
    for i in range(b):
        for blk in range(got.shape[1]):
            rows = slice(blk * tokens, min(ql, (blk + 1) * tokens))
            for t in range(pitch):
                x, c = m[i, 0, rows, 64 * t:64 * t + 64].cpu(), causal[rows, 64 * t:64 * t + 64]
                want = 0 if not x.any() else 1 if x.shape[1] == 64 and x.all() else 3 if torch.equal(x, c) else 2
                assert got[i, blk, t] == want, (i, blk, t)


@pytest.mark.parametrize("hq,hkv,ql,n", [(32, 8, 1, 1026), (32, 8, 3, 9000), (8, 2, 93, 4097), (32, 8, 100, 5000),
                                         (16, 8, 200, 257)])
def test_library_chosen_splits_need_the_workspace_the_query_tells(gpu, hq, hkv, ql, n):
    """With num_splits 0 the call takes the splits of tc_prefill_num_splits, also for K/V whose rows lie too far
    apart for one 32-bit range: the workspace of that count is enough, and all of it is needed."""
    lib = _lib.load()
    q, k, v = workloads.prefill_inputs(n, q_len=ql, n=n, q_heads=hq, kv_heads=hkv, device=gpu)
    m, vis = masks("chunk", ql, n, 1, gpu, 0)
    want = reference(q, k, v, vis, SCALE)
    s = lib.tc_prefill_num_splits(1, ql, n, hq, hkv)
    need = lib.tc_prefill_workspace_bytes(1, ql, hq, s)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=gpu)
    stream = torch.cuda.current_stream().cuda_stream
    wide = -(-2 ** 30 // (n + 128) // 8) * 8  # elements between tokens: just past 2^31 bytes for n + 128 rows
    far = torch.zeros(2, n * wide, dtype=torch.float16, device=gpu).as_strided((2, hkv, n, 128), (n * wide, 128, wide, 1))
    far[0], far[1] = k[0], v[0]
    for kk, vv in ((k[0], v[0]), (far[0], far[1])):
        for bytes_given in (need, need - 16):
            out = torch.empty(1, ql, hq, 128, dtype=torch.float16, device=gpu)
            rc = lib.tc_prefill_attention(
                q.data_ptr(), _lib.i64x3(0, q.stride(1), q.stride(2)), kk.data_ptr(), _lib.i64x3(0, kk.stride(0), kk.stride(1)),
                vv.data_ptr(), _lib.i64x3(0, vv.stride(0), vv.stride(1)), None, None, None, 0, 1, ql, n, 1, hq, hkv, 128,
                _lib.TC_DTYPE_F16, SCALE, 0, ws.data_ptr(), max(bytes_given, 0), out.data_ptr(),
                _lib.i64x3(0, hq * 128, 128), stream)
            if bytes_given < need and s > 1:
                assert rc == _lib.TC_ERR_WORKSPACE
            else:
                assert rc == _lib.TC_OK, lib.tc_last_error()
                check(out, want, torch.float16)


def test_masks_made_in_inference_mode(gpu):
    """Such a mask has no version counter: each call classifies it as it is then."""
    hq, hkv, ql, n = 32, 8, 100, 900
    q, k, v = workloads.prefill_inputs(4, q_len=ql, n=n, q_heads=hq, kv_heads=hkv, device=gpu)
    with torch.inference_mode():
        m, vis = masks("chunk", ql, n, 1, gpu, 0)
        check(prefill.prefill_attention(q, k, v, m, SCALE), reference(q, k, v, vis, SCALE), torch.float16)
        m[..., 100:500] = False
        check(prefill.prefill_attention(q, k, v, m, SCALE), reference(q, k, v, m[:, 0], SCALE), torch.float16)
