"""GPU tests of the F16 / BF16 attention kernels (16 query heads, 2 KV heads, head_dim 256):
against the oracle's float64 attention at block and workgroup edges, and against the
general kernel (reached by rows that are not 16-byte aligned) on rows with infinities and
NaN, in which a product of split operands could end as inf - inf."""
import sys

import numpy as np
import pytest

from attn_checks import assert_attn_close

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

F16, BF16 = 1, 2
QUANTS = [pytest.param(F16, id="f16"), pytest.param(BF16, id="bf16")]


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def pk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import paramecia_amd
    paramecia_amd.lib()
    return paramecia_amd


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def normal(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


@pytest.mark.parametrize("quant", QUANTS)
@pytest.mark.parametrize("B,S", [(1, 0), (1, 1), (1, 31), (1, 32), (2, 33), (1, 64), (3, 65), (1, 700),
                                 (1, 9001), (1, 33000), (33, 40)])
def test_half_decode(pk, orc, B, S, quant):
    """Fused steps (the new row's bytes and the output), then the same keys attended alone."""
    say(f"half decode quant={quant} B={B} S={S}")
    rng = np.random.default_rng(S * 5 + B)
    g = pk.PreallocatedQuantizedKvCache(B, 2, S + 1, 256, pk.KvCacheQuantization(quant))
    c = orc.Cache(quant, B, 2, 256, S + 1)
    k, v, q = normal(rng, B, 2, S + 1, 256), normal(rng, B, 2, S + 1, 256), normal(rng, B, 1, 16, 256)
    k[..., 7] *= 20.0
    v[..., 9] *= 20.0
    q[:, :, 3] *= 1e-3  # rows of unlike size
    if S > 0:
        g.append_quantized(dev(k[:, :, :S]), dev(v[:, :, :S]))
    out = g.append_attend(dev(k[:, :, S:]), dev(v[:, :, S:]), dev(q), 1 / 16)
    assert c.append(k, v) == 0
    ref = c.attend(q, 1 / 16, S, True, mode="f64")
    assert_attn_close(out.cpu().numpy(), ref)
    for a, b in zip(g.raw_bytes(), c.valid_bytes()):
        assert np.array_equal(a.cpu().numpy(), b)
    assert_attn_close(g.attend(dev(q), 1 / 16, S).cpu().numpy(), ref)


@pytest.mark.parametrize("quant", QUANTS)
def test_half_decode_batched(pk, orc, quant):
    """Sequences of 0 to 3000 keys in one call, more of them than a launch takes."""
    say(f"half decode batched quant={quant}")
    run_half_batched(pk, orc, quant, 3000)


@pytest.mark.parametrize("quant", QUANTS)
def test_half_decode_batched_few_partials(pk, orc, quant):
    """At most 700 keys, 22 partials: the combine with one workgroup per head and row."""
    say(f"half decode batched, few partials quant={quant}")
    run_half_batched(pk, orc, quant, 700)


def run_half_batched(pk, orc, quant, most):
    rng = np.random.default_rng(7)
    lens = [0, 1, 32, 33, most, 64] + [int(x) for x in rng.integers(0, 200, 30)]
    caches, refs = [], []
    n = len(lens)
    kn, vn, q = normal(rng, n, 2, 256), normal(rng, n, 2, 256), normal(rng, n, 16, 256)
    for i, S in enumerate(lens):
        g = pk.PreallocatedQuantizedKvCache(1, 2, S + 1, 256, pk.KvCacheQuantization(quant))
        c = orc.Cache(quant, 1, 2, 256, S + 1)
        if S > 0:
            k, v = normal(rng, 1, 2, S, 256), normal(rng, 1, 2, S, 256)
            g.append_quantized(dev(k), dev(v))
            assert c.append(k, v) == 0
        assert c.append(kn[i][None, :, None], vn[i][None, :, None]) == 0
        refs.append(c.attend(q[i][None, None], 1 / 16, S, True, mode="f64")[0, 0])
        caches.append(g)
    out = pk.append_attend_batched(caches, dev(kn), dev(vn), dev(q), 1 / 16).cpu().numpy()
    assert_attn_close(out, np.stack(refs))


@pytest.mark.parametrize("quant", QUANTS)
@pytest.mark.parametrize("B,S,L,causal", [(1, 0, 2, True), (1, 0, 16, True), (1, 0, 17, True), (1, 31, 33, True),
                                          (2, 500, 37, True), (1, 700, 3, False), (1, 9000, 5, True),
                                          (1, 0, 1000, True), (1, 0, 2048, False)])
def test_half_prefill(pk, orc, B, S, L, causal, quant):
    """Chunks at tile and block edges, unsplit and with few and many key splits."""
    say(f"half prefill quant={quant} B={B} S={S} L={L} causal={causal}")
    rng = np.random.default_rng(S + L)
    g = pk.PreallocatedQuantizedKvCache(B, 2, S + L, 256, pk.KvCacheQuantization(quant))
    c = orc.Cache(quant, B, 2, 256, S + L)
    k, v, q = normal(rng, B, 2, S + L, 256), normal(rng, B, 2, S + L, 256), normal(rng, B, L, 16, 256)
    k[..., 7] *= 20.0
    v[..., 9] *= 20.0
    q[:, :, 3] *= 1e-3
    g.append_quantized(dev(k), dev(v))
    assert c.append(k, v) == 0
    out = g.attend(dev(q), 1 / 16, S, causal)
    assert_attn_close(out.cpu().numpy(), c.attend(q, 1 / 16, S, causal, mode="f64"))


def both(pk, quant, k, v, q, q_offset, causal):
    """(outputs of the aligned rows, outputs of the general kernel: the same rows moved by 8 bytes)."""
    S = k.shape[2]
    g = pk.PreallocatedQuantizedKvCache(1, 2, S, 256, pk.KvCacheQuantization(quant))
    g.append_quantized(dev(k), dev(v))
    kp, vp, _, st = g.get_kv_storage()
    kb, vb = g.raw_bytes()
    moved = []
    for x in (kb, vb):
        t = torch.zeros(x.numel() + 64, dtype=torch.uint8, device="cuda")
        t[8:8 + x.numel()] = x
        moved.append(t)
    kq = pk.KvCacheQuantization(quant)
    a = pk.flash_attn(kq, dev(q), kp, vp, st, 1 / 16, 2, S, q_offset, causal)
    b = pk.flash_attn(kq, dev(q), moved[0].data_ptr() + 8, moved[1].data_ptr() + 8, st, 1 / 16, 2, S,
                      q_offset, causal)
    return a.cpu().numpy(), b.cpu().numpy()


@pytest.mark.parametrize("quant", QUANTS)
@pytest.mark.parametrize("what", ["k_inf", "k_nan", "v_inf", "v_nan", "q_inf", "q_big", "last_v_inf"])
@pytest.mark.parametrize("l", [1, 20])
def test_half_nonfinite(pk, quant, what, l):
    """Also of a key that the causal limit hides from most of a chunk's queries."""
    say(f"half non-finite quant={quant} {what} l={l}")
    rng = np.random.default_rng(3)
    S = 333
    k, v, q = normal(rng, 1, 2, S, 256), normal(rng, 1, 2, S, 256), normal(rng, 1, l, 16, 256)
    if what == "k_inf":
        k[0, 0, 100, 5], k[0, 1, 200, 6] = np.inf, -np.inf
    elif what == "k_nan":
        k[0, 0, 100, 5] = np.nan
    elif what == "v_inf":
        v[0, 0, 40, 5], v[0, 1, 300, 9] = np.inf, -np.inf
    elif what == "v_nan":
        v[0, 1, 40, 5] = np.nan
    elif what == "q_inf":
        q[0, 0, 3, 8] = np.inf
    elif what == "q_big":
        q[0, 0, 3] *= 1e37
    else:
        v[0, 0, S - 1, 1] = np.inf
    a, b = both(pk, quant, k, v, q, S - l, True)
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b))
    # finite values: both are within the attention tolerance of the true ones
    np.testing.assert_allclose(a, b, atol=2e-3, rtol=1e-3)


@pytest.mark.parametrize("quant", QUANTS)
@pytest.mark.parametrize("scale", [0.0, -0.1, 1e-3, 4.0])
@pytest.mark.parametrize("l", [1, 18])
def test_half_scales(pk, orc, quant, scale, l):
    """Scales that no model has: none, a negative one (the general kernel), scores that all
    but clamp."""
    say(f"half scale quant={quant} scale={scale} l={l}")
    rng = np.random.default_rng(11)
    S = 70
    g = pk.PreallocatedQuantizedKvCache(1, 2, S, 256, pk.KvCacheQuantization(quant))
    c = orc.Cache(quant, 1, 2, 256, S)
    k, v, q = normal(rng, 1, 2, S, 256), normal(rng, 1, 2, S, 256), normal(rng, 1, l, 16, 256)
    g.append_quantized(dev(k), dev(v))
    assert c.append(k, v) == 0
    out = g.attend(dev(q), scale, S - l).cpu().numpy()
    np.testing.assert_allclose(out, c.attend(q, scale, S - l, True, mode="f64"), atol=2e-3, rtol=1e-3)


@pytest.mark.parametrize("quant", QUANTS)
@pytest.mark.parametrize("S,L", [(12290, 1), (1536, 512), (1000, 1000)])
def test_half_dominant_key(pk, quant, S, L):
    """A first key that outweighs the others by e^14 with a V row of almost nothing: the output
    is made of weights near e^-14, and stays as exact as f32 products make it (measured on the
    general kernel: 4.5e-7, 7.5e-7 for 12290 keys)."""
    say(f"half dominant key quant={quant} S={S} L={L}")
    g = torch.Generator(device="cuda").manual_seed(S + L)
    k = torch.randn((1, 2, S, 256), device="cuda", generator=g)
    v = torch.randn((1, 2, S, 256), device="cuda", generator=g)
    u = torch.randn((2, 256), device="cuda", generator=g)
    k[:, :, 0] = u * (14 * 16 / 256)
    v[:, :, 0] *= 1e-3
    q = 0.2 * torch.randn((1, L, 16, 256), device="cuda", generator=g)
    q += u[torch.arange(16, device="cuda") // 8]
    c = pk.PreallocatedQuantizedKvCache(1, 2, S, 256, pk.KvCacheQuantization(quant))
    c.append_quantized(k, v)
    got = c.attend(q, 1 / 16, S - L).double()
    kd, vd = (x.double() for x in c.get_kv())
    hidden = torch.arange(S, device="cuda") > torch.arange(L, device="cuda")[:, None] + S - L
    err = ref2 = 0.0
    for h in range(16):
        s = (q[0, :, h].double() @ kd[0, h // 8].t() / 16).masked_fill(hidden, -float("inf"))
        ref = torch.softmax(s, -1) @ vd[0, h // 8]
        err += (got[0, :, h] - ref).square().sum().item()
        ref2 += ref.square().sum().item()
    say(f"error {(err / ref2) ** 0.5:.2e}")
    assert (err / ref2) ** 0.5 < 9e-7
