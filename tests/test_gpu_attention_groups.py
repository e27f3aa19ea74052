"""Attention with several query heads of a KV head in one workgroup: the
heads a workgroup takes (4, 2 or 1) follow the group size and the number of
workgroups; the chunk merge takes up to 128 chunks."""
import numpy as np
import pytest

from tests.gpu_util import REL_L2, dev, host, rel_l2, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from qstream_amd import qsf_hip
    qsf_hip.init(0)
    return qsf_hip


def _s():
    return torch_cuda().cuda.current_stream()


# (heads, KV heads, head_dim, position): 4, 2 and 1 heads a workgroup at each
# head_dim, a group of 6 (2 at a time) and of 3 (1), a partial last chunk,
# the new row at a chunk's first and last place, one chunk more than a wave
# merges at once (65 chunks) and the longest cache (128 chunks)
SHAPES = [(32, 8, 128, 4099), (32, 8, 64, 4096), (64, 16, 256, 2047), (16, 8, 128, 4223), (16, 8, 64, 4100),
          (16, 8, 256, 4100), (12, 2, 128, 8320), (24, 8, 128, 1500), (8, 8, 128, 8191), (8, 2, 64, 16383),
          (32, 8, 128, 2000)]


@pytest.mark.parametrize("nh,nkv,hd,position", SHAPES)
def test_grouped_heads(hip, oracle, nh, nkv, hd, position):
    """Against the scalar oracle (fp32 sums in another order: the 1e-5 bar),
    each KV head's own call (one head a workgroup: the same bits, a head's
    arithmetic does not depend on its company), and the fused RoPE + store
    (the same bits as the separate calls)."""
    torch = torch_cuda()
    rng = np.random.default_rng(nh + hd + position)
    max_seq = position + 1
    kc = rng.integers(-127, 128, (nkv, max_seq, hd)).astype(np.int8)
    vc = rng.integers(-127, 128, (nkv, max_seq, hd)).astype(np.int8)
    ks = (rng.random((nkv, max_seq)) * 0.02).astype(np.float32)
    vs = (rng.random((nkv, max_seq)) * 0.02).astype(np.float32)
    q = rng.standard_normal(nh * hd).astype(np.float32)
    k, v = (rng.standard_normal(nkv * hd).astype(np.float32) for _ in range(2))
    out = torch.full((nh * hd,), np.nan, device="cuda:0")
    hip.attention(dev(q), dev(kc), dev(vc), dev(ks), dev(vs), max_seq, nh, nkv, hd, position, out, stream=_s())
    got = host(out)
    err = rel_l2(got, oracle.attention(q, kc, vc, ks, vs, max_seq, nh, nkv, hd, position))
    print(f"attention nh {nh} nkv {nkv} hd {hd} pos {position}: rel_l2 {err:.2e}")
    assert err <= REL_L2
    g = nh // nkv
    for h in (0, nkv - 1):
        one = torch.full((g * hd,), np.nan, device="cuda:0")
        hip.attention(dev(q[h * g * hd:(h + 1) * g * hd]), dev(kc[h]), dev(vc[h]), dev(ks[h]), dev(vs[h]), max_seq,
                      g, 1, hd, position, one, stream=_s())
        assert np.array_equal(host(one).view(np.uint32), got[h * g * hd:(h + 1) * g * hd].view(np.uint32))
    rope = hip.Rope(hd, 10000.0)
    outs = []
    for fused in (False, True):
        dq, dk, dv = dev(q), dev(k), dev(v)
        a = [dev(x.copy()) for x in (kc, vc, ks, vs)]
        o = torch.full((nh * hd,), np.nan, device="cuda:0")
        if fused:
            rope.apply_store_attend(dq, dk, dv, nh, nkv, position, *a, max_seq, o, stream=_s())
        else:
            rope.apply_and_store(dq, dk, dv, nh, nkv, position, *a, max_seq, stream=_s())
            hip.attention(dq, *a, max_seq, nh, nkv, hd, position, o, stream=_s())
        outs.append([host(x).view(np.uint8) for x in (*a, o)])
    rope.free()
    for name, x, y in zip(("kc", "vc", "ks", "vs", "out"), *outs):
        assert np.array_equal(x, y), name


@pytest.mark.parametrize("nh,nkv,hd,position", [(8, 2, 128, 300), (4, 4, 64, 127), (8, 1, 256, 4223), (32, 8, 128, 4100)])
def test_large_queries_and_infinite_scales(hip, oracle, nh, nkv, hd, position):
    """Queries whose products with the codes alone pass fp32's range while those
    with the dequantised row do not (plain call, and the fused one, whose new
    row of 1e-29 takes most heads' weight or none of it), and an Inf scale over a row with a zero code: NaN for the
    heads of that KV head, the others untouched."""
    torch = torch_cuda()
    rng = np.random.default_rng(hd + position)
    max_seq, g = position + 1, nh // nkv
    kc = rng.integers(-127, 128, (nkv, max_seq, hd)).astype(np.int8)
    vc = rng.integers(-127, 128, (nkv, max_seq, hd)).astype(np.int8)
    tiny = np.float32(2.0) ** np.float32(-120)
    ks = (rng.random((nkv, max_seq)) * 0.02).astype(np.float32) * tiny
    vs = (rng.random((nkv, max_seq)) * 0.02).astype(np.float32)
    q = rng.standard_normal(nh * hd).astype(np.float32) / tiny
    out = torch.full((nh * hd,), np.nan, device="cuda:0")
    hip.attention(dev(q), dev(kc), dev(vc), dev(ks), dev(vs), max_seq, nh, nkv, hd, position, out, stream=_s())
    got = host(out)
    assert np.isfinite(got).all()
    assert rel_l2(got, oracle.attention(q, kc, vc, ks, vs, max_seq, nh, nkv, hd, position)) <= REL_L2

    rope = hip.Rope(hd, 10000.0)
    k, v = (rng.standard_normal(nkv * hd).astype(np.float32) * np.float32(0.3) for _ in range(2))
    dq, dk, dv = dev(q), dev(k * np.float32(1e-29)), dev(v)
    a = [dev(x.copy()) for x in (kc, vc, ks, vs)]
    outs = []
    for fused in (False, True):
        b, o = [x.clone() for x in a], torch.full((nh * hd,), np.nan, device="cuda:0")
        q2, k2 = dq.clone(), dk.clone()
        if fused:
            rope.apply_store_attend(q2, k2, dv, nh, nkv, position, *b, max_seq, o, stream=_s())
        else:
            rope.apply_and_store(q2, k2, dv, nh, nkv, position, *b, max_seq, stream=_s())
            hip.attention(q2, *b, max_seq, nh, nkv, hd, position, o, stream=_s())
        outs.append(host(o))
    rope.free()
    assert np.isfinite(outs[0]).all() and np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))

    q, ks, p = q * tiny, ks / tiny, position // 2
    clean = torch.full((nh * hd,), np.nan, device="cuda:0")
    hip.attention(dev(q), dev(kc), dev(vc), dev(ks), dev(vs), max_seq, nh, nkv, hd, position, clean, stream=_s())
    kc[0, p, 3], ks[0, p] = 0, np.inf
    hip.attention(dev(q), dev(kc), dev(vc), dev(ks), dev(vs), max_seq, nh, nkv, hd, position, out, stream=_s())
    got = host(out)
    assert np.isnan(oracle.attention(q, kc, vc, ks, vs, max_seq, nh, nkv, hd, position)[:g * hd]).all()
    assert np.isnan(got[:g * hd]).all()
    assert np.array_equal(got[g * hd:].view(np.uint32), host(clean)[g * hd:].view(np.uint32))
