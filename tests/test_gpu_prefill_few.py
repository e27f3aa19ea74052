"""The 4-bit batched product's kernels by size: few tokens (16 or 32 weight rows
a workgroup, K split over its waves, weights staged in LDS by the chunk), and
tiles of 128 columns where they take fewer rounds than tiles of 112."""
import numpy as np
import pytest

from qstream_amd import qsf_format as F
from tests.gpu_util import REL_L2, host, rel_l2, torch_cuda
from tests.test_gpu_prefill import case, run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from qstream_amd import qsf_hip
    qsf_hip.init(0)
    return qsf_hip


# tokens at the row tiles' edges (16 from x as it lies, 32, 64, past 64); one
# unit of K, fewer and more units than waves, a chunk's 64 units and one more,
# all four chunks of a lone workgroup and a fifth, partial blocks of every
# size, weight rows past a tile of 16 and of 32, enough workgroups for two
# weight tiles each, chunks held one (x as it lies) or two at a time by workgroups
# that share a CU
SHAPES = [(1, 15, 32, 64), (16, 17, 64, 64), (17, 33, 72, 64), (15, 16, 512, 64), (32, 31, 576, 64),
          (33, 40, 4096, 64), (64, 20, 4160, 64), (65, 48, 4168, 64), (3, 50, 16384, 64), (5, 18, 16456, 64),
          (40, 18, 20480, 64), (16, 100, 136, 128), (20, 70, 8264, 128), (64, 33, 264, 256), (9, 65, 16648, 256),
          (100, 4100, 128, 64), (130, 2730, 200, 128), (128, 4096, 520, 256), (50, 8200, 4168, 64),
          (16, 4112, 8264, 128), (5, 5000, 12360, 64), (20, 4112, 12360, 64)]


@pytest.mark.parametrize("m,n,k,bs", SHAPES)
def test_few_tokens(hip, oracle, m, n, k, bs):
    """Against the scalar oracle (fp32 sums in another order: the 1e-5 bar)
    and, with the bits, the two halves (pack, then the GEMM)."""
    torch = torch_cuda()
    payload, xb = case(m * 7 + n + k, m, n, k, bs)
    got = run(hip, payload, xb, m, n, k, bs)
    rows = np.unique(np.r_[0:min(n, 40), max(0, n - 40):n])
    rb = ((k + bs - 1) // bs) * (4 + bs // 2)
    sub = b"".join(bytes(payload[r * rb:(r + 1) * rb]) for r in rows)
    err = rel_l2(got[:, rows], oracle.prefill_4bit(np.frombuffer(sub, np.uint8), xb, m, len(rows), k, bs))
    print(f"few tokens {m}x{n}x{k} bs{bs}: rel_l2 {err:.3e}")
    assert err <= REL_L2
    assert np.isfinite(got).all()
    t = hip.Tensor(payload, F.Q4, n, k, bs)
    dx = torch.from_numpy(xb.view(np.int16).copy()).to("cuda:0")
    packed = torch.full((hip.prefill_pack_bytes(m, k, bs) + 256,), 255, dtype=torch.uint8, device="cuda:0")
    y = torch.full((m, n), float("nan"), device="cuda:0")
    addr = (packed.data_ptr() + 255) & ~255
    hip.prefill_pack(dx, m, k, bs, addr, stream=torch.cuda.current_stream())
    t.prefill_packed(addr, m, y, stream=torch.cuda.current_stream())
    assert np.array_equal(host(y).view(np.uint32), got.view(np.uint32))
    t.free()


@pytest.mark.parametrize("m", [9, 24, 48])
@pytest.mark.parametrize("bs", [64, 128])
def test_special_values(hip, m, bs):
    """Inf and NaN of x stay in their token; a block whose scale or zero is
    Inf or NaN stays in its row (also where it is the row's last)."""
    n, k = 40, 1096
    payload, xb = case(m, m, n, k, bs)
    clean = run(hip, payload, xb, m, n, k, bs)
    xs = xb.copy()
    xs[1, 5], xs[4, k - 1] = 0x7F80, 0x7FC0
    p = np.frombuffer(payload, np.uint8).copy()
    nb, bb = (k + bs - 1) // bs, 4 + bs // 2
    for row, b, off in ((3, 0, 0), (17, nb - 1, 2)):
        at = (row * nb + b) * bb + off
        p[at:at + 2] = np.frombuffer(np.uint16(0x7C00 if off else 0x7E00).tobytes(), np.uint8)
    got = run(hip, p, xs, m, n, k, bs)
    keep_t = [t for t in range(m) if t not in (1, 4)]
    keep_r = [r for r in range(n) if r not in (3, 17)]
    assert not np.isfinite(got[[1, 4]]).any()
    assert not np.isfinite(got[np.ix_(keep_t, [3, 17])]).any()
    assert np.array_equal(got[np.ix_(keep_t, keep_r)].view(np.uint32), clean[np.ix_(keep_t, keep_r)].view(np.uint32))


@pytest.mark.parametrize("off,m", [(0, 2), (2, 2), (0, 40), (2, 40)])
@pytest.mark.parametrize("k,bs", [(64, 64), (576, 64), (4160, 64), (136, 128), (264, 256), (512, 256)])
def test_infinite_last_block(hip, k, bs, off, m):
    """A last block whose scale or zero is Inf gives Inf, as the scalar matvec
    does for x > 0 and codes > 0, whatever the row's unit count leaves of a
    round of the waves (units past the row add nothing, not Inf * 0)."""
    n = 20
    payload, _ = case(k, m, n, k, bs)
    xb = np.full((m, k), 0x3F80, np.uint16)                     # 1.0
    p = np.frombuffer(payload, np.uint8).copy()
    nb, bb = (k + bs - 1) // bs, 4 + bs // 2
    blocks = p[:n * nb * bb].reshape(n, nb, bb)
    blocks[5, nb - 1, 4:] |= 0x11                               # codes of at least 1
    blocks[5, nb - 1, off:off + 2] = np.frombuffer(np.uint16(0x7C00).tobytes(), np.uint8)
    got = run(hip, p, xb, m, n, k, bs)
    assert np.isposinf(got[:, 5]).all()
    assert np.isfinite(np.delete(got, 5, axis=1)).all()


# shapes whose tiles of 112 need a second round of 256 workgroups and whose
# tiles of 128 do not: full and partial last tiles both ways, every block
# size, ragged k, rows of more blocks than the wide tile's zero stash holds
@pytest.mark.parametrize("m,n,k,bs", [(1999, 4096, 264, 64), (2048, 4081, 512, 128), (2000, 4000, 328, 256),
                                      (4096, 2000, 21760, 64)])
def test_wide_tiles(hip, oracle, m, n, k, bs):
    payload, xb = case(m + n + k, m, n, k, bs)
    got = run(hip, payload, xb, m, n, k, bs)
    assert np.isfinite(got).all()
    rows = np.unique(np.r_[0, 111, 112, 127, 128, 255, 256, n - 130:n - 126, n - 1])
    toks = np.unique(np.r_[0:4, 255:258, m - 3:m])
    rb = ((k + bs - 1) // bs) * (4 + bs // 2)
    sub = b"".join(bytes(payload[r * rb:(r + 1) * rb]) for r in rows)
    ref = oracle.prefill_4bit(np.frombuffer(sub, np.uint8), np.ascontiguousarray(xb[toks]), len(toks), len(rows), k, bs)
    err = rel_l2(got[np.ix_(toks, rows)], ref)
    print(f"wide tiles {m}x{n}x{k} bs{bs}: rel_l2 {err:.3e}")
    assert err <= REL_L2


# (rows, tokens, tile): one round of tiles of 128 columns against two of 112 (the
# tile kernel from 257 to 320 tokens), 2 M tiles of them, and sizes beside them
# that the few-token kernel keeps (its workgroups cost less than a round)
@pytest.mark.parametrize("n,m,tile", [(16384, 257, True), (16384, 320, True), (14337, 257, True), (32768, 128, True),
                                      (14336, 128, False), (4096, 257, False), (8192, 320, False)])
def test_few_or_tile(hip, n, m, tile):
    """Which kernel took a call, by its bits: those of the first m tokens of a
    call too large for the few-token kernel, or not."""
    k, bs, most = 328, 64, 1030
    payload, xb = case(n + m, most, n, k, bs)
    got = run(hip, payload, xb[:m], m, n, k, bs)
    ref = run(hip, payload, xb, most, n, k, bs)[:m]
    assert rel_l2(got, ref) <= REL_L2
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)) == tile
