"""The f32-out H-TILE kernels weight by weight: x rows with a single nonzero element, so each output
is one product, RN(cell * absmax) x, bit for bit. A sum's bound cannot see a plane of the weights
that is lost or read from the wrong word (2^-16 of a weight hides in (K + 2) 2^-23 sum |w x|); this
does. Every k of K is taken once: each lane group, MFMA step, 64-block, chunk, K split and wave's part,
the half last chunk at K % 128 == 64, partial chunks, odd rows.

The element is 1 or, with scales around 2^100, the smallest normal BF16: sums of cells times x
formed before the scale is applied would lose bits there. A subnormal x is less exact (the matrix
core aligns its products as if x were 2^-126): its sums are checked with |x| taken as at least that."""
import numpy as np
import pytest

from glint_amd import glint_hip as H
from oracle import glint_oracle as G
from tests.gpu_util import dev, host, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiny", [False, True])
@pytest.mark.parametrize("M,N,K,bs", [
    # k_htile_rl3 with one, two and four 16-row blocks of x, K split and a half-used last line
    (8, 130, 1152, 64), (32, 70, 640, 64), (64, 130, 1152, 64),
    # k_htile_f3 on 64- and 128-row tiles, whole and half last chunks, split and not
    (65, 130, 1152, 64), (128, 24576, 256, 64), (16, 130, 704, 64), (100, 300, 320, 64), (128, 24576, 192, 64),
    # k_htile_any: even and odd K, blocks from 32 and below, one to eight waves with chunks, two strips
    (5, 33, 1160, 64), (7, 33, 1161, 32), (20, 20, 400, 20), (17, 17, 401, 7), (33, 50, 264, 48), (64, 40, 1031, 33),
    (130, 4111, 264, 64), (130, 4111, 265, 128)])
def test_single_products(M, N, K, bs, tiny):
    print(f"htile single products M={M} N={N} K={K} bs={bs} tiny={tiny}", flush=True)
    rng = np.random.default_rng(M + N + K + bs)
    n = N * K
    hole, plug = (rng.integers(0, 256, (n + 1) // 2, dtype=np.uint8) for _ in range(2))
    am = rng.uniform(0.01, 1.0, (n + bs - 1) // bs).astype(np.float32)
    one, val = 0x3F80, 1.0
    if tiny:
        am, one, val = (am * np.float32(2.0 ** 100)).astype(np.float32), 0x0080, 2.0 ** -126
    w = G.expand(hole, plug, am, n, bs).reshape(N, K)  # f32 products
    pin = [dev(a) for a in (hole, plug, am)]
    for k0 in range(0, K, M):
        ks = (k0 + np.arange(M)) % K
        x = np.zeros((M, K), np.uint16)
        x[np.arange(M), ks] = one
        y = host(H.htile_f32(*pin, dev(x).reshape(M, K), N, K, bs)).reshape(M, N)
        want = (w[:, ks].T.astype(np.float64) * val).astype(np.float32)  # a power of two: exact
        assert np.array_equal(y, want), (k0, np.abs(y / want - 1).max())


@pytest.mark.parametrize("M,N,K,bs", [(8, 130, 256, 64), (32, 70, 128, 64), (64, 130, 384, 64), (65, 130, 128, 64),
                                      (128, 24576, 128, 64), (9, 300, 64, 64), (100, 300, 192, 64), (20, 20, 130, 32)])
def test_subnormal_x_under_large_scales(oracle, M, N, K, bs):
    """BF16 subnormals and numbers just above, scales around 2^100: K additions, each rounded to at
    most 2^-23 of sum |w| max(|x|, 2^-126)."""
    print(f"htile small x M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M + N + K)
    hole, plug = (rng.integers(0, 256, N * K // 2, dtype=np.uint8) for _ in range(2))
    am = (rng.uniform(0.01, 1.0, N * K // bs + 1) * 2.0 ** 100).astype(np.float32)
    x = (rng.integers(0, 0x0200, M * K) | (rng.integers(0, 2, M * K) << 15)).astype(np.uint16)
    y = host(H.htile_f32(dev(hole), dev(plug), dev(am), dev(x).reshape(M, K), N, K, bs)).reshape(M, N)
    ref, _ = (a.reshape(M, N) for a in oracle.htile_f64(hole, plug, am, x, M, N, K, bs))
    up = np.maximum(x & 0x7FFF, 0x0080).astype(np.uint16)
    _, asum = (a.reshape(M, N) for a in oracle.htile_f64(hole, plug, am, up, M, N, K, bs))
    assert (np.abs(y - ref) <= (K + 2) * 2.0 ** -23 * asum).all()


@pytest.mark.parametrize("N", [70, 8200])
def test_single_products_m1_tiles(N):
    """M = 1 beyond the GEMV's K: 64 x 64 tiles, and 64 x 128 ones where those fill the CUs; k at the
    ends of a 64-wide step, of a K split and between."""
    torch = torch_cuda()
    K = 32832
    print(f"htile single products M=1 N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(N)
    hole, plug = (torch.randint(0, 256, (N * K // 2,), dtype=torch.uint8, device="cuda", generator=g) for _ in range(2))
    am = torch.rand(N * K // 64, device="cuda", generator=g) + 0.01
    for k in (0, 1, 31, 32, 63, 64, 8191, 8192, 8255, 8256, 16448, 20000, 24639, 32767, 32768, 32831):
        x = torch.zeros(K, dtype=torch.bfloat16, device="cuda")
        x[k] = 1.0
        i = torch.arange(N, device="cuda") * K + k
        h, p = (((t[i >> 1] >> (4 * (k & 1))) & 15).cpu().numpy() for t in (hole, plug))
        want = G.CELLS_F32[h, p] * am[i // 64].cpu().numpy()
        assert np.array_equal(host(H.htile_f32(hole, plug, am, x, N, K, 64)).reshape(-1), want), k
