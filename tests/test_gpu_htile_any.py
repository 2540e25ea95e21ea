"""k_htile_any: the H-TILE linear of every shape the aligned kernels do not take.

Both outputs against the oracle's float64 sum within (K + 2) 2^-23 sum |w x| (every product
is exact; the sum has at most K f32 roundings, each below half an ulp of a partial sum that
sum |w x| bounds; a factor of 2 covers the matrix core's own addition order), BF16 out with
half a BF16 ulp of the value on top. Sizes at the edges of a 128-wide chunk, of the 8 waves'
shares, of the 16-row strips and of the 16-, 32- and 64-row blocks of x; odd K, where rows
start in the middle of a byte; blocks below, at and above the 32 elements of a lane's group,
and one block for the whole matrix; planes and x at odd addresses."""
import numpy as np
import pytest

from glint_amd import glint_hip as H
from oracle import glint_oracle as G
from tests.gpu_util import bf16_bits, dev, host, torch_cuda

pytestmark = pytest.mark.gpu


def _inputs(M, N, K, bs, seed=0):
    rng = np.random.default_rng(1000 * M + 10 * N + K + bs + seed)
    n = N * K
    hole = rng.integers(0, 256, (n + 1) // 2, dtype=np.uint8)
    plug = rng.integers(0, 256, (n + 1) // 2, dtype=np.uint8)
    am = (rng.uniform(0.01, 1.0, (n + bs - 1) // bs) * rng.choice([1.0, 0.0], (n + bs - 1) // bs, p=[0.9, 0.1])).astype(np.float32)
    x = bf16_bits(rng.normal(0, 1, M * K).astype(np.float32))
    return hole, plug, am, x


def _run(M, N, K, bs, hole, plug, am, x, shift=0):
    dh, dp, dx, da = dev(hole, shift), dev(plug, shift), dev(x, shift), dev(am)
    f = host(H.htile_f32(dh, dp, da, dx, N, K, bs)).reshape(M, N)
    b = G.bf16_bits_to_f32(host(H.htile_bf16(dh, dp, da, dx, N, K, bs), np.uint16).reshape(-1)).reshape(M, N)
    return f, b


@pytest.mark.parametrize("M,N,K,bs,shift", [
    (1, 1, 1, 1, 0), (1, 17, 127, 64, 0), (2, 16, 128, 32, 1), (16, 15, 129, 64, 0), (17, 33, 130, 128, 1),
    (16, 40, 1023, 64, 0), (32, 31, 1025, 32, 0), (33, 16, 1024, 33, 1), (64, 50, 1152, 31, 0), (65, 64, 1151, 64, 1),
    (5, 7, 2177, 1, 0), (20, 21, 260, 5, 0), (70, 100, 999, 1 << 20, 0), (129, 4200, 264, 64, 0), (130, 4111, 265, 48, 1),
    (3, 100, 4104, 64, 0), (1, 3, 9000, 64, 1), (8, 64, 4096, 64, 1)])
def test_every_shape_vs_float64(oracle, M, N, K, bs, shift):
    print(f"htile_any M={M} N={N} K={K} bs={bs} shift={shift}", flush=True)
    ins = _inputs(M, N, K, bs)
    f, b = _run(M, N, K, bs, *ins, shift=shift)
    ref, asum = (a.reshape(M, N) for a in oracle.htile_f64(*ins, M, N, K, bs))
    bound = (K + 2) * 2.0 ** -23 * asum + 1e-37
    assert (np.abs(f - ref) <= bound).all()
    assert (np.abs(b - ref) <= np.abs(ref) * 2.0 ** -8 + bound * 1.01).all()


def _fma_sum(oracle, hole, plug, am, x, M, N, K, bs):
    """One f32 FMA per weight in k order (products that overflow alone may not overflow there)."""
    w = G.expand(hole, plug, am, N * K, bs).reshape(N, K)
    xf = G.bf16_bits_to_f32(x).reshape(M, K)
    acc = np.zeros(M * N, np.float32)
    for k in range(K):
        acc = oracle.fmaf(np.tile(w[:, k], M), np.repeat(xf[:, k], N), acc)
    return acc.reshape(M, N)


@pytest.mark.parametrize("M,N,K,bs", [(3, 20, 200, 64), (20, 18, 333, 20), (66, 33, 1100, 64)])
@pytest.mark.parametrize("what", ["x inf", "x nan", "x subnormal", "scale inf", "scale nan", "scale tiny", "scale huge"])
def test_special_values_as_the_scalar_sum(oracle, M, N, K, bs, what):
    """Infinities, NaN and the ends of the f32 range come out as one f32 FMA per weight in k
    order gives them: the same class everywhere (the zeros of a split weight meet no infinity),
    and the value within the sum's bound where it is finite."""
    print(f"htile_any M={M} N={N} K={K} bs={bs} {what}", flush=True)
    hole, plug, am, x = _inputs(M, N, K, bs, seed=1)
    am = np.maximum(am, np.float32(0.01))
    am[1], am[-1] = 0.5, 0.25
    if what == "x inf":
        x[K // 2], x[-1] = 0x7F80, 0xFF80
    elif what == "x nan":
        x[K - 1] = 0x7FC1
    elif what == "x subnormal":
        x[:K] = np.arange(K, dtype=np.uint16) % 128  # row 0: zero and every subnormal magnitude
    elif what == "scale tiny":
        am[:] = np.float32(2.0 ** -125)
    else:
        am[1] = am[-1] = {"scale inf": np.inf, "scale nan": np.nan, "scale huge": np.float32(3e38)}[what]
    f, b = _run(M, N, K, bs, hole, plug, am, x)
    with np.errstate(all="ignore"):
        want = _fma_sum(oracle, hole, plug, am, x, M, N, K, bs)
        ref, asum = (a.reshape(M, N) for a in oracle.htile_f64(hole, plug, am, x, M, N, K, bs))
        assert np.array_equal(np.isnan(f), np.isnan(want)) and np.array_equal(np.isinf(f), np.isinf(want))
        assert np.array_equal(np.sign(f[np.isinf(f)]), np.sign(want[np.isinf(want)]))
        fin = np.isfinite(want)
        # K roundings of the f32 subnormal spacing 2^-149 at most, beside the relative bound
        bound = (K + 2) * (2.0 ** -23 * asum + 2.0 ** -149)
        assert (np.abs(f - ref)[fin] <= bound[fin]).all()
        assert np.array_equal(np.isnan(b), np.isnan(want))
        assert (np.abs(b - ref)[fin] <= (np.abs(ref) * 2.0 ** -8 + bound * 1.01 + 2.0 ** -133)[fin]).all()


@pytest.mark.parametrize("M,N,K,bs", [(16, 17, 5, 2), (17, 16, 128, 32), (33, 40, 129, 32), (64, 30, 263, 48),
                                      (65, 4111, 393, 64), (130, 4111, 264, 33), (2, 50, 777, 5), (20, 100, 999, 1 << 20)])
def test_second_way_in_k_order(oracle, M, N, K, bs):
    """An infinite x in the last element, and a scale below 2^-90: every workgroup forms its outputs
    by one f32 FMA per weight in k order, bit for bit the emulation's, at the edges of its 128-wide
    steps of K, of a thread's 8 elements and of the tiles (one and two strips of W)."""
    print(f"htile_any second way M={M} N={N} K={K} bs={bs}", flush=True)
    hole, plug, am, x = _inputs(M, N, K, bs, seed=2)
    am = (am * np.float32(1e-33)).astype(np.float32)
    am[0] = 1e-30
    x[-1] = 0x7F80
    f, _ = _run(M, N, K, bs, hole, plug, am, x)
    with np.errstate(all="ignore"):
        want = _fma_sum(oracle, hole, plug, am, x, M, N, K, bs)
    assert np.array_equal(np.isnan(f), np.isnan(want))
    met = ~np.isnan(want)
    rows = np.arange(N) * K  # strips of W that met a nonzero scale: all outputs of these are the second way's
    first, last = rows // bs, (rows + K - 1) // bs
    tiny = np.array([(am[a:b + 1] != 0).any() for a, b in zip(first, last)])
    met &= tiny[None, :]
    assert met.any() and np.array_equal(f[met] + 0.0, want[met] + 0.0)


def test_special_values_time():
    """NaN in every row of x, and every scale below 2^-90: the second way takes less than 12 times
    the common one (one thread per output over global memory took 150 to 300 times)."""
    torch = torch_cuda()
    M, N, K, bs = 130, 5000, 5000, 64
    print("htile_any time of the second way", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    pin = H.encode_bf16((torch.randn(N * K, device="cuda", generator=g) * 0.02).to(torch.bfloat16), bs)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    xn = x.clone()
    xn[:, 7] = float("nan")

    def us(pin, x):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record()
        for _ in range(5):
            H.htile_bf16(*pin, x, N, K, bs)
        e[1].record()
        torch.cuda.synchronize()
        return e[0].elapsed_time(e[1]) * 200
    us(pin, x)
    for other in ((pin, xn), ((pin[0], pin[1], pin[2] * 1e-33), x)):
        t = sorted(us(*other) / us(pin, x) for _ in range(5))
        assert t[2] < 12, t
