"""int8_mma_gemm on the 256 x 256 DMA tiles: its convert-free epilogue and the plain one that a
tile with sx outside [2^-30, 2^11) or sw outside 0 and [2^-40, 2^60) takes. Both are the
emulation's f32 operations, so every output is compared bit for bit: scales at the ends of the
range, zero, negative, below, above, infinite and NaN, in some tiles only; columns not a multiple
of 4 and y at an odd address (no 16-byte stores); one scale anywhere in a tile, at every part of
the look over it; and the time with such scales beside the time without."""
import numpy as np
import pytest

from glint_amd import glint_hip as H
from tests.gpu_util import bf16_bits, dev, first_diff, host, torch_cuda

pytestmark = pytest.mark.gpu


def _check(oracle, x, wq, sw, m, n, k, rows, shift=0):
    torch = torch_cuda()
    buf = torch.full((m * n + 8,), 9.0, device="cuda")
    dx, dq, ds = dev(x), dev(wq), dev(sw)
    xq = torch.empty(m * k, dtype=torch.int8, device="cuda")
    sx = torch.empty(m * k // 64, device="cuda")
    lin = H.Int8MmaLinear(dq.data_ptr(), ds.data_ptr(), n, k)
    assert H.p7_lib().int8_mma_gemm(H._p(dx), lin, H.VP(buf.data_ptr() + 4 * shift), m, H._p(xq), H._p(sx), H._stream()) == 0
    got = host(buf)
    assert (got[:shift] == 9.0).all() and (got[shift + m * n:] == 9.0).all()
    got = got[shift:shift + m * n].reshape(m, n)
    oxq, osx = oracle.quant_act(x, m, k)
    assert host(xq).tobytes() == oxq.tobytes() and host(sx).tobytes() == osx.tobytes()
    nkb = k // 64
    for r in rows:
        with np.errstate(all="ignore"):
            want = oracle.int8_mma_emu(oxq[r * k:(r + 16) * k], osx[r * nkb:(r + 16) * nkb], wq, sw, 16, n, k)
        a, b = got[r:r + 16], want
        same = (a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))
        assert same.all(), (r, first_diff(a.view(np.uint32), b.view(np.uint32)))


@pytest.mark.parametrize("n,shift", [(24576, 0), (24575, 0), (24576, 1)])
def test_scales_in_range(oracle, n, shift):
    m, k = 512, 192
    print(f"int8 scales in range n={n} shift={shift}", flush=True)
    rng = np.random.default_rng(n + shift)
    # sx = amax / 127 from just above 2^-36 to just below 2^7, rows of extreme products
    mag = np.float32(2.0) ** rng.integers(-28, 13, m * k // 64).repeat(64)
    x = bf16_bits((rng.uniform(-1, 1, m * k) * mag).astype(np.float32))
    wq = rng.integers(-128, 128, n * k, dtype=np.int64).astype(np.int8)
    sw = (np.float32(2.0) ** rng.integers(-36, 7, n * k // 64) * rng.uniform(1, 2, n * k // 64)).astype(np.float32)
    sw *= rng.choice(np.float32([1, -1, 0]), sw.size, p=[0.8, 0.1, 0.1])
    x[:k] = bf16_bits(np.full(k, 100.0, np.float32))
    wq[:k], wq[k:2 * k] = 127, -128  # the largest |ic|, both signs
    _check(oracle, x, wq, sw, m, n, k, (0, 256, m - 16), shift)


@pytest.mark.parametrize("what", ["x tiny", "x huge", "x inf", "sw tiny", "sw huge", "sw inf", "sw nan"])
def test_scales_out_of_range(oracle, what):
    """The rows or columns with the scale, and tiles without one, all equal the emulation."""
    m, n, k = 512, 24576, 192
    print(f"int8 scales {what}", flush=True)
    rng = np.random.default_rng(len(what))
    x = bf16_bits(rng.normal(0, 1, m * k).astype(np.float32)).reshape(m, k)
    wq = rng.integers(-127, 128, n * k, dtype=np.int8)
    sw = rng.uniform(1e-3, 2e-2, (n, k // 64)).astype(np.float32)
    if what.startswith("x"):
        x[5, 64:128] = {"x tiny": bf16_bits(np.full(64, 1e-30, np.float32)), "x huge": bf16_bits(np.full(64, 1e30, np.float32)),
                        "x inf": bf16_bits(np.full(64, np.inf, np.float32))}[what]
    else:
        sw[300, 1] = {"sw tiny": 1e-20, "sw huge": 1e20, "sw inf": np.inf, "sw nan": np.nan}[what]
    _check(oracle, x.reshape(-1), wq, sw.reshape(-1), m, n, k, (0, 256))


@pytest.mark.parametrize("k", [64, 256, 320, 2112])
def test_one_scale_anywhere_in_a_tile(oracle, k):
    """A lone tiny scale whose outputs the scaled accumulators could not hold, at another row and
    slice in each tile: whole rounds of the look, the last round, the rest behind it."""
    m, n, nkb = 2047, 6143, k // 64
    print(f"int8 scales one anywhere k={k}", flush=True)
    rng = np.random.default_rng(k)
    x = bf16_bits(rng.normal(0, 1, m * k).astype(np.float32)).reshape(m, nkb, 64)
    wq = rng.integers(-127, 128, n * k, dtype=np.int8)
    sw = rng.uniform(1e-3, 2e-2, (n, nkb)).astype(np.float32)
    for t in range(24):  # column tiles: the first and the last row of a wave's 64, slices from both ends
        r, c = 256 * t + min((64 * t + (63 if t & 4 else 0)) % 256, n - 1 - 256 * t), (t // 8 * nkb // 2 + t % 2 * (nkb - 1)) % nkb
        sw[r] = 0.0
        sw[r, c] = np.float32(1.2345e-35) * (t + 1)
    rows = []
    for t in range(8):  # row tiles
        r, c = min(256 * t + 64 * (t % 4) + (63 if t & 4 else 0), m - 1), (t * 5) % nkb
        x[r] = 0
        x[r, c] = bf16_bits((rng.normal(0, 1, 64) * 1e-33).astype(np.float32))
        rows.append(min(r, m - 16))
    _check(oracle, x.reshape(-1), wq, sw.reshape(-1), m, n, k, rows)


@pytest.mark.parametrize("what", ["x tiny", "x huge", "sw tiny"])
def test_scales_out_of_range_cost_no_second_walk(what):
    """One such scale in every tile takes less than half as long again as none (the plain epilogue
    measured 1.0 to 1.15 times the other; a tile walked twice is at least 2)."""
    torch = torch_cuda()
    m, n, k = 2048, 8192, 2048
    print(f"int8 scales time {what}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn(m, k, device="cuda", generator=g).to(torch.bfloat16)
    q = torch.randint(-127, 128, (n * k,), device="cuda", generator=g, dtype=torch.int8)
    sw = torch.rand(n, k // 64, device="cuda", generator=g) * 0.019 + 1e-3
    x2, sw2 = x.clone(), sw.clone()
    if what == "sw tiny":
        sw2[9::256, 3] = 1e-20
    else:
        x2[9::256, 64:128] = 1e-12 if what == "x tiny" else 1e9
    xq, sx = torch.empty(m * k, dtype=torch.int8, device="cuda"), torch.empty(m * k // 64, device="cuda")

    def us(xx, ss):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record()
        for _ in range(20):
            H.int8_mma_gemm(xx, q, ss, n, k, xq, sx)
        e[1].record()
        torch.cuda.synchronize()
        return e[0].elapsed_time(e[1]) * 50
    us(x, sw)
    t = sorted(us(x2, sw2) / us(x, sw) for _ in range(7))
    assert t[3] < 1.5, t
