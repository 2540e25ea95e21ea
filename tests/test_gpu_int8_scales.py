"""int8_mma_gemm on the 256 x 256 DMA tiles: its convert-free epilogue and the walk that scales
outside [2^-36, 2^7) take. Both are the emulation's f32 operations, so every output is compared
bit for bit: scales at the ends of the range, zero, negative, below, above, infinite and NaN, in
some tiles only; columns not a multiple of 4 and y at an odd address (no 16-byte stores)."""
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
