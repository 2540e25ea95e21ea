"""k_encode_blocks and k_expand_runs at the forms they take: blocks of 32, 64 and 128, BF16 and
F32 input, tensors that end in a partial 512-element chunk (encode) or 2048-element chunk
(expand), at one chunk, at the last wave of a workgroup, and past the resident grid. The format
defines every byte, so the comparison with the oracle is exact."""
import numpy as np
import pytest

from glint_amd import glint_hip as H
from tests.gpu_util import bf16_bits, dev, first_diff, host

pytestmark = pytest.mark.gpu


def _weights(n, seed):
    """N(0, 0.02^2) with, at every block scale, blocks of zeros, NaN, infinities, subnormal,
    tiny and huge values."""
    rng = np.random.default_rng(seed)
    w = rng.normal(0, 0.02, n).astype(np.float32)
    for i, v in enumerate((0.0, np.nan, np.inf, 1e-40, 1e-30, 1e30)):
        w[i * 300:i * 300 + 140] *= np.float32(0.0) if v == 0.0 else np.float32(1.0)
        if v != 0.0:
            w[i * 300 + 7:i * 300 + 140:50] = v
    w[-1:] = -0.0 if n % 2 else 0.5
    return w


@pytest.mark.parametrize("n", [512, 513, 575, 1023, 2047, 2048, 2049, 8192 + 1, 16 * 512 + 511, 4096 * 512 + 33,
                               8192 * 512 * 2 + 300])
@pytest.mark.parametrize("bs", [32, 64, 128])
def test_encode_expand_bytes(oracle, n, bs):
    print(f"codec n={n} bs={bs}", flush=True)
    with np.errstate(all="ignore"):
        w = _weights(max(n, 2048), n + bs)[:n]
        u16 = bf16_bits(w)
        for name, got, want in (("bf16", H.encode_bf16(dev(u16), bs), oracle.encode_bf16(u16, bs)),
                                ("f32", H.encode_f32(dev(w), bs), oracle.encode_f32(w, bs))):
            for g, e, part in zip(got, want, ("hole", "plug", "absmax")):
                assert host(g).tobytes() == e.tobytes(), f"{name} {part}: {first_diff(host(g), e)}"
        hole, plug, am = want
        d = [dev(a) for a in want]
        assert host(H.expand_f32(*d, n, bs)).tobytes() == oracle.expand_f32(hole, plug, am, n, bs).tobytes()
        assert host(H.expand_bf16(*d, n, bs), np.uint16).tobytes() == oracle.expand_bf16(hole, plug, am, n, bs).tobytes()


@pytest.mark.parametrize("n", [2049, 4095, 70001])
def test_nothing_past_the_end_is_written(n):
    """Planes, absmax and the expanded tensor sit in front of sentinel bytes."""
    import torch
    rng = np.random.default_rng(n)
    w = dev(bf16_bits(rng.normal(0, 0.02, n)))
    npk, nam = (n + 1) // 2, (n + 63) // 64
    bufs = [torch.full((npk + 64,), 0xA5, dtype=torch.uint8, device="cuda"), torch.full((npk + 64,), 0xA5, dtype=torch.uint8, device="cuda"),
            torch.full((nam + 16,), 7.25, device="cuda")]
    H.encode_bf16(w, 64, out=tuple(bufs))
    out = torch.full((n + 16,), 7.25, device="cuda")
    H.expand_f32(*bufs, n, 64, out=out)
    torch.cuda.synchronize()
    assert (bufs[0][npk:] == 0xA5).all() and (bufs[1][npk:] == 0xA5).all()
    assert (bufs[2][nam:] == 7.25).all() and (out[n:] == 7.25).all()
