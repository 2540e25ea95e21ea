"""k_gemv_km_fold_part (8 to 64 channels per wave) and the batched correction, bit for bit
against the oracle, whose summation orders they keep: every channel count per wave, those a
64-block's boundary cuts (24, 40, 48, 56), rows past the last whole workgroup, lists shorter than
a part, than a batch of 8 entries, and longer, one block's channels and every block's."""
import numpy as np
import pytest

from glint_amd import glint_hip as H
from oracle import glint_oracle as G
from tests.gpu_util import dev, first_diff, host, torch_cuda

pytestmark = pytest.mark.gpu


def _km(oracle, N, K):
    rng = np.random.default_rng(N + 3 * K)
    pin = oracle.encode_f32(rng.normal(0, 0.02, N * K).astype(np.float32), 64)
    x = G.f32_to_bf16_bits(rng.normal(0, 1, K).astype(np.float32))
    return oracle.kmajor_pack(*pin, N, K), x


@pytest.mark.parametrize("reserve", [False, True])
@pytest.mark.parametrize("N,K,ksg", [(32, 64, 1), (544, 128, 1), (512, 192, 1), (1056, 256, 1), (96, 320, 1), (64, 384, 1),
                                     (608, 448, 1), (520 * 4, 512, 1), (64, 576, 1), (1024, 3072, 16), (544, 5120, 16),
                                     (96, 7168, 16), (2080, 4096, 16)])
def test_fold_parts(oracle, N, K, ksg, reserve):
    torch = torch_cuda()
    print(f"fold parts N={N} K={K} ksg={ksg} reserve={reserve}", flush=True)
    (hk, pk, sk), x = _km(oracle, N, K)
    s = torch.cuda.Stream()
    if reserve:  # the slices then meet inside the kernel
        assert H.encode_lib().glint_htile_workspace_reserve(H._stream(s)) == 0
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = [host(H.gemv_km_fold(dev(hk), dev(sk), dev(x), N, K, ksg)) for _ in range(2)]
    if reserve:
        assert H.encode_lib().glint_htile_workspace_release(H._stream(s)) == 0
    want = oracle.gemv_km_fold(hk, sk, x, N, K, ksg)
    for g in got:
        assert g.tobytes() == want.tobytes(), first_diff(g.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("ks", [1, 8])
@pytest.mark.parametrize("count", [0, 1, 7, 8, 9, 63, 64, 65, 500, 640])
def test_correction_batches(oracle, count, ks):
    torch_cuda()
    N, K = 544, 640
    print(f"correction count={count} ks={ks}", flush=True)
    (hk, pk, sk), x = _km(oracle, N, K)
    rng = np.random.default_rng(count + ks)
    idx = np.sort(rng.choice(K, count, replace=False)).astype(np.int32)
    if count == 63:
        idx = np.arange(64, 127, dtype=np.int32)  # one block
    y0 = rng.normal(0, 1, N).astype(np.float32)
    pad = np.zeros(K, np.int32)
    pad[:count] = idx
    got = host(H.apply_corr_km(dev(hk), dev(pk), dev(sk), dev(x), dev(pad), dev(np.array([count], np.int32)), dev(y0), N, K, ks))
    want = oracle.apply_corr_km(hk, pk, sk, x, idx, N, K, y0, ks)
    assert got.tobytes() == want.tobytes(), first_diff(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("ks", [1, 8])
@pytest.mark.parametrize("per_wave", [1, 2, 3, 4, 5])
def test_correction_short_parts(oracle, per_wave, ks):
    """Parts of one to five entries per wave (loaded two, four or eight at once), the last wave's
    shorter, with and without neighbours in a block."""
    torch_cuda()
    N, K = 544, 640
    (hk, pk, sk), x = _km(oracle, N, K)
    y0 = np.random.default_rng(ks).normal(0, 1, N).astype(np.float32)
    for short in (0, 1):
        count = per_wave * 8 * ks - short * (per_wave * 4 - 1)
        for idx in (np.arange(count), np.sort(np.random.default_rng(count).choice(K, count, replace=False))):
            print(f"correction parts of {per_wave} count={count} ks={ks}", flush=True)
            pad = np.zeros(K, np.int32)
            pad[:count] = idx
            got = host(H.apply_corr_km(dev(hk), dev(pk), dev(sk), dev(x), dev(pad), dev(np.array([count], np.int32)),
                                       dev(y0), N, K, ks))
            want = oracle.apply_corr_km(hk, pk, sk, x, idx.astype(np.int32), N, K, y0, ks)
            assert got.tobytes() == want.tobytes(), first_diff(got.view(np.uint32), want.view(np.uint32))
