"""f32 out at M = 5 and 6 under graph capture: the two small-M launches, bit for bit, whether the
stream has a split-K workspace or not, so a graph of them outlives the workspace's release."""
import numpy as np
import pytest

from glint_amd import glint_hip as H
from tests.gpu_util import dev, host, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reserve", [False, True])
@pytest.mark.parametrize("M", [5, 6])
def test_small_m_capture_needs_no_workspace(M, reserve):
    torch = torch_cuda()
    N, K = 1024, 8192  # K is split there
    print(f"capture M={M} reserve={reserve}", flush=True)
    rng = np.random.default_rng(M)
    pin = [dev(rng.integers(0, 256, N * K // 2, dtype=np.uint8)) for _ in range(2)]
    pin.append(dev(rng.uniform(0.01, 1.0, N * K // 64).astype(np.float32)))
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    y = torch.zeros((M, N), device="cuda")
    want = np.concatenate([host(H.htile_f32(*pin, x[:4], N, K)), host(H.htile_f32(*pin, x[4:], N, K))])
    s = torch.cuda.Stream()
    lib = H.encode_lib()
    if reserve:
        assert lib.glint_htile_workspace_reserve(H._stream(s)) == 0
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        H.htile_f32(*pin, x, N, K, out=y)
    for i in range(4):
        if i == 2 and reserve:
            assert np.array_equal(host(y), want)  # what follows holds only for these launches
            assert lib.glint_htile_workspace_release(H._stream(s)) == 0
        y.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        assert np.array_equal(host(y), want), i
        with torch.cuda.stream(s):  # the stream's own eager calls, split
            e = host(H.htile_f32(*pin, x, N, K))
        assert np.allclose(e, want, rtol=0, atol=1e-4 * np.abs(want).max())
    lib.glint_htile_workspace_release(H._stream(s))
