"""rt_test_decode's copy to host memory: one piece, ragged last pieces, more pieces than pinned slots, a matrix over the
device buffer's 64 MB, into fresh and into reused memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kqt,N,K", [(2, 64, 256), (3, 2112, 1024), (1, 4160, 4608), (4, 8256, 8192)])
def test_codes_reach_the_host(gpu, lib, tmp_path, kqt, N, K):
    from lazyweights_amd import Runtime, bundle
    H = {1: 2.3, 2: 3.4, 3: 4.3, 4: 2.6}[kqt]
    bundle.write_synthetic_bundle(str(tmp_path), [("a", kqt, N, K, H, 41), ("b", kqt, 64, K, H, 42)], threads=16)
    a, _ = bundle.synth_matrix(kqt, N, K, H, 41, threads=16)
    b, _ = bundle.synth_matrix(kqt, 64, K, H, 42, threads=16)
    with Runtime(tmp_path) as rt:
        assert np.array_equal(rt.test_decode("a"), a)
        assert np.array_equal(rt.test_decode("b"), b)
        out = np.full((N + 1, K), 0xAA, np.uint8)
        for _ in range(2):
            assert lib.rt_test_decode(rt.h, b"a", out.ctypes.data) == 0
        assert np.array_equal(out[:N], a) and (out[N] == 0xAA).all()


def test_two_threads_on_one_handle(gpu, lib, tmp_path):
    """Calls that overlap on one handle take its kept buffers in turn."""
    from concurrent.futures import ThreadPoolExecutor

    from lazyweights_amd import Runtime, bundle
    mats = [("a", 1, 1024, 4096, 2.3, 51), ("b", 3, 2112, 1024, 4.3, 52)]
    bundle.write_synthetic_bundle(str(tmp_path), mats, threads=16)
    want = {m[0]: bundle.synth_matrix(*m[1:], threads=16)[0] for m in mats}
    with Runtime(tmp_path) as rt, ThreadPoolExecutor(2) as pool:
        got = list(pool.map(lambda n: (n, rt.test_decode(n)), ["a", "b"] * 4))
        for name, codes in got:
            assert np.array_equal(codes, want[name])
