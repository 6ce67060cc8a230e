"""GPU tests (-m gpu): the 256 x 256 product at the edges of its pipeline and of its tile order."""
import ctypes as C

import numpy as np
import pytest

import nvr_import


@pytest.mark.gpu
# K-tiles: 15 (odd), 17, two tiles a workgroup and more; columns in panels of 5 and 4, of 8 and of 3; row blocks: one row left, 8 rows left
@pytest.mark.parametrize("T,K,N", [(4353, 960, 2304), (8200, 1088, 4096), (20000, 1024, 768)])
def test_product_at_the_edges_of_its_tile_order(T, K, N):
    nvr = nvr_import.load()
    rng = np.random.default_rng(T)
    x, W = (rng.standard_normal((T, K), dtype=np.float32)).astype(np.float16), (rng.standard_normal((N, K), dtype=np.float32) * np.float32(0.05)).astype(np.float16)
    d_x, d_W, d_y = nvr.DeviceBuffer.from_numpy(x), nvr.DeviceBuffer.from_numpy(W), nvr.DeviceBuffer(T * N * 2)
    first = None
    for _ in range(3):
        d_y.zero()
        nvr.check(nvr.lib().nvr_linear(d_x.ptr, K, d_W.ptr, T, K, N, d_y.ptr, 0, None))
        got = d_y.to_numpy((T, N), np.float16)
        assert first is None or np.array_equal(first.view(np.uint16), got.view(np.uint16))
        first = got
    want = x.astype(np.float32) @ W.astype(np.float32).T
    # half an ulp of the rounding to 16 bits (2^-11), and sums of K products of about 0.05 in 32 bits in either order (K roundings of at most 2^-24 of a sum of about 0.05 sqrt K each)
    assert np.all(np.abs(first.astype(np.float32) - want) <= 2.0 ** -11 * np.abs(want) + 2 * K * 2.0 ** -24 * 0.25 * K ** 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("T,K,N", [(192, 128, 272), (257, 192, 4112), (513, 320, 2576)])     # two, three and five K-tiles; the vocabulary's last tile of 16 columns; 2, 34 and 33 tiles
def test_head_at_the_edges_of_its_pipeline(T, K, N):
    nvr = nvr_import.load()
    rng = np.random.default_rng(T)
    x, W = (rng.standard_normal((T, K), dtype=np.float32)).astype(np.float16), (rng.standard_normal((N, K), dtype=np.float32) * np.float32(0.05)).astype(np.float16)
    d_x, d_W, d_y = nvr.DeviceBuffer.from_numpy(x), nvr.DeviceBuffer.from_numpy(W), nvr.DeviceBuffer(T * N * 4)
    parts = C.c_int32(0)
    d_pv, d_pi = nvr.DeviceBuffer(2048 * T * 4), nvr.DeviceBuffer(2048 * T * 4)
    nvr.check(nvr.lib().nvr_lm_head(d_x.ptr, K, d_W.ptr, T, K, N, d_y.ptr, d_pv.ptr, d_pi.ptr, C.byref(parts), None))
    assert parts.value == (N + 255) // 256
    got, want = d_y.to_numpy((T, N), np.float32), x.astype(np.float64) @ W.astype(np.float64).T
    assert np.all(np.abs(got - want) <= K * 2.0 ** -24 * 0.25 * K ** 0.5 + 1e-6)
    value, index = d_pv.to_numpy((parts.value, T), np.float32), d_pi.to_numpy((parts.value, T), np.int32)
    best = value.argmax(0)
    assert np.array_equal(index[best, np.arange(T)], got.argmax(1)) and np.array_equal(value.max(0), got.max(1))
