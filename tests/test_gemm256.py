"""GPU tests (-m gpu): the 256 x 256 product at the edges of its pipeline and of its tile order."""
import ctypes as C

import numpy as np
import pytest

import nvr_import


@pytest.mark.gpu
# K-tiles: 15 (odd), 17, 16; 162 tiles, 256 (and rows behind them on the smaller tiles) and 237; columns in panels of 5 and 4, of 8 and of 3; row blocks: one row left, 32 rows left
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
# two, three and five K-tiles; the vocabulary's last tile of 16 columns; 2, 34 and 33 tiles, and several tiles a workgroup: 291 and 582
@pytest.mark.parametrize("T,K,N", [(192, 128, 272), (257, 192, 4112), (513, 320, 2576), (513, 128, 24592), (700, 192, 49424)])
def test_head_at_the_edges_of_its_pipeline(T, K, N):
    nvr = nvr_import.load()
    rng = np.random.default_rng(T)
    x, W = (rng.standard_normal((T, K), dtype=np.float32)).astype(np.float16), (rng.standard_normal((N, K), dtype=np.float32) * np.float32(0.05)).astype(np.float16)
    x[5], x[7] = 0, np.nan                                  # a row of equal logits, and one of no number
    d_x, d_W, d_y = nvr.DeviceBuffer.from_numpy(x), nvr.DeviceBuffer.from_numpy(W), nvr.DeviceBuffer(T * N * 4)
    parts = C.c_int32(0)
    d_pv, d_pi = nvr.DeviceBuffer(2048 * T * 4), nvr.DeviceBuffer(2048 * T * 4)
    nvr.check(nvr.lib().nvr_lm_head(d_x.ptr, K, d_W.ptr, T, K, N, d_y.ptr, d_pv.ptr, d_pi.ptr, C.byref(parts), None))
    assert parts.value == (N + 255) // 256
    got, want = d_y.to_numpy((T, N), np.float32), x.astype(np.float64) @ W.astype(np.float64).T
    assert np.isnan(got[7]).all()
    got[7], want[7] = 0, 0
    assert np.all(np.abs(got - want) <= K * 2.0 ** -24 * 0.25 * K ** 0.5 + 1e-6)
    value, index = d_pv.to_numpy((parts.value, T), np.float32), d_pi.to_numpy((parts.value, T), np.int32)
    first = np.arange(parts.value, dtype=np.int32) * 256
    assert np.array_equal(index[:, 5], first) and not value[:, 5].any()                  # (the first of equal ones)
    assert np.all(value[:, 7] == -np.inf) and np.all(index[:, 7] == 0x7fffffff)          # (no entry is larger than the lowest value)
    value[:, 7], index[:, 7] = 0, first
    best = value.argmax(0)
    assert np.array_equal(index[best, np.arange(T)], got.argmax(1)) and np.array_equal(value.max(0), got.max(1))


def _bits(a, dtype):
    a = np.ascontiguousarray(a, np.float32)
    if dtype == "float16":
        return a.astype(np.float16).view(np.uint16)
    u = a.view(np.uint32)
    return ((u + 0x7fff + ((u >> 16) & 1)) >> 16).astype(np.uint16)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
# More tiles than workgroups, so that a tile's first K-tile runs with the stores of the tile before it under way (32 of them, of a gated unit 16), ragged last row blocks, even and odd numbers of
# K-tiles, the smallest that these entry points bring here: 4 and 5 (456 tiles); the residual form's 13 (405 tiles)
@pytest.mark.parametrize("kind,T,K,N", [("plain", 9721, 256, 3072), ("plain", 9721, 320, 3072), ("silu", 9721, 256, 1536), ("silu", 9721, 320, 1536), ("residual", 11272, 832, 2304)])
def test_several_tiles_a_workgroup(kind, T, K, N, dtype):
    """All rows at once, three times, against the same rows a thousand at a time, which the smaller tiles take: bit for bit (the order of a row's sums is the same on either)."""
    nvr = nvr_import.load()
    l, rng = nvr.lib(), np.random.default_rng(T + K)
    x, W = _bits(rng.standard_normal((T, K), dtype=np.float32), dtype), _bits(rng.standard_normal((2 * N if kind == "silu" else N, K), dtype=np.float32) * np.float32(0.05), dtype)
    h = _bits(rng.standard_normal((T, N), dtype=np.float32), dtype)
    d_x, d_W, d_one, d_h, d_y, d_n = (nvr.DeviceBuffer.from_numpy(a) for a in (x, W, _bits(np.ones(N), dtype), h, h, h))

    def product(at, rows):
        args = d_x.ptr + at * K * 2, K, d_W.ptr, rows, K, N, d_y.ptr + at * N * 2
        nvr.check(l.nvr_linear_silu_mul(*args, None) if kind == "silu" else l.nvr_linear(*args, 0, None))
    nvr.check(l.nvr_ops_set_dtype(dtype.encode()))
    try:
        for at in range(0, T, 1000):
            product(at, min(1000, T - at))
        if kind == "residual":
            nvr.check(l.nvr_add_rmsnorm(d_h.ptr, d_y.ptr, d_one.ptr, 1e-6, T, N, d_n.ptr, None))
        want = (d_h if kind == "residual" else d_y).to_numpy((T, N), np.uint16)
        assert np.unique(want[::97, :64], axis=0).shape[0] > T // 100
        for _ in range(3):
            if kind == "residual":
                d_y = nvr.DeviceBuffer.from_numpy(h)
                nvr.check(l.nvr_linear_add_residual(d_x.ptr, K, d_W.ptr, T, K, N, d_y.ptr, None))
            else:
                d_y.zero()
                product(0, T)
            got = d_y.to_numpy((T, N), np.uint16)
            assert np.array_equal(got, want), np.flatnonzero((got != want).any(1))[:8]
    finally:
        nvr.check(l.nvr_ops_set_dtype(b"float16"))
