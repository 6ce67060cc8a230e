"""The 256 x 256 product: its emitted code (CPU: products and their accumulators are inline asm, so hazards between them and ordinary instructions are not the compiler's to
count) and its results at the edges of its pipeline and of its tile order (GPU)."""
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

import nvr_import

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LLVM = "/opt/rocm/llvm/bin/"


def _registers(operand):
    m = re.match(r"([av])\[(\d+):(\d+)\]$", operand)
    if m:
        return {(m.group(1), i) for i in range(int(m.group(2)), int(m.group(3)) + 1)}
    m = re.match(r"([av])(\d+)$", operand)
    return {(m.group(1), int(m.group(2)))} if m else set()


def _states(line):
    """Wait states of an instruction."""
    return int(line[1]) + 1 if line[0] == "s_nop" else 1


@pytest.mark.parametrize("build", ["gemm256.hip.o", "gemm256.hip.bf16.o"])
def test_emitted_code_keeps_the_wait_states_around_its_products(build, tmp_path):
    obj = os.path.join(ROOT, "nano-vllm-rs_amd", "csrc", "build", "kernels", build)
    if not os.path.exists(obj) or not os.path.exists(LLVM + "llvm-objdump"):
        pytest.skip("no object file or no disassembler here")
    fat, code = str(tmp_path / "fat"), str(tmp_path / "code")
    subprocess.check_call([LLVM + "llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, obj, str(tmp_path / "copy")])
    subprocess.check_call([LLVM + "clang-offload-bundler", "--type=o", "--unbundle", "--input=" + fat, "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--output=" + code])
    text = subprocess.run([LLVM + "llvm-objdump", "-d", code], check=True, capture_output=True, text=True).stdout
    kernels = re.split(r"^[0-9a-f]+ <(\S*gemm256_kernel\S*)>:$", text, flags=re.M)[1:]
    assert kernels
    for name, body in zip(kernels[::2], kernels[1::2]):
        lines = [re.split(r"[ ,]+", l.split("//")[0].strip()) for l in body.split("\n") if l.startswith("\t")]
        written, products = {}, 0
        for i, l in enumerate(lines):
            if l[0].startswith("v_mfma"):
                products += 1
                sources, states, j = set().union(*(_registers(o) for o in l[2:5])), 0, i - 1
                while states < 2 and j >= 0:                              # an ordinary write of a source: two wait states
                    if lines[j][0].startswith("v_") and not lines[j][0].startswith("v_mfma"):
                        assert not _registers(lines[j][1]) & sources, (name, lines[j], l)
                    states += _states(lines[j])
                    j -= 1
                written.update((r, i) for r in _registers(l[1]))
            elif l[0].startswith(("v_", "global_store", "ds_write")):
                for r in set().union(*(_registers(o) for o in l[1:])) & written.keys():      # an ordinary read or write of a result: 18 behind a product of eight passes or fewer
                    states = 0
                    for k in range(written.pop(r) + 1, i):
                        states += _states(lines[k])
                        if states >= 18:
                            break
                    assert states >= 18, (name, l)
        assert products >= 256, name


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
