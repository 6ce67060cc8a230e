"""Prompt attention that brings the gated unit's weights into the caches: which steps do (the rule itself, on the CPU), and that nothing but time depends on it (-m gpu)."""
import os
import subprocess

import numpy as np
import pytest

import nvr_import
import test_kernel_routes_gpu as routes

nvr = nvr_import.load()
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-rs_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "kernels.h"
int main(int argc, char **argv) {
    for (int i = 1; i + 2 < argc; i += 3) {
        const long T = atol(argv[i]), K = atol(argv[i + 1]), I = atol(argv[i + 2]);
        const nvr::kt::half_bits w = 0;
        const nvr::kt::Ahead a = nvr::k::linear_silu_ahead(&w, T, K, I), b = nvr::kb::linear_silu_ahead(&w, T, K, I);
        std::printf("%d %d %d %d\n", a.units, a.unit, b.units, b.unit);
    }
}
"""


def _ahead(tmp_path, shapes):
    """(units, pieces of 16 bytes in a unit) of each (T, K, I), from the library's own objects."""
    subprocess.check_call(["make", "-C", CSRC, "-j8"], stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    hipcc, build = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), os.path.join(CSRC, "build")
    kernels = sorted(os.path.join(build, "kernels", f) for f in os.listdir(os.path.join(build, "kernels")) if f.endswith(".hip.o") or f.endswith(".hip.bf16.o"))
    subprocess.check_call([hipcc, "--offload-arch=gfx950", "-std=c++17", "-x", "hip", "-I", os.path.join(CSRC, "kernels"), "-c", str(tmp_path / "main.cpp"), "-o", str(tmp_path / "main.o")])
    subprocess.check_call([hipcc, "--offload-arch=gfx950", str(tmp_path / "main.o"), os.path.join(build, "common.cpp.o"), *kernels, "-ldl", "-o", str(tmp_path / "main")])
    out = subprocess.check_output([str(tmp_path / "main"), *(str(n) for s in shapes for n in s)], text=True)
    rows = [tuple(int(n) for n in line.split()) for line in out.splitlines()]
    assert len(rows) == len(shapes) and all(r[:2] == r[2:] for r in rows)      # (both 16-bit types)
    return [r[:2] for r in rows]


def test_steps_that_bring_weights(tmp_path):
    """The steps of the GPU tests bring what they are there for, and every step that brings anything brings the weights once, whole: in units that end where they do."""
    cases = [(sum(lengths), 256, inter) for inter, lengths in routes.AHEAD_PROMPTS]
    swept = [(T, K, I) for T in (1, 33, 56, 64, 65, 127, 128, 129, 200, 257, 320, 321, 384, 385, 509, 512, 513, 640, 1000, 1280, 1281, 1600, 3000) for K in (32, 96, 256, 1024, 1056, 2048)
             for I in (64, 128, 192, 384, 512, 1152, 2304, 3072, 3456, 6144)]
    got = _ahead(tmp_path, cases + [(T, 256, 3072) for T in PAIRED_STEPS] + swept)
    for (T, K, I), (units, unit) in zip(cases, got):
        assert (units > 0) == (I != 2112), (T, I)                              # (columns in no eighths)
        if units:
            assert unit == (48 * K // 8 if routes.AHEAD_96_ROWS[T, I] else I // 8 * K // 8)
    assert all(units > 0 for units, _ in got[len(cases):len(cases) + len(PAIRED_STEPS)])
    brought = 0
    for (T, K, I), (units, unit) in zip(swept, got[len(cases) + len(PAIRED_STEPS):]):
        assert (units == 0) == (unit == 0) and (units == 0 or (units * unit * 16 == 2 * I * K * 2 <= 24 << 20 and units % 8 == 0)), (T, K, I)
        brought += units > 0
    assert brought > 100


# heads, kv heads (tiles of 128, 64 and 32 positions), positions of a cached prefix in blocks of 16 and 64, the sequence that is compared, the others of the step; as two sequences the step has 160
# workgroups of attention at most, as many 168 and more
PAIRS = [(16, 8, 0, 16, 180, 150, 18), (8, 8, 0, 16, 180, 150, 20), (32, 8, 0, 16, 180, 150, 16), (16, 8, 0, 16, 45, 20, 20), (16, 8, 0, 16, 1000, 216, 5),
         (16, 8, 192, 16, 180, 150, 18), (16, 8, 192, 64, 180, 150, 18), (8, 8, 64, 16, 100, 230, 20), (8, 8, 64, 64, 100, 230, 20), (32, 8, 128, 16, 200, 130, 16), (32, 8, 128, 64, 200, 130, 16)]
PAIRED_STEPS = sorted({p[4] + p[5] for p in PAIRS})


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("heads,kv,prefix,page,length,others,cut", PAIRS)
def test_weights_brought_ahead_change_nothing(heads, kv, prefix, page, length, others, cut, dtype):
    """A sequence's keys and values of the second and third layer, in a step that brings weights and in one with as many rows, hence the same products, whose sequences are too many for it: bit for
    bit.  Prompts from their own rows and behind a cached prefix."""
    tile = 128 * kv // heads
    tiles = lambda *lengths: kv * sum(-(-n // tile) for n in lengths)
    ends = [others * i // cut for i in range(cut + 1)]
    pieces = [b - a for a, b in zip(ends, ends[1:])]
    assert tiles(length, others) <= 160 < tiles(length, *pieces)
    model = nvr.ModelConfig(vocab_size=512, hidden_size=256, intermediate_size=3072, num_hidden_layers=3, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128,
                            max_position_embeddings=2048, tie_word_embeddings=1, seed=heads + page)
    blocks, got = 2 * (prefix + length + others) // page + 2 * cut + 8, []
    for cuts in ([others], pieces, [others]):
        runner = nvr.ModelRunner(nvr.Config(skip_block_size_check=1, dtype=dtype, max_num_seqs=32, max_num_batched_tokens=2048, max_model_len=2048, kvcache_block_size=page, num_kvcache_blocks=blocks), model)
        manager = nvr.BlockManager(blocks, page)
        sequence = lambda tokens: nvr.Sequence(tokens, nvr.SamplingParams(temperature=0.0, ignore_eos=True), page)
        head = nvr.synthetic_tokens(prefix, 5, 1, 512) if prefix else np.empty(0, np.int64)
        if prefix:
            first = sequence(head)
            manager.allocate(first)
            runner.execute_model([first], True)
        rest = nvr.synthetic_tokens(others, 5, 3, 512)
        batch = [sequence(np.concatenate([head, nvr.synthetic_tokens(length, 5, 2, 512)]))] + [sequence(part) for part in np.split(rest, np.cumsum(cuts)[:-1])]
        for s in batch:
            manager.allocate(s)
        assert batch[0].num_cached_tokens == prefix
        runner.execute_model(batch, True)
        rows = (np.asarray(batch[0].block_table, np.int64)[:, None] * page + np.arange(page)).ravel()[prefix:prefix + length]
        mine = []
        for layer in (1, 2):
            for pointer in runner.kv_cache(layer):
                cache = np.empty((blocks * page, kv * 128), np.uint16)
                nvr.check(nvr.lib().nvr_memcpy_d2h(cache.ctypes.data, pointer, cache.nbytes))
                mine.append(cache[rows])
        got.append(mine)
    for layer in range(4):
        assert np.unique(got[0][layer], axis=0).shape[0] == length
        assert np.array_equal(got[0][layer], got[1][layer]) and np.array_equal(got[0][layer], got[2][layer])
