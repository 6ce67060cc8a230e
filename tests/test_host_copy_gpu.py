"""GPU test (-m gpu): logits into a program's own memory, by the runtime's copy and by several threads (csrc/host_copy.h)."""
import ctypes as C
import threading

import numpy as np
import pytest

import nvr_import

nvr = nvr_import.load()
pytestmark = pytest.mark.gpu


def test_logits_arrive_whole_in_any_memory_and_number_of_pieces():
    vocab, batch = 70032, 41                                  # 280128 bytes a row: 30 rows are the first that take several threads (8 MiB), 41 are 10 pieces of 1 MiB and a part of one
    model = nvr.ModelConfig(vocab_size=vocab, hidden_size=128, intermediate_size=256, num_hidden_layers=1, num_attention_heads=2, num_key_value_heads=1, head_dim=64,
                            max_position_embeddings=64, tie_word_embeddings=1, seed=3)
    runner = nvr.ModelRunner(nvr.Config(skip_block_size_check=1, max_num_seqs=batch, max_num_batched_tokens=batch * 8, max_model_len=32, kvcache_block_size=16, num_kvcache_blocks=2 * batch), model)
    manager = nvr.BlockManager(2 * batch, 16)
    seqs = [nvr.Sequence(nvr.synthetic_tokens(3 + i % 5, 5, i, vocab), nvr.SamplingParams(temperature=0.0, ignore_eos=True), 16) for i in range(batch)]
    for s in seqs:
        manager.allocate(s)
    pointer = runner.execute_model(seqs, True)
    want = np.empty((batch, vocab), np.float32)
    nvr.check(nvr.lib().nvr_memcpy_d2h(want.ctypes.data, pointer, want.nbytes))
    assert np.unique(want[:, :64], axis=0).shape[0] > 30
    for rows in (1, 29, 30, 31, batch):
        assert np.array_equal(runner.logits(rows), want[:rows]), rows
    device = nvr.DeviceBuffer(want.nbytes)                    # memory of the runtime's own: its copy
    device.zero()
    nvr.check(nvr.lib().nvr_runner_copy_logits(runner.h, device.ptr, batch))
    assert np.array_equal(device.to_numpy(want.shape, np.float32), want)
    hip = nvr.lib()                                           # (finds the runtime that it has loaded)
    pinned = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(pinned), C.c_size_t(want.nbytes), 0) == 0
    try:
        held = np.frombuffer((C.c_char * want.nbytes).from_address(pinned.value), np.float32).reshape(want.shape)
        held[:] = 0
        nvr.check(nvr.lib().nvr_runner_copy_logits(runner.h, pinned, batch))
        assert np.array_equal(held, want)
    finally:
        assert hip.hipHostFree(pinned) == 0
    got = [[], []]                                            # two callers at once: they take turns
    def caller(mine):
        for _ in range(4):
            mine.append(runner.logits(batch))
    threads = [threading.Thread(target=caller, args=(mine,)) for mine in got]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert [len(mine) for mine in got] == [4, 4] and all(np.array_equal(one, want) for mine in got for one in mine)
