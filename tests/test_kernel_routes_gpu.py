"""GPU tests (-m gpu) of kernels and dispatch rules at the sizes where they change hands: edges of tiles, remainders, the smallest and largest of a
route's range, against the oracle or against the general path of the same operation."""
import ctypes as C

import numpy as np
import pytest

import nvr_import
import oracle
from oracle import model_oracle as mo

nvr = nvr_import.load()
pytestmark = pytest.mark.gpu

F16 = np.float16


def dev(a):
    return nvr.DeviceBuffer.from_numpy(np.ascontiguousarray(a))


def _small(dtype, batch, **kw):
    m = mo.small()
    model = nvr.ModelConfig(vocab_size=m.vocab_size, hidden_size=m.hidden_size, intermediate_size=m.intermediate_size, num_hidden_layers=m.num_hidden_layers,
                            num_attention_heads=m.num_attention_heads, num_key_value_heads=m.num_key_value_heads, head_dim=m.head_dim,
                            max_position_embeddings=m.max_position_embeddings, rms_norm_eps=m.rms_norm_eps, rope_theta=m.rope_theta,
                            tie_word_embeddings=m.tie_word_embeddings, init_std=m.init_std, seed=m.seed)
    cfg = nvr.Config(skip_block_size_check=1, max_num_seqs=batch, max_num_batched_tokens=batch * 24, max_model_len=64, kvcache_block_size=16,
                     num_kvcache_blocks=4 * batch, dtype=dtype, **kw)
    return cfg, model, m.vocab_size


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("batch", [1, 33])
def test_execute_model_stores_the_logits_with_the_step_as_on_demand(dtype, batch):
    """execute_model of a greedy batch writes the f32 logits in the step's own LM head; an engine's step leaves them to a second launch on demand: same
    bits, same tokens, prefill and decode steps (eager and replayed), one row block and more."""
    cfg, model, vocab = _small(dtype, batch)
    prompts = [nvr.synthetic_tokens(3 + i % 17, 5, i, vocab) for i in range(batch)]
    sp = nvr.SamplingParams(temperature=0.0, max_tokens=6, ignore_eos=True)
    nvr.lib().nvr_seq_reset_id_counter()
    eng = nvr.LLMEngine(cfg, model)
    for p in prompts:
        eng.add_request(p, sp)
    want = []
    while not eng.is_finished():
        rec = eng.step()
        want.append((rec["tokens"], eng.model_runner.logits(batch).copy()))
    runner = nvr.ModelRunner(cfg, model)
    bm = nvr.BlockManager(4 * batch, 16)
    seqs = [nvr.Sequence(p, sp, 16) for p in prompts]
    for s in seqs:
        bm.allocate(s)
    for i, (tokens, logits) in enumerate(want):
        runner.execute_model(seqs, i == 0)
        assert runner.sample_tokens(seqs) == tokens, i
        assert np.array_equal(runner.logits(batch), logits), i
        for s, t in zip(seqs, tokens):
            s.append_token(t)
            bm.may_append(s)
