"""Steps that are queued without waiting: a step at another batch size replaces
the captured graph of a step whose launches may still be in the queue."""
import numpy as np
import pytest

from strict_amd import llm
from test_gpu_llm import GPT2_SMALL_TEST, _randomize_small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("logits", [False, True])
def test_batch_sizes_change_while_steps_are_queued(ctx, logits):
    tokens = np.random.default_rng(6).integers(0, GPT2_SMALL_TEST.vocab, (40, 4))
    with llm.Model(ctx, GPT2_SMALL_TEST.with_(max_batch=4)) as m:
        m.init_random(seed=3, stddev=0.02)
        _randomize_small_params(m, 1)

        def run(wait):
            out = []
            for b in (2, 3, 4, 2, 4, 3):
                m.reset(b)
                for t in tokens:
                    m.step(t[:b], logits=logits)
                    if wait:
                        ctx.sync()
                if b == 3:  # the others stay queued behind the next batch's
                    m.step(tokens[0, :b], logits=True)
                    out.append(m.logits().copy())
            return out

        for x, y in zip(run(False), run(True)):
            assert np.array_equal(x, y)
