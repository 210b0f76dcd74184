"""Logits at some places of a step: the same bits from a captured step, which has its bucket's rows, and kernel by kernel."""
import pytest
import torch

from denno_beta_amd.engine import StepEntry
from denno_beta_amd.engine.graphs import BUCKETS, PORTION_REQUESTS, PORTION_ROWS, wanted_rows


def entries(lengths, wanted):
    """Requests of these lengths; the last place of the first `wanted` of them."""
    return [StepEntry(i, list(range(1, n + 1)), [n - 1] if i < wanted else []) for i, n in enumerate(lengths)]


@pytest.mark.parametrize("n", [1, 3, 16, 17, 33, 64, 65, 100])
def test_rows_that_a_captured_step_computes(n):
    for wanted in sorted({0, 1, n // 2, n}):
        # decoded tokens: every row of the bucket
        assert wanted_rows(entries([1] * n, wanted), 256) == (min(b for b in BUCKETS if b >= n) if wanted else 0)
        # portions: as many as there are requests
        assert wanted_rows(entries([2] * n, wanted), 256) == (min(b for b in PORTION_REQUESTS if b >= n) if wanted else 0)
    # more places than requests: every row
    e = entries([3] * n, n)
    for x in e:
        x.want = [0, 1, 2]
    assert wanted_rows(e, 256) == min(b for b in PORTION_ROWS if b >= 3 * n)
    # steps that are never captured: the places themselves
    assert wanted_rows(entries([PORTION_ROWS[-1] + 1] + [1] * (n - 1), n), 256) == n


@pytest.mark.gpu
@pytest.mark.parametrize("vocab", [12320, 50257])
def test_captured_steps_have_the_bits_of_steps_kernel_by_kernel(vocab):
    """A vocabulary's product of 17 rows and more is another kernel than that of up to 16: 20 requests of which 10 want their logits."""
    from denno_beta_amd.config import EngineOptions
    from denno_beta_amd.engine import ModelRunner
    cfg = dict(architectures=["GPT2LMHeadModel"], n_layer=1, n_embd=1024, n_head=16, vocab_size=vocab, n_positions=64, layer_norm_epsilon=1e-5,
               activation_function="gelu_new")
    got = []
    for graphs in (True, False):
        r = ModelRunner.from_random(cfg, 3, EngineOptions(dtype="bfloat16", page_size=16, max_live=32, cache_tokens=32 * 64, use_graphs=graphs))
        for i in range(20):
            r.start_request(i)
        steps = []
        for lengths in ([2] * 20, [2] * 20, [2] * 20, [1] * 20, [1] * 20):
            for wanted in (10, 20):
                out = r.step([StepEntry(e.rid, [(7 * e.rid + t) % vocab for t in e.tokens], e.want) for e in entries(lengths, wanted)])
                assert tuple(out.shape) == (wanted, vocab)
                steps.append(out.clone())
        if graphs:
            assert r.graphs.portions and r.graphs.graphs
        got.append(steps)
    for i, (a, b) in enumerate(zip(*got)):
        assert torch.equal(a, b), i
