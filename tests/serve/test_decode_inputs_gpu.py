"""Captured decode steps whose host runs ahead: the inputs of many steps in a row are staged without a wait in between, and every step still sees
its own tokens, positions, pages and lengths (against an engine without graphs)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3])
def test_steps_staged_ahead_of_the_device(rows):
    from llmctl.serve.engine import InferenceEngine
    from llmctl.serve.scheduler import PrefillChunk

    es = [InferenceEngine("tiny", device="cuda", max_batch_size=4, num_kv_blocks=64, block_size=16, max_model_len=256, use_graphs=g,
                          prefix_caching=False, seed=3) for g in (True, False)]
    gen = torch.Generator().manual_seed(0)
    toks = lambda n: torch.randint(0, 500, (n,), generator=gen).tolist()
    prompts, news = [toks(7 + 9 * i) for i in range(rows)], [toks(rows) for _ in range(24)]
    outs = []
    for e in es:
        seqs = []
        for p in prompts:
            s = e.open_sequence(p)
            e.prefill([PrefillChunk(s, 0, len(p))])
            e.scheduler.computed(s, len(p))
            seqs.append(s)
        got = []
        if e is es[0]:
            e._capture(e._bucket(rows))
            torch.cuda._sleep(200_000_000)  # the device is busy while the host stages the steps
        for new in news:
            for s, t in zip(seqs, new):
                e.scheduler.extend(s, [t])
                s._decode_slot = int(e.kv.slots(s.seq_id, s.num_tokens - 1, 1)[0])
            got.append(e.decode(seqs).clone())
            for s in seqs:
                e.scheduler.computed(s, 1)
        outs.append(got)
    for a, b in zip(*outs):
        assert (a.float() - b.float()).norm() <= 2e-2 * b.float().norm()  # bf16: an output may round the other way in every layer
