"""A prompt's layers from one native call: the same bits as the engine's loop over its layers, on every route of the products; and who keeps the loop."""
import dataclasses
import json

import pytest
import torch

pytestmark = pytest.mark.gpu


def _engine(tmp_path, **kw):
    from llmctl.models import get_model_config
    from llmctl.serve.engine import InferenceEngine

    cfg = dataclasses.replace(get_model_config("gpt2-125m"), layers=2, **kw)
    path = tmp_path / "model.json"
    path.write_text(json.dumps(cfg.to_dict()))
    eng = InferenceEngine(str(path), device="cuda", max_batch_size=4, max_batch_tokens=8192, max_model_len=1024, block_size=16, num_kv_blocks=200,
                          prefix_caching=False, seed=3)
    torch.manual_seed(5)
    with torch.no_grad():
        for n, p in eng.model.named_parameters():
            if p.dim() == 1:
                p.add_(0.1 * torch.randn_like(p))
    return eng


def _step(eng, lens, seed=0):
    from llmctl.serve.scheduler import PrefillChunk

    g = torch.Generator().manual_seed(seed)
    seqs = [eng.open_sequence(torch.randint(0, eng.cfg.vocab_size, (n,), generator=g).tolist()) for n in lens]
    logits = eng.prefill([PrefillChunk(s, 0, s.num_tokens) for s in seqs])
    for s in reversed(seqs):
        eng.scheduler.finish(s, "stop")
    return logits, eng.kv_cache.k.clone(), eng.kv_cache.v.clone()


@pytest.mark.parametrize("lens", [(33,), (40, 1), (100,), (300,), (450,), (257, 300, 43), (1000,), (1000, 900, 77)])
@pytest.mark.parametrize("kw", [{}, dict(hidden=512, heads=4, kv_heads=2, ffn=2048)])
def test_same_bits_as_the_loop(tmp_path, lens, kw):
    eng = _engine(tmp_path, **kw)
    calls, own = [], eng._prompt_layers
    eng._prompt_layers = lambda *a: calls.append(own(*a)) or calls[-1]
    got = _step(eng, lens)
    assert len(calls[0]) == 2
    eng = _engine(tmp_path, **kw)  # (whose cache hands out the same blocks)
    eng._prompt_layers = lambda *a: ()
    for a, b in zip(got, _step(eng, lens)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("lens,route", [((100,), "small"), ((1000,), "tiles"), ((1000, 900, 850), "library")])
def test_routes_of_the_gelu(tmp_path, lens, route):
    """The up projection on gemm_small, on the prompt tiles, and as the library's product with a pass for the GELU."""
    from llmctl.exec.linear import prompt_forms

    eng = _engine(tmp_path)
    x = torch.empty(sum(lens), eng.cfg.hidden, device="cuda", dtype=torch.bfloat16)
    with torch.inference_mode():
        form, = prompt_forms(x, ((eng.cfg.ffn, eng.cfg.hidden, True),))
    assert route == ("small" if form < 0 else "tiles" if form else "library")
    test_same_bits_as_the_loop(tmp_path, lens, {})


def test_patched_methods_and_ops_keep_the_loop(tmp_path, monkeypatch):
    from llmctl import ops
    from llmctl.serve.engine import InferenceEngine

    eng = _engine(tmp_path)
    run = lambda: eng._prompt_layers(torch.randn(64, 768, device="cuda", dtype=torch.bfloat16), torch.full((64,), -1, device="cuda"), None)
    with torch.inference_mode():
        assert len(run()) == 2
        for where, name in ((InferenceEngine, "_mlp"), (InferenceEngine, "_norm"), (ops, "flash_attention"), (ops, "decode_linear")):
            own = getattr(where, name)
            with monkeypatch.context() as m:
                m.setattr(where, name, lambda *a, **k: own(*a, **k))
                assert not run()
        assert len(run()) == 2


def test_others_keep_the_loop(tmp_path):
    eng = _engine(tmp_path)
    run = lambda n: eng._prompt_layers(torch.randn(n, 768, device="cuda", dtype=torch.bfloat16), torch.full((n,), -1, device="cuda"), None)
    with torch.inference_mode():
        assert len(run(64)) == 2 and not run(32)
        layer = eng.model.layers[1]
        keep = layer.w_up
        layer.w_up = torch.nn.Parameter(torch.randn(keep.shape[1], keep.shape[0], device="cuda", dtype=torch.bfloat16).t(), requires_grad=False)
        assert not run(64)  # a weight whose rows are not contiguous
        layer.w_up = torch.nn.Parameter(keep.float(), requires_grad=False)
        assert not run(64)
        layer.w_up = keep
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not run(64)
        eng._mlp = eng._mlp
        assert not run(64)
