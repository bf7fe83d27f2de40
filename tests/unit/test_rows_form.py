"""The rule of the prompt products' tiles against the times that its figures are from: up to 1024 rows nothing that it takes is much slower than the library's product, whichever the
file, and what it takes for the host's sake costs the chip a few us."""
import importlib
import re
from pathlib import Path

import pytest

L = importlib.import_module("llmctl.exec.linear")
PROFILES = Path(__file__).resolve().parents[2] / "profiles"


def _times():
    """(rows, outputs, K, library's us, {(tiles, ranges of K): us})"""
    for name in ("few_rows_products.txt", "short_prompt_products.txt"):
        for line in (PROFILES / name).read_text().splitlines():
            if m := re.match(r"(\d+) (\d+) (\d+) \| ([\d.]+) \| \S+ \| (.*)$", line):
                yield *map(int, m.groups()[:3]), float(m[4]), {(int(a), int(b)): float(t) for a, b, t in re.findall(r"(\d):(\d+) ([\d.]+)", m[5])}
    for line in (PROFILES / "prompt_products.txt").read_text().splitlines():
        if m := re.match(r"(\d+) (\d+) (\d+) \| ([\d.]+) \| ([\d.]+) ([\d.]+) \|", line):
            yield *map(int, m.groups()[:3]), float(m[4]), {(1, 1): float(m[5]), (2, 1): float(m[6])}


def _picks(eager):
    for M, N, K, library, own in _times():
        code = L.rows_form(M, N, K, False, eager)
        form = code & 3, (code >> 2) + 1
        if M <= 1024 and code and form in own:
            yield M, N, K, library, own[form]


def test_picks_are_faster():
    picks = list(_picks(False))
    assert len(picks) >= 560 and all(own <= 1.26 * library and own <= library + 8.7 for *_, library, own in picks)
    assert sum(own > library for *_, library, own in picks) <= 40 and sum(own > library + 3.7 for *_, library, own in picks) <= 1
    assert sum(own for *_, own in picks) < 0.83 * sum(library for *_, library, _ in picks)


def test_choices_are_near_the_best():
    own = best = 0.0
    for M, N, K, library, ours in _times():
        code = L.rows_form(M, N, K)
        form = code & 3, (code >> 2) + 1
        if M <= 1024 and (not code or form in ours):
            own += ours[form] if code else library
            best += min(library, *ours.values())
    assert own < 1.032 * best


def test_what_the_host_saves_costs_the_chip_little():
    picks = list(_picks(True))
    assert len(picks) >= 950 and all(own <= library + 8.7 for *_, library, own in picks) and sum(own > library + 5.2 for *_, library, own in picks) <= 1
    assert sum(own for *_, own in picks) < 0.9 * sum(library for *_, library, _ in picks)


@pytest.mark.parametrize("M,N,K", [(900, 2048, 2048), (450, 3712, 2048), (350, 5136, 2048), (288, 6144, 2048), (288, 5136, 2048), (288, 32000, 2048), (100, 4096, 4096), (200, 8192, 2048), (1000, 11008, 512)])
def test_the_librarys(M, N, K):
    """(288 x 32000 x 2048 is more than the host's sake allows)"""
    assert L.rows_form(M, N, K) == 0 and (N < 32000 or L.rows_form(M, N, K, False, True) == 0)


def test_training_under_tensor_parallelism_does_not_ask_for_the_hosts_sake(monkeypatch):
    import torch

    tp = importlib.import_module("llmctl.parallel.async_tp")
    asked, own = [], L.forward_linear
    monkeypatch.setattr(L, "forward_linear", lambda x, w, b=None, layout="eager": asked.append(layout) or own(x, w, b, layout))
    monkeypatch.setattr(tp, "_matmul_rs", lambda x, group, mm: mm(x))
    x, w = torch.randn(4, 16), torch.randn(8, 16)
    out = torch.zeros(4, 12)[:, :8]
    tp._fwd_into(w, None)(x, out)
    y = tp._RowSP.apply(x, w, None)
    assert torch.equal(out, y) and torch.allclose(y, x @ w.t(), atol=1e-5) and len(asked) == 2 and "eager" not in asked


def test_a_vector_is_a_weight_too():
    import torch

    from llmctl.ops import hybrid as hops

    x, w = torch.randn(40, 16), torch.randn(16)
    for f in (hops.linear, hops.odd_linear):
        assert torch.equal(f(x, w), torch.nn.functional.linear(x, w))


def test_a_recording_takes_the_routes_of_the_steps_ahead_of_it(monkeypatch):
    """A library product that a recording is the first to call ends the process: the stream's state moves no product, and who records says so for the steps ahead too."""
    import threading
    import types

    import torch

    ran = []
    fake = types.SimpleNamespace(gemm_rows=lambda x, w, b, form, splits, act: ran.append((form, splits)) or torch.empty(x.shape[0], w.shape[0]),
                                 gemm_small=lambda x, w, y, *a: ran.append("small"))
    monkeypatch.setattr(L, "native", lambda: fake)
    monkeypatch.setattr(L, "_small_ok", lambda *a: True)

    def routes(M, N, K):
        x = torch.empty(M, K)
        w = types.SimpleNamespace(shape=(N, K), dim=lambda: 2, is_cuda=True, requires_grad=False, stride=lambda i: K)
        got = []
        for f in (lambda: L.rows_linear(x, w), lambda: L.small_linear(x, w, None, "eager"), lambda: L.small_linear_f32(x, w)):
            ran.clear()
            got.append((f() is not None, *ran))
        return got

    moved = 0
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    with torch.no_grad():
        for M, N, K in ((33, 3072, 1024), (40, 2048, 2048), (100, 1024, 1024), (256, 2048, 2048), (300, 768, 768), (300, 3072, 768), (1500, 1024, 512), (2048, 2048, 2048)):
            plain = routes(M, N, K)
            monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
            assert routes(M, N, K) == plain
            with L.recorded_step():
                recorded, other = routes(M, N, K), []
                t = threading.Thread(target=lambda: other.append(L._steps.recorded))
                t.start(), t.join()
                assert other == [False]
            monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
            with L.recorded_step():
                assert routes(M, N, K) == recorded
            assert routes(M, N, K) == plain
            code = L.rows_form(M, N, K)
            assert recorded[0] == ((True, (code & 3, (code >> 2) + 1)) if code else (False,)) and recorded[1][0] == L.small_pays("fwd", M, N, K) and not recorded[2][0]
            moved += recorded != plain
    assert moved >= 4
