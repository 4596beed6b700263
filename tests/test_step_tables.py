"""The flat table of a step, whose neighbouring single tokens are described together: against its definition, entry by entry."""
import numpy as np
import pytest
import torch

from nanoinfer_amd.engine.runner import StepContext, StepEntry, StepError
from test_runner_books import make_runner


def _ready(lengths, done):
    runner = make_runner()
    entries = [StepEntry(f"r{i}", [(7 * i + 3 * k) % 97 for k in range(n)], [n - 1]) for i, n in enumerate(lengths)]
    runner._done = {e.request: d for e, d in zip(entries, done)}
    assert runner.cache.reserve_all([(e.request, d + len(e.tokens)) for e, d in zip(entries, done)])
    return runner, entries


@pytest.mark.parametrize("lengths", [[1], [5], [1, 1, 1], [1, 4, 1, 1], [9, 1], [1, 1, 20], [3, 2], [1, 2, 1, 3, 1]])
def test_tables_follow_their_definition(lengths):
    done = [(0, 7, 8, 30, 15)[i % 5] for i in range(len(lengths))]
    runner, entries = _ready(lengths, done)
    flat, layout, n_rows = runner._describe(entries, StepContext(runner.device))
    ps, group, T = runner.page_size, runner.cache.groups[0], sum(lengths)
    want = [t for e in entries for t in e.tokens]
    want += [d + k for n, d in zip(lengths, done) for k in range(n)]
    want += [i for i, n in enumerate(lengths) for _ in range(n)]
    want += [sum(lengths[:i + 1]) - 1 for i in range(len(lengths))]
    want += [group.tables[e.request][(d + k) // ps] * ps + (d + k) % ps for e, d in zip(entries, done) for k in range(len(e.tokens))]
    assert flat.dtype == np.int32 and flat[:len(want)].tolist() == want
    assert n_rows == len(lengths) and layout.groups[0][0] == 3 * T + n_rows


@pytest.mark.parametrize("lengths,who", [([1, 1], 1), ([4, 1], 1), ([1, 4], 1), ([1, 4, 1], 0)])
def test_a_page_given_back_is_refused(lengths, who):
    runner, entries = _ready(lengths, [9] * len(lengths))
    runner.cache.groups[0].tables[f"r{who}"][1] = -1
    with pytest.raises(StepError, match=f"'r{who}': position 9 "):
        runner._describe(entries, StepContext(runner.device))
