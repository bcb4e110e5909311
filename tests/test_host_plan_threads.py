"""The register programs of a column, compiled when first asked for, by several
threads at once: compiled once, and whole for each of them."""
import os
import sys
import threading
import time

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(__file__))
from test_host_column import _random_model, _ray, _trace  # noqa: E402

from temgymcore_amd import _program  # noqa: E402


@pytest.mark.parametrize("which", ["plan", "template"])
def test_programs_are_compiled_once(which):
    model = _random_model(np.random.default_rng(3), 5)
    ray = _ray()
    tr, sym, out = _trace(ray, model)
    owner = _program.build_plan(tr, out, sym_in=sym)
    if which == "template":
        leaves = []
        _program._structure_key((tuple(model), ray), leaves, {})
        owner = _program._PlanTemplate(owner, leaves)
    compile_, calls = owner._programs, []

    def slow():
        calls.append(1)
        time.sleep(0.05)
        return compile_()

    owner._programs = slow
    got, errors, barrier = [], [], threading.Barrier(4)

    def ask():
        barrier.wait()
        try:
            got.append(owner.programs)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=ask) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors and len(calls) == 1 and len(got) == 4
    assert all(g is got[0] for g in got) and len(got[0]) >= 1
