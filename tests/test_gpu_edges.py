"""Kernels at the edges of their size ranges, against the oracle."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("props, atoms", [(7, "dense"), (64, "dense"), (65, "dense"), (130, "reachable"), (512, "dense"), (1000, "dense"),
                                          (130, "lazy"), (1090, "dense")])
def test_search_fingerprint_over_row_widths(props, atoms):
    """Narrow rows (1, 2, 4, 8 and 16 words: nibble tables), wider ones and lazily grown rows (a wave per row): the
    fingerprint does not depend on the slots, so a lazy search has the dense oracle's."""
    from mymyr_amd import gen, search
    from mymyr_amd.task import Task
    from oracle import port

    text = gen.random_strips(props, 60, init_atoms=max(3, props // 8), goal_atoms=2, seed=4)
    kw = dict(max_depth=2, stop_at_goal=False)
    r = search.brfs(Task.from_text(text, atoms), fingerprint=True, **kw)
    p = port.brfs(port.Task(text, "dense"), max_states=1 << 40, **kw)
    assert (r.states, r.fingerprint) == (p["states"], p["fingerprint"])
