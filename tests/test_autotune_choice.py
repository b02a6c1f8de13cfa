"""Which settings the autotuner keeps (oak_amd/autotune.py): the graph only where its
replays gain more than runs of one setting differ (no GPU)."""
import json

import pytest

from oak_amd import autotune


def _times(*rows):
    return {json.dumps(dict(zip(("graph", "order", "slots"), r[:3])), sort_keys=True): r[3] for r in rows}


@pytest.mark.parametrize("plain,graph,chosen", [
    (39.889, 39.869, 0), (35.244, 35.202, 0), (28.026, 27.996, 0), (100.0, 98.5, 0),
    (100.0, 97.0, 1), (2.0, 1.2, 1), (1.0, 1.0, 0), (1.0, 3.0, 0)])
def test_graph_has_to_gain(plain, graph, chosen):
    t = _times((0, 0, 2, plain * 1.01), (0, 1, 3, plain), (1, 1, 3, graph), (1, 0, 4, graph * 1.02))
    s = autotune.choose(t)
    assert s["graph"] == chosen
    assert (s["order"], s["slots"]) == (1, 3)


def test_space_without_the_other():
    assert autotune.choose(_times((1, 0, 2, 5.0), (1, 1, 3, 4.0))) == {"graph": 1, "order": 1, "slots": 3}
    assert autotune.choose({'{"slots": 2}': 5.0, '{"slots": 3}': 4.9}) == {"slots": 3}


def test_shipped_table_follows_the_rule():
    for k, ent in autotune.load_table().items():
        assert ent["settings"] == autotune.choose(ent["ms"]), k
