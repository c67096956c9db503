"""The autotuner's choice among candidates timed at one and at several sizes (CPU)."""
import importlib
import os

import pytest


@pytest.fixture
def weigh():
    kept = os.environ.get("DGK_NO_TUNING")
    try:
        return importlib.import_module("autotune").weigh  # sets the variable for its own process
    finally:
        if kept is None:
            del os.environ["DGK_NO_TUNING"]
        else:
            os.environ["DGK_NO_TUNING"] = kept


def test_weigh(weigh):
    a, b, c = (2, 100, 0, 0), (2, 100, 1, 6), (2, 200, 0, 6)
    assert weigh([{a: 10.0, b: 9.0, c: 9.5}])[0] == b
    assert weigh([{a: 10.0, b: 9.9, c: 9.95}])[0] == a  # another shape by less than 2%
    # b best at the first size, c over both: (1.056 * 1.0) < (1.0 * 1.2)
    best, score = weigh([{a: 10.0, b: 9.0, c: 9.5}, {a: 2.0, b: 1.8, c: 1.5}])
    assert best == c
    assert score[c] == pytest.approx((9.5 / 9.0) ** 0.5) and score[b] == pytest.approx(1.2 ** 0.5)
    assert weigh([{a: 10.0, b: 5.0}, {a: 1.0, c: 0.5}])[0] == a  # candidates of both sizes only
    # the candidate in use stays within 4% of the choice
    assert weigh([{a: 10.0, b: 9.9, c: 10.3}], c)[0] == c
    assert weigh([{a: 10.0, b: 9.0, c: 9.3}], c)[0] == c
    assert weigh([{a: 10.0, b: 9.0, c: 9.5}], c)[0] == b
    assert weigh([{a: 10.0, b: 9.0}], c)[0] == b
