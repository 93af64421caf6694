"""The dict that MemoryPool.lookup returns: what it makes on first access
(_Views) is there for every dict operation."""

import copy

import pytest
import torch

from model_amd.memory import _Result, _Views

NAMES = ("q", "slots", "weights")


def _result():
    made = []

    def make(name, v):
        def f():
            made.append(name)
            return v
        return f

    views = _Views({n: make(n, torch.full((2,), float(i))) for i, n in enumerate(NAMES)})
    return _Result({"out": torch.ones(2), "staged": None}, views), views, made


def test_reading_one_key_makes_one_view():
    res, views, made = _result()
    assert res["out"] is not None and made == []
    assert res["slots"] is res["slots"] is views["slots"] and made == ["slots"]
    with pytest.raises(KeyError):
        res["nothing"]


@pytest.mark.parametrize("look", [
    lambda r: [k for k in ("out", "staged", *NAMES) if k in r],
    lambda r: [k for k in ("out", "staged", *NAMES) if r.get(k, NAMES) is not NAMES],
    lambda r: list(r.keys()), lambda r: [k for k, _ in r.items()], lambda r: list(r), lambda r: list(dict(r)),
    lambda r: list({**r}), lambda r: list(r.copy()), lambda r: list({} | r), lambda r: list(r | {}),
    lambda r: list(reversed(r))[::-1], lambda r: list(copy.copy(r)), lambda r: list(copy.deepcopy(r)),
    lambda r: [r.popitem()[0] for _ in range(len(r))],
])
def test_every_dict_operation_sees_all_keys(look):
    res, _, _ = _result()
    want = [k for k in ("out", "staged", *NAMES)]
    res["weights"]  # one of them read before
    assert sorted(look(res)) == sorted(want)
    res, _, _ = _result()
    assert len(res) == 5 and len(list(res.values())) == 5 and "nothing" not in res and res.get("nothing") is None
    assert "q_hat" not in res  # made by a kernel, only where it is read


def test_caller_changes_stay():
    res, _, made = _result()
    res["slots"] = 3
    assert res.pop("q") is not None and "q" not in res and res.get("q") is None
    with pytest.raises(KeyError):
        res["q"]
    del res["weights"]
    assert sorted(res) == ["out", "slots", "staged"] and res["slots"] == 3 and "slots" not in made
    assert res.setdefault("weights", 5) == 5
    res.clear()
    assert len(res) == 0 and not list(res)
