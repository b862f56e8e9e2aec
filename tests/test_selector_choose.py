"""LearnedSelector.encode goes by its own `choose` (no GPU: the library calls are
recorded): one replaced in a subclass, on an instance or on the class steers the
encode, and the class's own runs as statistics, network and resolve."""
from types import SimpleNamespace

import pytest

from fastlanesgpu_amd import selector as sel


def workspace():
    return SimpleNamespace(cls=1, vmeta=2, aux=3, words=4, total=5, fallbacks=6, scratch=7, feat=8, conf=9,
                           stats_n=None, ready=None)


def fixed_choice(self, d_in, n, ws, stream=None):
    """Another rule's classes and confidences."""
    self.seen = (d_in, n, ws, stream)


@pytest.mark.parametrize("where", ["subclass", "instance", "class", "nowhere"])
def test_encode_takes_the_choice_of_choose(monkeypatch, where):
    calls = []
    monkeypatch.setattr(sel, "call", lambda name, *a: calls.append(name))
    cls = sel.LearnedSelector
    if where == "subclass":
        cls = type("Fixed", (sel.LearnedSelector,), {"choose": fixed_choice})
    elif where == "class":
        monkeypatch.setattr(sel.LearnedSelector, "choose", fixed_choice)
    learned = cls(SimpleNamespace(wb=11), conf_min=0.5)
    if where == "instance":
        learned.choose = fixed_choice.__get__(learned)
    ws = workspace()
    learned.encode(16, 5000, ws, 0)
    if where == "nowhere":
        assert calls == ["fls_mixed_stats_device", "fls_mlp_forward", "fls_mixed_resolve_device",
                         "fls_mixed_pack_device"]
    else:
        assert learned.seen == (16, 5000, ws, 0)
        assert calls == ["fls_mixed_plan_device", "fls_mixed_pack_device"]
