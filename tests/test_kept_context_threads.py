"""The context that is kept after its collection, where two threads collect at
once: between any two steps of one collection the other may empty the list or
fill it.  Every context is closed or kept, and one at most is kept."""
import pytest

import rawspec_amd as R
from tests.test_view_lifetime import _Stub


class _Shared(list):
    """Another collection (`other`) runs right before the list's n-th pop or
    append."""

    def __init__(self, items, method, n, other):
        super().__init__(items)
        self.at, self.n, self.other = method, n, other

    def _step(self, method):
        if method == self.at:
            self.n -= 1
            if self.n == 0:
                self.other(self)

    def pop(self):
        self._step("pop")
        return super().pop()

    def append(self, sp):
        self._step("append")
        super().append(sp)


def _lent(closed):
    sp = _Stub(closed)
    sp.initialized = sp._lent = True
    return sp


def _empty(kept):
    taken = list(kept)
    kept.clear()
    for sp in taken:
        sp.close()


@pytest.mark.parametrize("method", ["pop", "append"])
@pytest.mark.parametrize("n", [1, 2])
@pytest.mark.parametrize("other", ["empties", "fills"])
@pytest.mark.parametrize("before", [0, 1])
def test_two_threads_collect(monkeypatch, method, n, other, before):
    closed = []
    keep = [_lent(closed) for _ in range(before)]
    mine, theirs = _lent(closed), _lent(closed)
    serials = {sp._serial for sp in keep + [mine]}

    def fill(kept):
        serials.add(theirs._serial)
        list.append(kept, theirs)

    kept = _Shared(keep, method, n, _empty if other == "empties" else fill)
    monkeypatch.setattr(R, "_kept", kept)
    mine.__del__()
    left = [sp._serial for sp in kept]
    assert len(left) <= 1
    assert sorted(closed + left) == sorted(serials)
    # the stubs' own collection closes them
    for sp in keep + [mine, theirs]:
        sp._lent = False
