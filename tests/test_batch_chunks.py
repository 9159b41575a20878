"""Batch.chunks is a list that makes its chunks on demand (no GPU: the handles
come from a stand-in for the library)."""
import copy

import pytest

from buff_amd import _native as N

COUNT = 5


class Lib:
    def __init__(self):
        self.calls = []

    def buff_batch_chunk(self, batch, i, h):
        self.calls.append(i)
        h._obj.value = 1000 + i
        return 0


@pytest.fixture
def made(monkeypatch):
    fake = Lib()
    monkeypatch.setattr(N, "lib", lambda: fake)
    return N._BatchChunks(None, 1, COUNT), fake


def handles(chunks):
    return [c.handle for c in chunks]


WHOLE = [1000 + i for i in range(COUNT)]


def test_an_index_makes_one(made):
    chunks, fake = made
    assert len(chunks) == COUNT and bool(chunks) and fake.calls == []
    assert chunks[-1].handle == 1004 and chunks[4] is chunks[-1] and fake.calls == [4]
    assert handles(chunks[1:3]) == [1001, 1002] and type(chunks[1:3]) is list and fake.calls == [4, 1, 2]
    for i in (COUNT, -COUNT - 1):
        with pytest.raises(IndexError):
            chunks[i]
    with pytest.raises(TypeError):
        chunks["0"]


# every way a list is read or changed sees the chunks, not the places kept for them
@pytest.mark.parametrize("use, want", [
    (lambda c: handles(c), WHOLE),
    (lambda c: handles(list(c)), WHOLE),
    (lambda c: handles([*c]), WHOLE),
    (lambda c: handles(tuple(c)), WHOLE),
    (lambda c: handles(reversed(c)), WHOLE[::-1]),
    (lambda c: handles(c.copy()), WHOLE),
    (lambda c: handles(copy.copy(c)), WHOLE),
    (lambda c: handles(c + []), WHOLE),
    (lambda c: handles([] + c), WHOLE),
    (lambda c: handles(c * 2), WHOLE * 2),
    (lambda c: handles(2 * c), WHOLE * 2),
    (lambda c: handles(sorted(c, key=lambda k: -k.handle)), WHOLE[::-1]),
    (lambda c: [a.handle for a, _ in zip(c, c)], WHOLE),
    (lambda c: (c.reverse(), handles(c))[1], WHOLE[::-1]),
    (lambda c: (c.pop(0).handle, handles(c)), (1000, WHOLE[1:])),
    (lambda c: (c.append(7), c[-1], len(c))[1:], (7, COUNT + 1)),
    (lambda c: (c.__delitem__(0), handles(c))[1], WHOLE[1:]),
    (lambda c: None in c, False),
    (lambda c: c == [None] * COUNT, False),
    (lambda c: [None] * COUNT == c, False),
    (lambda c: c == list(c) and list(c) == c and not c != c[:], True),
    (lambda c: c.index(c[3]), 3),
    (lambda c: c.count(c[2]), 1),
    (lambda c: "None" in repr(c), False),
])
def test_list(made, use, want):
    chunks, _ = made
    assert isinstance(chunks, list) and use(chunks) == want


def test_extend_and_slice_assignment(made):
    chunks, _ = made
    a = [0]
    a += chunks
    assert handles(a[1:]) == WHOLE
    b = [0, 1, 2]
    b[1:2] = chunks
    assert handles(b[1:-1]) == WHOLE


def test_drop(made):
    chunks, fake = made
    first, gone = chunks[0], chunks[1]
    chunks.remove(gone)
    chunks.drop()
    assert first.handle is None and gone.handle is None and handles(chunks) == [None] * (COUNT - 1)


def test_drop_before_use(made):
    chunks, fake = made
    chunks.drop()
    assert handles(chunks) == [None] * COUNT and fake.calls == []
