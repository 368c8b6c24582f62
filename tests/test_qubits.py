"""Qubit classes of a user's own: hashing, copying and pickling are those of plain Python objects."""

import copy
import dataclasses
import pickle

import pytest

import cirq_amd as cirq
from cirq_amd.qubits import Qid


@dataclasses.dataclass(frozen=True, eq=False)
class FrozenQubit(Qid):
    label: str

    def _comparison_key(self):
        return (self.label,)


class SlottedQubit(Qid):
    __slots__ = ("label",)

    def __init__(self, label):
        self.label = label

    def _comparison_key(self):
        return (self.label,)


class OffsetQubit(cirq.LineQubit):
    """A subclass of a built-in qubit whose key is its own and may change."""

    offset = 0

    def _comparison_key(self):
        return (self._x + self.offset,)


@pytest.mark.parametrize("cls", [FrozenQubit, SlottedQubit])
def test_hash_copy_and_pickle_of_subclasses(cls):
    q, same, other = cls("a"), cls("a"), cls("b")
    assert hash(q) == hash(same) and {q: 1}[same] == 1 and q != other
    for twin in (copy.copy(q), copy.deepcopy(q), pickle.loads(pickle.dumps(q)), pickle.loads(pickle.dumps(q, 2))):
        assert twin == q and hash(twin) == hash(q) and twin.label == "a"
    assert sorted([other, q]) == [q, other]


def test_hash_follows_the_key():
    q = OffsetQubit(3)
    before = hash(q)
    q.offset = 2
    assert hash(q) != before and hash(q) == hash(q._cmp_tuple())


@dataclasses.dataclass(frozen=True, eq=False)
class FrozenLineQubit(cirq.LineQubit):
    _x: int = 0


@pytest.mark.parametrize("q", [cirq.LineQubit(7), cirq.GridQubit(2, -1), cirq.NamedQubit("a12b3"), OffsetQubit(4), FrozenLineQubit(3)])
def test_hash_is_that_of_the_comparison_tuple(q):
    plain = dict(vars(q))
    for _ in range(2):
        assert hash(q) == hash(q._cmp_tuple())
    for twin in (copy.copy(q), copy.deepcopy(q), *(pickle.loads(pickle.dumps(q, k)) for k in range(pickle.HIGHEST_PROTOCOL + 1))):
        assert vars(twin) == plain  # no hash of this process
        assert twin == q and hash(twin) == hash(q)


def test_attributes_of_builtin_qubits_are_copied():
    q = cirq.LineQubit(1)
    hash(q)
    q.note = "kept"
    assert copy.copy(q).note == pickle.loads(pickle.dumps(q)).note == "kept"
