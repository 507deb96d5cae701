"""The binding's weight structs, without a device."""
from types import SimpleNamespace

import fusekit_amd.native as fk


def _weight():
    W = fk.DeviceWeight.__new__(fk.DeviceWeight)
    W.n, W.k, W.bits, W.group = 48, 128, 4, 64
    W.w, W.scales, W.biases = (SimpleNamespace(ptr=p) for p in (0x1000, 0x2000, 0x3000))
    return W


def _fields(c):
    return c.w, c.scales, c.biases, c.n, c.k, c.bits, c.group


def test_a_struct_that_a_caller_changes_is_not_the_operators():
    W = _weight()
    whole = _fields(W.c)
    for _ in range(2):                       # before and after an operator has made its own
        mine = W.c
        mine.n, mine.w = 16, 0x1400          # a piece of the matrix
        assert _fields(W.c) == whole and _fields(mine)[3] == 16
        assert _fields(fk._w(W)) == whole


def test_operators_follow_a_weight_s_buffers_and_sizes():
    W = _weight()
    fk._w(W)
    W.w.ptr = 0x9000                         # the buffer's own address
    assert fk._w(W).w == 0x9000
    W.scales = SimpleNamespace(ptr=0xA000)   # another buffer
    W.n = 32
    assert _fields(fk._w(W)) == _fields(W.c) == (0x9000, 0xA000, 0x3000, 32, 128, 4, 64)
    W.bits, W.scales, W.biases = 16, None, None
    assert _fields(fk._w(W)) == (0x9000, None, None, 32, 128, 16, 64)


def test_an_operand_with_a_struct_of_its_own_is_taken_by_that():
    c = fk.Weight(1, 2, 3, 4, 64, 4, 64)
    assert fk._w(SimpleNamespace(c=c)) is c
