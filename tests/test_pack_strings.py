"""Packing of string keys: the joined form equals the key-by-key form for every kind
of key list it may meet."""
import numpy as np
import pytest

gra = pytest.importorskip("gpurecsplit_amd")


@pytest.mark.parametrize("keys", [
    [], ["a"], ["", "", "x"], ["abc", "d" * 300, "ef"], ["naïve", "abc", "漢字", ""], [b"", b"ab\x00", b"\xff"],
    ["a", b"b", "c"], [b"b", "a"], [bytearray(b"xy"), b"z"], ["x", bytearray(b"y")], ("t", "u"), [b"a", bytearray(b"bc")],
])
def test_packed_bytes_and_offsets(keys):
    blob, off = gra._pack_strings(keys)
    each = [k.encode() if isinstance(k, str) else bytes(k) for k in keys]
    assert blob == b"".join(each)
    assert off.dtype == np.uint64 and off.tolist() == np.cumsum([0] + [len(b) for b in each]).tolist()
    blob2, off2 = gra._pack_strings(k for k in keys)
    assert blob2 == blob and np.array_equal(off, off2)
