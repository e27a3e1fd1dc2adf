"""Staged leaf search: leaves at and around the smallest staged size (12 keys), every
leaf size whose first stage takes another number of keys, both parities of the
halves (a leaf's even keys may be the larger or the smaller half), sets that end
with a staged leaf, and both remaps, byte for byte against the oracle."""
import pytest

from oracle_lib import OracleMPHF, splitmix_keys

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gra():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gpurecsplit_amd
    return gpurecsplit_amd


@pytest.mark.parametrize("leaf,bucket,n,rotate,remap64", [
    (11, 33, 1500, True, False), (12, 12, 240, True, False), (12, 40, 4000, True, False), (13, 39, 2000, True, False),
    (14, 14, 400, True, False), (15, 45, 900, True, False), (16, 16, 320, True, False), (17, 30, 500, True, False),
    (18, 36, 720, True, False), (19, 19, 95, True, False), (20, 20, 60, True, False),
    (11, 30, 900, False, False), (12, 24, 600, False, False), (13, 13, 260, False, False), (14, 28, 280, False, False),
    (15, 15, 90, False, False), (12, 30, 900, True, True), (13, 26, 400, False, True), (16, 33, 330, True, True),
])
def test_staged_leaves_match_oracle(gra, leaf, bucket, n, rotate, remap64):
    print(f"leaf={leaf} bucket={bucket} n={n} rotate={rotate} remap64={remap64}", flush=True)
    keys = splitmix_keys(leaf * 131 + n, n)
    got = gra.GPURecSplit(keys, bucket, leaf_size=leaf, rotate=rotate, remap64=remap64).serialize()
    assert got == OracleMPHF.build(keys, leaf, bucket, rotate=int(rotate) | (2 if remap64 else 0), threads=8).serialize()
