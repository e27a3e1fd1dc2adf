"""Buckets above 512 keys as whole trees, a workgroup each: just past that size, near the
bucket limit, one bucket and many, both leaf modes and remaps, byte for byte against
the oracle, by an ordinary build, a plan and the level kernels; a duplicate key."""
import numpy as np
import pytest

from oracle_lib import OracleMPHF, splitmix_keys

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gpurecsplit_amd
    return gpurecsplit_amd, torch


@pytest.mark.parametrize("leaf,bucket,n,rotate,remap64", [
    (2, 600, 5000, True, False), (3, 2000, 2000, True, False), (4, 1000, 5908, True, False),
    (4, 2700, 27_000, True, False), (6, 530, 300_000, True, False), (8, 1000, 9001, True, True),
    (8, 2000, 100_000, True, False), (9, 513, 513, True, False), (10, 2600, 26_000, True, False),
    (10, 700, 40_000, False, False), (10, 900, 9000, False, True), (11, 1000, 9000, True, False),
])
def test_large_trees_match_oracle(env, leaf, bucket, n, rotate, remap64):
    gra, torch = env
    print(f"leaf={leaf} bucket={bucket} n={n} rotate={rotate} remap64={remap64}", flush=True)
    keys = splitmix_keys(leaf * 31 + bucket + n, n)
    exp = OracleMPHF.build(keys, leaf, bucket, rotate=int(rotate) | (2 if remap64 else 0), threads=8).serialize()
    rs = gra.GPURecSplit(keys, bucket, leaf_size=leaf, rotate=rotate, remap64=remap64)
    assert rs.serialize() == exp
    plan = gra.Plan(n, bucket, leaf, rotate=rotate, remap64=remap64)
    d = torch.from_numpy(keys.view(np.int64)).cuda()
    assert plan.build(d) == exp
    assert plan.build(d) == exp
    plan.close()
    ctx = gra.Context(0)
    ctx.set_tune("tree=0", leaf)
    level = gra.GPURecSplit(keys, bucket, leaf_size=leaf, rotate=rotate, remap64=remap64, ctx=ctx)
    assert level.serialize() == exp
    for k in ("evals", "seeds", "nodes"):
        assert level.stats()[k] == rs.stats()[k], k
    ctx.close()


def test_duplicate_key_in_a_large_bucket(env):
    gra, _ = env
    keys = splitmix_keys(5, 8000)
    keys[7000] = keys[3]
    with pytest.raises(gra.RecSplitError, match="(?i)duplicate"):
        gra.GPURecSplit(keys, 1500, leaf_size=8)
