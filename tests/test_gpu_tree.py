"""Whole trees of small buckets in one kernel: one wave per bucket (many buckets), a
workgroup per bucket (few), buckets of 0, 1, 2 and exactly leaf-size keys, buckets at
the kernel's size limit and past it, both remaps and leaf modes, byte for byte against
the oracle; a plan whose keys crowd one bucket beyond its likely size; duplicates."""
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


def _oracle(keys, leaf, bucket, rotate=True, remap64=False):
    return OracleMPHF.build(keys, leaf, bucket, rotate=int(rotate) | (2 if remap64 else 0), threads=8).serialize()


@pytest.mark.parametrize("leaf,bucket,n,rotate,remap64", [
    (8, 100, 1, True, False), (8, 100, 2, True, False), (8, 8, 800, True, False), (8, 1, 500, True, False),
    (2, 3, 7000, True, False), (5, 5, 30000, True, False), (8, 100, 250_000, True, False), (9, 60, 4000, True, False),
    (10, 450, 9000, True, False), (10, 480, 20000, True, False), (10, 520, 6000, True, False), (12, 12, 600, True, False),
    (12, 100, 700, True, False), (12, 100, 60_000, True, False), (13, 26, 5000, True, False),
    (8, 100, 9000, False, False), (11, 50, 5000, False, False), (8, 100, 30_000, True, True), (12, 60, 3000, True, True),
    (7, 70, 2000, False, True),
])
def test_trees_match_oracle(env, leaf, bucket, n, rotate, remap64):
    gra, torch = env
    print(f"leaf={leaf} bucket={bucket} n={n} rotate={rotate} remap64={remap64}", flush=True)
    keys = splitmix_keys(leaf * 1009 + bucket + n, n)
    exp = _oracle(keys, leaf, bucket, rotate, remap64)
    rs = gra.GPURecSplit(keys, bucket, leaf_size=leaf, rotate=rotate, remap64=remap64)
    assert rs.serialize() == exp
    plan = gra.Plan(n, bucket, leaf, rotate=rotate, remap64=remap64)
    assert plan.build(torch.from_numpy(keys.view(np.int64)).cuda()) == exp
    plan.close()
    ctx = gra.Context(0)
    ctx.set_tune("tree=0", leaf)
    level = gra.GPURecSplit(keys, bucket, leaf_size=leaf, rotate=rotate, remap64=remap64, ctx=ctx)
    assert level.serialize() == exp
    for k in ("evals", "seeds", "nodes"):
        assert level.stats()[k] == rs.stats()[k], k
    ctx.close()


def test_plan_with_a_crowded_bucket(env):
    """One bucket of 900 keys where 100 are expected: the plan's second tree launch."""
    gra, torch = env
    keys = splitmix_keys(31, 20_000)
    keys[:800, 0] = np.uint64(5)
    print("plan leaf=8 bucket=100 crowded", flush=True)
    exp = _oracle(keys, 8, 100)
    plan = gra.Plan(20_000, 100, 8)
    d = torch.from_numpy(keys.view(np.int64)).cuda()
    assert plan.build(d) == exp
    fresh = splitmix_keys(32, 20_000)
    assert plan.build(torch.from_numpy(fresh.view(np.int64)).cuda()) == _oracle(fresh, 8, 100)
    assert plan.build(d) == exp
    plan.close()
    assert gra.GPURecSplit(keys, 100, leaf_size=8).serialize() == exp


@pytest.mark.parametrize("n", [3000, 300_000])
def test_duplicates_are_reported_and_the_context_recovers(env, n):
    gra, _ = env
    print(f"duplicates n={n}", flush=True)
    keys = splitmix_keys(77, n)
    good = keys.copy()
    keys[n - 1] = keys[17]
    with pytest.raises(gra.RecSplitError) as e:
        gra.GPURecSplit(keys, 100, leaf_size=8)
    assert e.value.code == 4
    assert gra.GPURecSplit(good, 100, leaf_size=8).serialize() == _oracle(good, 8, 100)
