"""Packed aggregation search: every leaf size whose levels use it (both field widths,
fans 5 to 9), sets of one node, many nodes and nodes of other sizes beside the full
ones, byte for byte against the oracle, through the ordinary build and a plan; the
kernels it replaces (tuning key pk off) build the same bytes."""
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


@pytest.mark.parametrize("leaf,bucket,n", [
    (13, 65, 65), (13, 65, 3000), (14, 84, 1500), (15, 450, 2000), (15, 90, 90), (16, 112, 112), (16, 560, 1120),
    (16, 700, 6000), (17, 500, 1000), (18, 126, 252), (20, 160, 160),
])
def test_packed_levels_match_oracle(env, leaf, bucket, n):
    gra, torch = env
    print(f"leaf={leaf} bucket={bucket} n={n}", flush=True)
    keys = splitmix_keys(leaf * 17 + bucket + n, n)
    exp = OracleMPHF.build(keys, leaf, bucket, threads=8).serialize()
    assert gra.GPURecSplit(keys, bucket, leaf_size=leaf).serialize() == exp
    d = torch.from_numpy(keys.view(np.int64)).cuda()
    plan = gra.Plan(n, bucket, leaf)
    assert plan.build(d) == exp
    plan.close()
    ctx = gra.Context(0)
    ctx.set_tune("pk=0", leaf)
    assert gra.GPURecSplit(keys, bucket, leaf_size=leaf, ctx=ctx).serialize() == exp
    ctx.close()
