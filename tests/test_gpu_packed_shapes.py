"""Packed levels at the sizes between which their launch changes: levels of too little
work for them (tuning key pk=2 packs those too, few nodes: three waves per SIMD),
levels of many small nodes (four waves per SIMD), byte for byte against the byte table
(pk=0), which the oracle tests cover, and the small ones against the oracle."""
import pytest

from oracle_lib import OracleMPHF, splitmix_keys

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import gpurecsplit_amd
    return gpurecsplit_amd


def _build(gra, keys, leaf, bucket, tune):
    ctx = gra.Context(0)
    ctx.set_tune(tune, leaf)
    rs = gra.GPURecSplit(keys, bucket, leaf_size=leaf, ctx=ctx)
    out, evals = rs.serialize(), rs.stats()["evals"]
    rs.close()
    ctx.close()
    return out, evals


@pytest.mark.parametrize("leaf,bucket,n", [
    (13, 65, 65), (13, 65, 3000), (14, 84, 1500), (15, 450, 2000), (15, 90, 90), (16, 112, 112), (16, 560, 1120),
    (16, 700, 6000), (17, 500, 1000), (18, 126, 252), (20, 160, 160),
])
def test_small_packed_levels_match_oracle(env, leaf, bucket, n):
    print(f"leaf={leaf} bucket={bucket} n={n}", flush=True)
    keys = splitmix_keys(leaf * 17 + bucket + n, n)
    exp = OracleMPHF.build(keys, leaf, bucket, threads=8).serialize()
    assert _build(env, keys, leaf, bucket, "pk=2")[0] == exp


@pytest.mark.parametrize("leaf,bucket,n", [(13, 2000, 600_000), (14, 100, 500_000), (15, 500, 200_000),
                                           (16, 2000, 60_000), (18, 2000, 20_000)])
def test_large_packed_levels_match_byte_table(env, leaf, bucket, n):
    print(f"leaf={leaf} bucket={bucket} n={n}", flush=True)
    keys = splitmix_keys(leaf + bucket + n, n)
    exp = _build(env, keys, leaf, bucket, "pk=0,tree=0")
    assert _build(env, keys, leaf, bucket, "pk=1,tree=0") == exp
    assert _build(env, keys, leaf, bucket, "pk=2,tree=0") == exp
