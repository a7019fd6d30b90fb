"""The largest trees whose chunk summaries fit LDS beside the node arrays of a banded par sweep: a plan that is asked for is
made, and its sweeps equal the dense kernel's."""
import numpy as np
import pytest

from treesa_gpu_amd import capi, host

pytestmark = pytest.mark.gpu


def test_largest_banded_summaries():
    m, nlab = 5133, 8320  # two summary words per set; one tensor more does not fit
    rng = np.random.RandomState(3)
    ixs = [[] for _ in range(m)]
    for x in range(nlab):
        for v in rng.choice(m, 2, replace=False):
            ixs[v].append(x)
    inst = host.Instance(m=m, nlab=nlab, ixs=ixs, iy=[])
    lay = capi.layout(m, nlab, True)
    pop = inst.population(lay, host.random_tree(m, 5)[None], 2, seed=5)
    out = []
    for sums in (1, -1):
        cfg = capi.make_config(sc_target=8.0, seed=5, par_band=4, sums=sums, wide_wgs=1)
        with capi.Context(lay, inst.leaf(lay.W), inst.leaf_sc, cfg, 2) as ctx:
            assert f" sums={2 if sums > 0 else 0} " in ctx.describe()
            ctx.upload(pop)
            ctx.sweeps(capi.ORDER_PAR, 2.0, 0, 1)
            out.append(list(ctx.energy()) + [ctx.download()])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    lay = capi.layout(m + 1, nlab, True)
    inst = host.Instance(m=m + 1, nlab=nlab, ixs=ixs + [[0]], iy=[])
    with pytest.raises(capi.TsaError):
        capi.Context(lay, inst.leaf(lay.W), inst.leaf_sc, capi.make_config(par_band=4, sums=1, wide_wgs=1), 2)
