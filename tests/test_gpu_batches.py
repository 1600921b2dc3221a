"""Batches past the sizes at which the step changes its form: acoustic levels streamed past the caches
(three levels above 256 MiB), elastic steps of several shots per workgroup, and of 6144 tiles x
shots and more, whose point sources and receivers run in a launch of their own.  Three shots of the batch against the FP64 oracle (the other
shots' adjoint sources are zero, so the gradient is the three shots'), with the engines'
tolerances: traces within twice the FP32 gap of the oracle itself (at least 1e-5), gradients within
1e-4.  The same three shots alone, which take the other form, agree too: the acoustic traces bit for
bit, elastic ones (another kernel instance) within 1e-5."""
import numpy as np
import pytest

from tests import test_gpu_acoustic as ac
from tests import test_gpu_parity as el
from fwi2d_amd import workloads as W

pytestmark = pytest.mark.gpu
rel = el.rel


@pytest.fixture(scope="module")
def lib():
    import fwi2d_amd
    fwi2d_amd.load()
    return fwi2d_amd


def pick_traces(rxz, pick):
    r0 = np.cumsum([0] + [len(r) for r in rxz])
    return np.concatenate([np.arange(r0[s], r0[s + 1]) for s in pick])


def test_acoustic_streamed_levels(lib, orc64, orc32):
    nx, nz, ns, nt, h = 130, 83, 2100, 160, 0.01
    assert 3 * 4 * ns * nx * 84 > 256 << 20
    grid, model, _, _, _ = ac.case(nx=nx, nz=nz, nt=nt, ns=1)
    grid.update(gdamp_tmin=0.0, gdamp_tmax=0.2, gdamp_power=0.5)  # unequal weights of the snapshots
    rng = np.random.default_rng(0)
    sxz = np.stack([rng.uniform(0.1, (nx - 10) * h, ns), rng.uniform(0.05, (nz - 10) * h, ns)], 1)
    rxz = [np.stack([np.linspace(0.05, (nx - 4) * h, 5 + s % 3), np.full(5 + s % 3, 0.05 + 0.01 * (s % 4))], 1)
           for s in range(ns)]
    src = np.stack([W.ricker(nt, grid["dt"], 20.0 + s % 10) for s in range(ns)])
    pick = [1, 1007, 2098]
    tr = pick_traces(rxz, pick)
    few = (sxz[pick], [rxz[s] for s in pick])
    adj = np.zeros((sum(len(r) for r in rxz), nt), np.float32)
    adj[tr] = rng.standard_normal((len(tr), nt)) * np.hanning(nt)
    ref, gref = ac.oracle_run(orc64, grid, model, *few, src[pick], adj=adj[tr])
    gap = rel(ac.oracle_run(orc32, grid, model, *few, src[pick])[0], ref)
    e = ac.engine(lib, grid, model, sxz, rxz)
    out = e.forward(src, keep_snapshots=True)[tr]
    g = e.adjoint(adj)
    e.close()
    e = ac.engine(lib, grid, model, *few)
    alone = e.forward(src[pick], keep_snapshots=True)
    ga = e.adjoint(adj[tr])
    e.close()
    err, errs = rel(out, ref), [rel(g[c], gref[c]) for c in range(2)]
    print("traces %.3e (FP32 gap %.3e), gradients %.3e %.3e, alone %.3e" % (err, gap, *errs, rel(ga, g.astype(float))))
    assert err <= max(1e-5, 2 * gap)
    assert max(errs) <= 1e-4
    assert np.array_equal(out, alone)
    assert rel(ga, g.astype(np.float64)) <= 1e-6  # the same terms, the shots summed in other groups


# 9 x 3 tiles: 4131 and 6183 tiles x shots, groups of 2 and 3 shots, the last of 1
@pytest.mark.parametrize("vti", [False, True])
@pytest.mark.parametrize("ns, group", [(153, 2), (229, 3)])
def test_elastic_points_in_their_own_launch(lib, orc64, orc32, vti, ns, group):
    prob, model, sxz, rxz, src, nt, dt = el.engine_case(nx=130, nz=150, nt=240, ns=ns, vti=vti)
    rxz = [r[:12 + s % 5] for s, r in enumerate(rxz)]
    src = np.stack([np.stack([W.ricker(nt, dt, 20.0 + s % 7) * a for s in range(ns)]) for a in (0.3, 1.0)])
    pick = [0, 77, ns - 1]
    tr = pick_traces(rxz, pick)
    few = (prob, model, sxz[pick], [rxz[s] for s in pick], src[:, pick], nt, dt)
    adj = np.zeros((2, sum(len(r) for r in rxz), nt), np.float32)
    adj[:, tr] = np.random.default_rng(3).standard_normal((2, len(tr), nt)) * np.hanning(nt)
    ref = el.oracle_forward(orc64, *few)
    gap = rel(el.oracle_forward(orc32, *few), ref)
    gref = el.oracle_gradient(orc64, *few, adj[:, tr], vti)
    one, alone = el.run_engine(lib, *few)
    assert one.stat("shots_per_block") == 1
    for fused in (0, 1):
        e, out = el.run_engine(lib, prob, model, sxz, rxz, src, nt, dt, sub=1, keep=True,
                               options=(("image_fused", fused),))
        assert e.stat("ntiles") * ns  == 27 * ns and e.stat("shots_per_block") == group
        assert e.stat("image_fused") == fused
        g = e.adjoint(adj)
        e.close()
        err, errs = rel(out[:, tr], ref), [rel(g[c], gref[c]) for c in range(3)]
        print("vti=%s image_fused=%d: traces %.3e (FP32 gap %.3e), gradients %s, alone %.3e"
              % (vti, fused, err, gap, ["%.3e" % v for v in errs], rel(alone, out[:, tr].astype(float))))
        assert err <= max(1e-5, 2 * gap)
        assert max(errs) <= 1e-4
        assert rel(alone, out[:, tr].astype(np.float64)) < 1e-5
    one.close()
