"""Batched uneven q-points (one grouped chi0 launch per k packet) against the
per-q pipeline and the oracle chain; graph replays against the eager run."""
import numpy as np
import pytest

from project1_amd import serving, spexhip
from tests.chain import einv_tol, eps_cond, oracle_for_request
from tests.conftest import normwise

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lattice(ctx):
    lat = serving.Lattice(ctx, nocc=3, nunocc=14, lcut=2, nrad=2, gcut=3.1, nfft=(16, 16, 16),
                          max_atoms=3, nb_max=110, ipw_target=40, seed=8)
    yield lat
    lat.free()


def uneven(lat, precision, nq=5, seed=4):
    """nq q-points of one 2^3 mesh with different q, nb, nunocc and nw."""
    g = np.random.default_rng(seed)
    specs = [serving.Spec(nmesh=2, nb=int(g.integers(50, 111)), nw=int(g.integers(1, 4)),
                          seed=500 + i, nunocc=int(g.integers(4, 15)), iq=1 + i)
             for i in range(nq)]
    return [serving.Request(lat, s, precision) for s in specs]


def per_q(lat, reqs):
    out = []
    for r in reqs:
        p = spexhip.QPipe(lat.ctx, r.desc, [])
        p.launch()
        p.wait()
        out.append(p.result())
        p.destroy()
    return out


@pytest.mark.parametrize("precision,tol", [(spexhip.PREC_FP64, 1e-12),
                                           (spexhip.PREC_SPLIT_FP32, 1e-8)])
def test_batch_matches_per_q_pipelines(lattice, precision, tol):
    reqs = uneven(lattice, precision)
    ref = per_q(lattice, [serving.Request(lattice, r.spec, spexhip.PREC_FP64) for r in reqs])
    conds = [eps_cond(ref[i][0], lattice.vhalf[: r.spec.nb, : r.spec.nb].astype(complex))
             for i, r in enumerate(reqs)]
    b = spexhip.Batch(lattice.ctx, [r.desc for r in reqs], kpacket=3)  # 8 k -> 3, 3, 2
    cfg, npacket, tune = b.config()
    assert npacket == 3 and 0 <= cfg < len(spexhip.chi0_configs()) and min(tune) > 0
    b.launch()
    ms = b.wait()
    for i, r in enumerate(reqs):
        chi, einv = b.result(i)
        e1, e2 = normwise(chi, ref[i][0]), normwise(einv, ref[i][1])
        print(f"prec={precision} q{i} nb={r.spec.nb} nunocc={r.desc.nunocc}: chi0 {e1} "
              f"eps^-1 {e2} cond(eps) {conds[i]:.2e} ({ms:.2f} ms)")
        # chi0 within tol; eps^-1 within what eps's condition number makes of
        # the chi0 difference and of FP64 rounding
        assert max(e1) < tol and max(e2) < einv_tol(conds[i], r.spec.nb, max(e1))
    b.destroy()
    for r in reqs:
        r.free()


def test_batch_vs_oracle_and_graph_replays(lattice):
    reqs = uneven(lattice, spexhip.PREC_FP64, nq=4, seed=9)
    b = spexhip.Batch(lattice.ctx, [r.desc for r in reqs], kpacket=5, config=3)
    b.launch()
    b.wait()
    eager = [b.result(i) for i in range(len(reqs))]
    rchi, reinv, cond = oracle_for_request(lattice, reqs[2])
    e1, e2 = normwise(eager[2][0], rchi), normwise(eager[2][1], reinv)
    print(f"batch q2 vs oracle: chi0 {e1} eps^-1 {e2} cond(eps) {cond:.2e}")
    assert max(e1) < 1e-12 and max(e2) < einv_tol(cond, reqs[2].spec.nb)
    other = spexhip.QPipe(lattice.ctx, reqs[0].desc, [])
    for rep in range(3):
        b.launch(graph=True)  # first: capture + replay, then replays
        b.wait()
        for i in range(len(reqs)):
            got = b.result(i)
            np.testing.assert_array_equal(got[0], eager[i][0])
            np.testing.assert_array_equal(got[1], eager[i][1])
        other.launch()  # eager work of another pipeline between the replays
        other.wait()
    other.destroy()
    b.destroy()
    for r in reqs:
        r.free()


def test_batch_ozaki_matches_per_q_and_footprint(lattice):
    """Ozaki form: per-q int8 rank-k launches on the q streams, one slice
    workspace per stream; against the FP64 per-q pipelines at 1e-8."""
    reqs = uneven(lattice, spexhip.PREC_OZAKI_INT8, nq=5, seed=11)
    ref = per_q(lattice, [serving.Request(lattice, r.spec, spexhip.PREC_FP64) for r in reqs])
    descs = [r.desc for r in reqs]
    assert spexhip.Batch.footprint(descs, 2) < spexhip.Batch.footprint(descs, 8)
    b = spexhip.Batch(lattice.ctx, descs, kpacket=3)
    cfg, npacket, _ = b.config()
    assert cfg == -1 and npacket == 3
    b.launch(graph=True)
    b.wait()
    for i, r in enumerate(reqs):
        chi, einv = b.result(i)
        e1 = normwise(chi, ref[i][0])
        print(f"ozaki batch q{i}: chi0 {e1}")
        assert max(e1) < 1e-8
    b.destroy()
    for r in reqs:
        r.free()


def test_batch_ozaki_budget_without_room_for_parts():
    """int8 form on two q-points whose few tiles are split: a budget that holds the batch but not
    the parts gives the same pair sums within 1e-8 (another order of the FP64 sums)."""
    out, budget = [], 0
    for _ in range(2):
        with spexhip.Context(0, hbm_budget=budget) as c:
            lat = serving.Lattice(c, nocc=4, nunocc=12, lcut=2, nrad=2, gcut=3.1,
                                  nfft=(16, 16, 16), max_atoms=3, nb_max=100, ipw_target=40, seed=8)
            reqs = [serving.Request(lat, serving.Spec(nmesh=3, nb=100, nw=3, seed=70 + i, iq=1 + i),
                                    spexhip.PREC_OZAKI_INT8) for i in range(2)]
            b = spexhip.Batch(c, [r.desc for r in reqs], kpacket=27)
            used = c.mem_used()[0]
            b.launch()
            b.wait()
            out.append([b.result(i, einv=False)[0] for i in range(2)])
            b.destroy()
        print(f"batch: {used} of {budget}")
        assert not budget or used <= budget
        budget = used - (1 << 20)
    for x, y in zip(*out):
        assert max(normwise(x, y)) < 1e-8
