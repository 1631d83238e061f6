"""Per-q pipeline (products -> chi0 -> eps^-1) vs the oracle chain, eager and
graph-replayed."""
import numpy as np
import pytest

import oracle
from project1_amd import spexhip, synth
from project1_amd.pipeline import Crystal, QJob
from tests.conftest import normwise

pytestmark = pytest.mark.gpu


def oracle_chain(job):
    """Oracle products -> chi0 (x2 spin) -> eps (dense v^1/2) -> eps^-1."""
    s = job.crystal.sys
    d = job.desc
    mt = oracle.wfprod_mt(s.types, s.cent, s.q, s.k1, s.k2, s.cmt, 0, d.nocc, d.nocc, d.nunocc)
    pw = oracle.wfprod_pw(s.k1, s.k2, s.g2, s.gpt, s.ngpt, s.cpw, s.gptm, s.vol, 0, d.nocc,
                          d.nocc, d.nunocc)
    M = np.concatenate([mt, pw], axis=1)
    w = oracle.weights_none(job.e_occ, job.e_unocc, job.omega)
    chi = 2 * oracle.chi0_herk(M, w).T  # (nw, npack)
    einv = np.stack([oracle.inverse_hpd_packed(oracle.dielectric_dense(chi[f], job.vh.astype(complex)))
                     for f in range(d.nw)])
    return chi, einv


@pytest.fixture(scope="module")
def crystal(ctx):
    c = Crystal(ctx, nmesh=2, nband=14, ngptm=60, seed=3, nfft=(16, 16, 16), gcut=3.1)
    yield c
    c.free()


@pytest.mark.parametrize("precision,tol", [(spexhip.PREC_FP64, 1e-12), (spexhip.PREC_OZAKI_INT8, 1e-8)])
def test_pipeline_vs_oracle_chain(ctx, crystal, precision, tol):
    job = QJob(ctx, crystal, nocc=4, nunocc=8, nw=3, precision=precision, seed=11)
    job.launch()
    ms = job.wait()
    chi, einv = job.pipe.result()
    rchi, reinv = oracle_chain(job)
    e1, e2 = normwise(chi, rchi), normwise(einv, reinv)
    print(f"pipeline prec={precision}: {ms:.2f} ms chi0 {e1} eps^-1 {e2}")
    assert max(e1) < tol and max(e2) < 100 * tol
    job.free()


def test_graph_replays_match_eager(ctx, crystal):
    job = QJob(ctx, crystal, nocc=3, nunocc=7, nw=2, precision=spexhip.PREC_OZAKI_INT8, seed=12,
               graph=False)
    job.launch()
    job.wait()
    ref = job.pipe.result()
    job.graph = True
    other = QJob(ctx, crystal, nocc=2, nunocc=5, nw=2, precision=spexhip.PREC_FP64, seed=13)
    for rep in range(3):
        job.launch()  # first: capture + replay; then replays
        job.wait()
        got = job.pipe.result()
        np.testing.assert_array_equal(got[0], ref[0])
        np.testing.assert_array_equal(got[1], ref[1])
        other.launch()  # eager work of another pipeline between the replays
        other.wait()
    job.free()
    other.free()


def test_pipeline_reports_not_pd(ctx, crystal):
    """A huge v^1/2 against a negative-definite chi0 cannot make eps indefinite,
    so force it through mixed-sign weights of the Ozaki form instead."""
    job = QJob(ctx, crystal, nocc=2, nunocc=4, nw=2, precision=spexhip.PREC_OZAKI_INT8, seed=14)
    # overwrite one occupied energy above the unoccupied ones -> a positive weight
    eo = job.e_occ.copy()
    eo[0, 0] = 10.0
    job.bufs[0].upload(eo)
    job.launch()
    with pytest.raises(spexhip.SpexError) as e:
        job.wait()
    assert e.value.code == spexhip.E_INVALID
    job.free()


@pytest.mark.parametrize("precision,tol", [(spexhip.PREC_FP64, 1e-13), (spexhip.PREC_OZAKI_INT8, 1e-8)])
def test_k_packets_match_one_packet(ctx, crystal, precision, tol):
    """kpacket = 3 of 8 k-points (packets 3, 3, 2; buffers sized for 3) gives
    the one-packet result up to the summation order of the packets."""
    one = QJob(ctx, crystal, nocc=3, nunocc=6, nw=2, precision=precision, seed=21)
    one.launch()
    one.wait()
    ref = one.pipe.result()
    d = one.desc
    d.kpacket = 3
    pk = spexhip.QPipe(ctx, d, [])
    assert spexhip.qpipe_footprint(d) < one.footprint
    pk.launch()
    pk.wait()
    got = pk.result()
    e1, e2 = normwise(got[0], ref[0]), normwise(got[1], ref[1])
    print(f"packets prec={precision}: chi0 {e1} eps^-1 {e2}")
    assert max(e1) < tol and max(e2) < 100 * tol
    pk.destroy()
    one.free()



def _given_products(c, precision, nk=8, nocc=8, nunocc=32, nb=130, nw=3):
    """A descriptor over given products whose pair sum splits its few tiles (19 MiB of parts in
    FP64, 5 MiB in the int8 form), and what it points to."""
    g = synth.rng(31)
    n = nk * nocc * nunocc
    M = (g.standard_normal((n, nb)) + 1j * g.standard_normal((n, nb))) / np.sqrt(n)
    eo, eu = synth.energies(g, nk, nocc, nunocc)
    om, _ = synth.gl_frequencies(nw)
    bufs = [c.to_dev(a) for a in (M, eo, eu, np.ones(nk, np.int32), om, np.full(nb, 1.3))]
    d = spexhip.QDesc()
    d.nk, d.nocc, d.nunocc, d.nb, d.nw, d.precision, d.alpha = nk, nocc, nunocc, nb, nw, precision, 2.0
    d.M_dev, d.ldm, d.nkpt_w, d.nsym1 = bufs[0].ptr, nb, nk, 1
    d.e_occ_dev, d.e_unocc_dev, d.nkpts_dev, d.omega_dev, d.vhalf_dev = (b.ptr for b in bufs[1:])
    return d, bufs


@pytest.mark.parametrize("precision", [spexhip.PREC_FP64, spexhip.PREC_SPLIT_FP32,
                                       spexhip.PREC_OZAKI_INT8])
def test_budget_without_room_for_parts(precision):
    """A context and a server whose budgets hold a pipeline but not the parts of its split tiles
    run it without them: the same bits in FP64 and split-FP32, 1e-8 in the int8 form (another
    order of its FP64 sums)."""
    ozaki = precision == spexhip.PREC_OZAKI_INT8
    with spexhip.Context(0) as c:
        d, bufs = _given_products(c, precision)
        used = c.mem_used()[0]
        p = spexhip.QPipe(c, d, bufs)
        p.launch()
        p.wait()
        want = p.result()
        p.destroy()
        # its other buffers take less than 6 MiB, the int8 form's beside the parts
        room = spexhip.qpipe_footprint(d) - (2 << 20) if ozaki else 6 << 20
        s = spexhip.Server(c, 2, room)
        rid = s.submit(d)
        s.wait(rid)
        got = [s.result(rid)]
        assert s.stats()["peak_hbm_bytes"] <= room
        s.release(rid)
        s.destroy()
    with spexhip.Context(0, hbm_budget=used + room) as c:
        d, bufs = _given_products(c, precision)
        p = spexhip.QPipe(c, d, bufs)
        assert c.mem_used()[0] <= used + room
        for graph in (False, True, True):
            p.launch(graph)
            p.wait()
            got.append(p.result())
        p.destroy()
    for r in got:
        for a, b in zip(r, want):
            if ozaki:
                assert max(normwise(a, b)) < 1e-8
            else:
                np.testing.assert_array_equal(a, b)
