"""Sweeps in which some passes update both parities in one launch and others do
not, against the same handle with single passes throughout (an HBM budget that
leaves no room for second buffers), bit for bit: the links of lattices whose
other fields are past the size for it, beside multicanonical and Metropolis
passes, with a lattice whose sweeps are spent, and where the buffers are taken
away between sweeps.  That the two handles take different launches is checked on
the CPU by test_host_side.py (which_sweeps_pair), at these sizes."""
import ctypes as C

import numpy as np
import pytest

from su2higgs_amd import abi
from su2higgs_amd.lattice import Batch

pytestmark = pytest.mark.gpu

FORMS = {"fp64": (abi.FP64, abi.LINKS_AUTO), "full": (abi.FP32, abi.LINKS_FULL),
         "packed": (abi.FP32, abi.LINKS_PACKED)}
MODELS = {
    "hu": dict(nhiggs=1, u1=1),
    "hsu": dict(nhiggs=1, u1=1, singlet=1),
    "ht": dict(nhiggs=1, triplet=1),
    "t": dict(nhiggs=0, triplet=1),
}


def params(form, L, seed, **kw):
    precision, links = FORMS[form]
    return abi.make_params(L=L, precision=precision, link_format=links, betasu2=6.0, betau1=12.0,
                           lambda_phi=0.02, seed=seed, **kw)


def no_room(ps):
    total = 0
    for p in ps:
        n = C.c_uint64()
        abi.check(abi.load().su2hip_footprint(C.byref(p), 0, C.byref(n)))
        total += n.value
    return total


def pair_of(ps, graph=True):
    """The handle with paired passes and the one without."""
    out = [Batch(ps), Batch(ps, hbm_budget=no_room(ps))]
    for b in out:
        for i in range(len(ps)):
            b.cold_start(i, 1.0, 0.5, 0.2)
        b.use_graph(graph)
    return out


def assert_same(a, b):
    assert a.budgets() == b.budgets()
    for i in a.params:
        fa, fb = a.get_fields(i), b.get_fields(i)
        for k in fa:
            if fa[k] is not None:
                assert np.array_equal(fa[k], fb[k]), (i, k)
        assert a.counters(i) == b.counters(i), i
        assert a.rng_get(i) == b.rng_get(i), i
    assert np.array_equal(a.measure_all(), b.measure_all())


@pytest.mark.parametrize("rounds", [1, 2])
@pytest.mark.parametrize("model", sorted(MODELS))
@pytest.mark.parametrize("form", sorted(FORMS))
def test_links_alone_are_paired(form, model, rounds):
    """36000 to 65536 (FP64) or 120000 sites: the passes of the other fields
    read links from their second buffers after an even number of rounds."""
    ext = [(40, 34, 30)] if rounds == 1 else [(24, 30, 26), (34, 26, 22)]
    a, b = pair_of([params(form, e, 11 + i, link_overrelax=rounds, scalar_sweeps=2, **MODELS[model])
                    for i, e in enumerate(ext)])
    for _ in range(2):
        for x in (a, b):
            x.update(2)
        assert_same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_beside_link_metropolis(form, graph):
    a, b = pair_of([params(form, (12, 10, 8), 5, nhiggs=1, u1=1, link_overrelax=1, update_links=2,
                           algorithm_su2link=abi.METROPOLIS)], graph)
    for x in (a, b):
        x.update(3)
    assert_same(a, b)
    a.close()
    b.close()


def weight(orderparam):
    bins = 20
    pos = np.concatenate([[-100.0], np.linspace(0.0, 4.0, bins + 1)])
    W = 0.5 * np.sin(np.arange(bins + 2))
    m = abi.Muca()
    m.enabled, m.orderparam, m.mode, m.checks_per_sweep, m.bins = 1, orderparam, abi.FAST, 3, bins
    m.min, m.max, m.wrk_min, m.wrk_max, m.do_acceptance, m.delta = 0.0, 4.0, 0.0, 4.0, 1, 0.3
    m.update_interval = 5
    return m, pos, W


@pytest.mark.parametrize("model,orderparam", [("hu", abi.PHISQ), ("ht", abi.SIGMASQ),
                                              ("ht", abi.PHI2MINUSSIGMA2), ("hsu", abi.PHISQ)])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_beside_multicanonical_passes(form, model, orderparam):
    ps = [params(form, e, 21 + i, link_overrelax=1, scalar_sweeps=2, **MODELS[model])
          for i, e in enumerate([(12, 10, 14), (8, 8, 8)])]
    a, b = pair_of(ps)
    for x in (a, b):
        x.update(1)
        x.muca_set(0, *weight(orderparam))
    for _ in range(2):
        for x in (a, b):
            x.update(3)
        assert_same(a, b)
        assert np.array_equal(a.muca_orderparam(0, False), b.muca_orderparam(0, False))
        for u, v in zip(a.muca_get(0)[1:], b.muca_get(0)[1:]):
            assert np.array_equal(u, v)
    a.close()
    b.close()


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_with_a_lattice_whose_sweeps_are_spent(form, graph):
    ps = [params(form, e, 31 + i, nhiggs=1, u1=1, singlet=1, link_overrelax=1)
          for i, e in enumerate([(12, 10, 14), (8, 8, 8), (4, 26, 12)])]
    a, b = pair_of(ps, graph)
    for x in (a, b):
        x.set_budget(1, 2)
        x.set_budget(0, 0)
        x.update(3)
    assert_same(a, b)
    assert a.budgets() == [0, 0, -1]
    for x in (a, b):
        x.set_budget(0, -1)
        x.update(2)
    assert_same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("form", sorted(FORMS))
def test_buffers_taken_and_given_back(form):
    """Paired sweeps, then a flow's buffers in place of the second ones, single
    passes, and paired ones again once the lattice that flowed has left."""
    ps = [params(form, (12, 10, 14), 41 + i, nhiggs=1, link_overrelax=1) for i in range(3)]
    room = no_room(ps) * 29 // 20
    a, b = Batch(ps, hbm_budget=room), Batch(ps, hbm_budget=room)
    c = Batch(ps)
    hs = (a, b, c)
    for x in hs:
        for i in range(3):
            x.cold_start(i, 1.0)
        x.use_graph(x is not b)
        x.update(2)
    rows = [x.flow(0, abi.FLOW_RK3, 0.05, 0.2, 2) for x in hs]
    for x in hs:
        x.muca_set(1, *weight(abi.PHISQ))
        x.update(2)
    for x, r in zip(hs, rows):
        assert np.array_equal(r, rows[0])
        assert_same(x, a)
    for x in hs:
        x.remove(0)
        x.update(2)
    assert_same(b, a)
    assert_same(c, a)
    for x in hs:
        x.close()


@pytest.mark.parametrize("precision", [abi.FP64, abi.FP32])
@pytest.mark.parametrize("graph", [False, True])
def test_single_passes_of_any_chunk_and_occupancy(precision, graph):
    """Handles without paired passes, whose passes launch with the chunk and
    the occupancy target set, make one and the same chain."""
    form = "fp64" if precision == abi.FP64 else "full"
    ps = [params(form, e, 51 + i, nhiggs=1, u1=1, link_overrelax=2)
          for i, e in enumerate([(8, 8, 8), (12, 10, 8), (16, 16, 16), (6, 8, 10)])]
    a = pair_of(ps, graph)[0]
    a.update(3)
    for chunk, waves in [(64, 5), (128, 0), (256, 5), (0, 0)]:
        b = Batch(ps, hbm_budget=no_room(ps))
        for i in range(len(ps)):
            b.cold_start(i, 1.0, 0.5, 0.2)
        b.use_graph(graph)
        for k in range(abi.K_MEASURE):
            b.set_chunk(k, chunk)
        b.set_waves(abi.K_LINK_OVERRELAX, waves)
        b.update(3)
        assert_same(a, b)
        b.close()
    a.close()


def test_tuned_single_passes_continue_the_chain():
    ps = [params("packed", e, 61 + i, nhiggs=1, u1=1, link_overrelax=2)
          for i, e in enumerate([(8, 8, 8), (16, 16, 16)])]
    a, b = pair_of(ps)
    b.update(2)
    b.autotune(repeats=20)
    b.update(2)
    a.update(4)
    assert_same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("links", [abi.LINKS_FULL, abi.LINKS_PACKED])
def test_fp32_fields_come_back_from_every_piece(links):
    """Scalars and angles as given and rounded to FP32; links, which are stored
    in a form of their own, within 8 units of 2^-23."""
    ext = [(6, 10, 4), (32, 32, 18), (64, 64, 34)]
    ps = [abi.make_params(L=e, precision=abi.FP32, link_format=links, nhiggs=1, u1=1, singlet=1) for e in ext]
    rng = np.random.default_rng(9)
    b = Batch(ps)
    for i, p in enumerate(ps):
        f = {k: None if v is None else rng.standard_normal(v.shape) for k, v in abi.field_arrays(p).items()}
        f["su2link"] /= np.linalg.norm(f["su2link"], axis=-1, keepdims=True)
        f["u1link"] = np.clip(f["u1link"], -3.0, 3.0)
        b.set_fields(i, f)
        got = b.get_fields(i)
        assert np.abs(got["su2link"] - f["su2link"]).max() < 8 * 2.0**-23
        for k in ("u1link", "doublet", "singlet"):
            assert np.array_equal(got[k], f[k].astype(np.float32).astype(np.float64)), (k, ext[i])
    b.close()
