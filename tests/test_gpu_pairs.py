"""Sweeps that update both parities of a field in one launch, against
the same passes launched one by one: the same bits and counts, since a link's
staple, draws and arithmetic do not depend on the launch that updates it.
Sizes: single tiles that span the lattice, ragged tiles, rows of the widest
kind, lattices of different shapes in one handle."""
import numpy as np
import pytest

from su2higgs_amd import abi
from su2higgs_amd.lattice import Batch

pytestmark = pytest.mark.gpu

SHAPES = {
    "span": [(4, 4, 2), (2, 4, 6), (8, 8, 8)],
    "ragged": [(34, 10, 14)],
    "wide": [(128, 6, 4), (4, 26, 12)],
    "mixed": [(24, 24, 24), (16, 30, 10), (12, 6, 50)],
}
MODELS = {
    "pure": dict(nhiggs=0),
    "hu": dict(nhiggs=1, u1=1),
    "triplet": dict(nhiggs=0, triplet=1),
}


@pytest.mark.parametrize("form", ["fp64", "full", "packed"])
@pytest.mark.parametrize("model", sorted(MODELS))
@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("rounds", [1, 2])
def test_paired_sweep_is_its_passes(shape, model, form, rounds):
    exts = SHAPES[shape]
    ps = [
        abi.make_params(
            L=e, precision=abi.FP64 if form == "fp64" else abi.FP32,
            link_format={"fp64": 0, "full": abi.LINKS_FULL, "packed": abi.LINKS_PACKED}[form],
            betasu2=6.0, betau1=12.0, seed=31 + i, link_overrelax=rounds, update_su2doublet=0,
            update_su2triplet=0, **MODELS[model])
        for i, e in enumerate(exts)
    ]
    a, b = Batch(ps), Batch(ps)
    for x in (a, b):
        for i in range(len(ps)):
            x.hot_start(i)
        x.use_graph(x is a)
    if form == "packed" and model == "hu":
        b.set_hop_cache(False)
    kinds = [abi.K_LINK_HEATBATH] + rounds * [abi.K_LINK_OVERRELAX]
    if "u1" in MODELS[model]:
        kinds.append(abi.K_U1_METROPOLIS)
    for _ in range(3):
        a.update(1)
        for k in kinds:
            for d in range(3):
                for par in range(2):
                    b.pass_(k, par, d)
        for i in range(len(ps)):
            fa, fb = a.get_fields(i), b.get_fields(i)
            for name in fa:
                if fa[name] is not None:
                    assert np.array_equal(fa[name], fb[name]), (name, exts[i])
            assert a.counters(i) == b.counters(i)
            assert a.rng_get(i) == b.rng_get(i)
    a.close()
    b.close()


FIELDS = {
    "hsu": dict(nhiggs=1, u1=1, singlet=1),
    "ht": dict(nhiggs=1, triplet=1),
}


@pytest.mark.parametrize("form", ["fp64", "full", "packed"])
@pytest.mark.parametrize("model", sorted(FIELDS))
@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("rounds", [1, 2])
def test_paired_scalar_rounds_are_their_passes(shape, model, form, rounds):
    exts = SHAPES[shape]
    ps = [
        abi.make_params(
            L=e, precision=abi.FP64 if form == "fp64" else abi.FP32,
            link_format={"fp64": 0, "full": abi.LINKS_FULL, "packed": abi.LINKS_PACKED}[form],
            betasu2=6.0, betau1=12.0, lambda_phi=0.02, seed=57 + i, link_overrelax=0,
            scalar_sweeps=rounds, **FIELDS[model])
        for i, e in enumerate(exts)
    ]
    a, b = Batch(ps), Batch(ps)
    for x in (a, b):
        for i in range(len(ps)):
            x.cold_start(i, 1.0, 0.5, 0.2)
        x.use_graph(x is a)
    kinds = [(abi.K_LINK_HEATBATH, 3)]
    if model == "hsu":
        kinds.append((abi.K_U1_METROPOLIS, 3))
    for s in range(rounds + 1):
        last = s == rounds
        kinds.append((abi.K_DOUBLET_METROPOLIS if last else abi.K_DOUBLET_OVERRELAX, 1))
        if model == "ht":
            kinds.append((abi.K_TRIPLET_METROPOLIS if last else abi.K_TRIPLET_OVERRELAX, 1))
        else:
            kinds.append((abi.K_SINGLET_METROPOLIS if last else abi.K_SINGLET_OVERRELAX, 1))
    for _ in range(3):
        a.update(1)
        for k, ndir in kinds:
            for d in range(ndir):
                for par in range(2):
                    b.pass_(k, par, d)
        for i in range(len(ps)):
            fa, fb = a.get_fields(i), b.get_fields(i)
            for name in fa:
                if fa[name] is not None:
                    assert np.array_equal(fa[name], fb[name]), (name, exts[i])
            assert a.counters(i) == b.counters(i)
            assert a.rng_get(i) == b.rng_get(i)
    a.close()
    b.close()
