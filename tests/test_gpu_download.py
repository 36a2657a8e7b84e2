"""Fields uploaded and fetched again, bit for bit, at the sizes where the way
they are fetched changes: one copy for all fields up to 2 MiB, pieces beyond,
more pieces than there are pinned slots, and back to a small one.  FP64 stores
the values as given."""
import numpy as np
import pytest

from su2higgs_amd import abi
from su2higgs_amd.lattice import Batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", [dict(nhiggs=1), dict(nhiggs=2, u1=1), dict(nhiggs=1, u1=1, singlet=1),
                                   dict(nhiggs=0, triplet=1)])
def test_fields_come_back_as_given(model):
    exts = [(2, 2, 2), (32, 32, 16), (32, 32, 18), (64, 64, 34), (6, 10, 4)]
    ps = [abi.make_params(L=e, precision=abi.FP64, **model) for e in exts]
    rng = np.random.default_rng(3)
    with_fields = []
    b = Batch(ps)
    for i, p in enumerate(ps):
        f = {k: None if v is None else rng.standard_normal(v.shape) for k, v in abi.field_arrays(p).items()}
        b.set_fields(i, f)
        with_fields.append(f)
    for _ in range(2):
        for i, f in enumerate(with_fields):
            got = b.get_fields(i)
            for k in f:
                assert (got[k] is None) == (f[k] is None)
                if f[k] is not None:
                    assert np.array_equal(got[k], f[k]), (k, exts[i])
    b.close()
