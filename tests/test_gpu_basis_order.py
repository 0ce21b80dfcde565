"""The device basis, whose representative choice rests on the device's
level-by-level computation of the reference's std::unordered_map iteration
order (basis.hip map_positions), against the CPU mirror (tests/hostcheck),
which replays the map's node list on the host: id[] and basis_C[] equal
element by element on medium sectors, and by SHA-256 on the benchmark
sector (2,348,125 states from 37.6M words) and the fixed-layer N_phi = 16
sector, whose mirror bases take a minute on the CPU
(tests/golden/make_basis_sha.py)."""
import hashlib
import json
import os

import numpy as np
import pytest

import blqh_amd
from tests import hostmirror

pytestmark = pytest.mark.gpu

MEDIUM = [(2, 12, 12, -1, -1, 1, 2), (2, 12, 12, 6, -1, 0, 0), (2, 14, 14, 7, -1, 7, 7), (4, 8, 8, 4, 4, 3, 5),
          (4, 8, 8, 4, -1, 0, 0), (1, 18, 6, -1, -1, 3, 5), (1, 16, 8, -1, -1, 2, 7)]


@pytest.mark.skipif(not os.path.exists(hostmirror.PATH), reason="host mirror not built")
@pytest.mark.parametrize("case", MEDIUM, ids=lambda c: "_".join(map(str, c)))
def test_device_basis_equals_mirror(case):
    S, nphi, nel, nu, nsu, J, K = case
    print(f"basis {case}", flush=True)
    B = blqh_amd.Basis(nphi, nel, nu, J, K, nspecies=S, nel_su=nsu)
    ids, per = hostmirror.basis(blqh_amd.Sector(*case))
    assert B.n == len(ids)
    np.testing.assert_array_equal(B.id, ids)
    np.testing.assert_array_equal(B.period, per)


with open(os.path.join(os.path.dirname(__file__), "golden", "basis_sha256.json")) as _f:
    LARGE = json.load(_f)


@pytest.mark.parametrize("key", sorted(LARGE))
def test_large_basis_checksum(key):
    S, nphi, nel, nu, nsu, J, K = map(int, key.split("_"))
    print(f"basis {key}", flush=True)
    B = blqh_amd.Basis(nphi, nel, nu, J, K, nspecies=S, nel_su=nsu)
    assert B.n == LARGE[key]["n"]
    h = hashlib.sha256()
    h.update(np.ascontiguousarray(B.id).astype("<u8").tobytes())
    h.update(np.ascontiguousarray(B.period).astype("<i2").tobytes())
    assert h.hexdigest() == LARGE[key]["sha256"]


@pytest.mark.parametrize("case", [(2, 2, 1, -1, -1, 0, 0), (2, 2, 1, -1, -1, -1, -1), (2, 16, 3, -1, -1, 1, 2),
                                  (4, 8, 2, 1, -1, 1, 1), (2, 17, 3, -1, -1, 1, 2), (2, 8, 8, -1, -1, -1, 3)],
                         ids=lambda c: "_".join(map(str, c)))
def test_lookup_tables_by_word_size(oracle_mod, case):
    """The lookup table and the halves' rank shares come from one launch: fewer table places than
    shares and more, words of 4 to 32 bits, and of 34, which have no shares.  Rows against the
    oracle's."""
    O = oracle_mod
    S, nphi, nel, nu, nsu, J, K = case
    B = blqh_amd.Basis(nphi, nel, nu, J, K, nspecies=S, nel_su=nsu)
    H = blqh_amd.Hamiltonian(B, blqh_amd.params(nphi, d=0.7, delta_sas=0.1))
    print(f"{case} n {H.n}", flush=True)
    OB = O.Basis(O.sector(*case))
    OH = O.Hamiltonian(OB, O.params(nphi, d=0.7, dsas=0.1))
    np.testing.assert_array_equal(B.id, OB.id)
    rp, col, val = H.export()
    np.testing.assert_array_equal(rp, OH.rowptr)
    np.testing.assert_array_equal(col.astype(np.int64), OH.col)
    np.testing.assert_allclose(val, OH.val, rtol=0, atol=1e-13 * np.abs(OH.val).max())
