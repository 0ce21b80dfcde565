"""The coded layout (SpMV kind 6: 4-byte entries whose values come from a table)
against scipy's CSR product of the exported matrix, at its edges: fewer rows than
a slice, a ragged last slice, one column panel and several, real and complex
values, a matrix whose values the table covers badly, each team size."""
import numpy as np
import pytest
import scipy.sparse as sp

import blqh_amd

pytestmark = pytest.mark.gpu

PLANS = [(6, 64, t, 0, r) for t in (256, 512, 1024) for r in (1, 2, 4, 8, 16) if r * 64 <= t]

# (name, (nspecies, nphi, nel, nel_up, nel_su, J, K), params)
SECTORS = [
    ("one_slice_real", (2, 4, 4, 2, -1, 0, 0), dict(d=1.0)),
    ("ragged_real", (2, 8, 8, 4, -1, 4, 4), dict(d=3.0)),
    ("ragged_complex", (2, 8, 8, -1, -1, 1, 3), dict(d=1.0, delta_sas=0.05)),
    ("twisted_many_values", (2, 10, 10, -1, -1, 3, 2), dict(d=0.7, delta_sas=0.05, theta_x=0.3, theta_y=1.1)),
    ("spinful_complex", (4, 6, 6, 3, 3, 0, 1), dict(d=1.0, delta_sas=0.05, delta_v=0.02, delta_z=0.01)),
    ("panels_real", (2, 14, 14, -1, -1, 0, 0), dict(d=1.0, delta_sas=0.05)),
    ("panels_complex", (2, 14, 14, -1, -1, 0, 3), dict(d=0.5, delta_sas=0.05)),
]


@pytest.fixture(scope="module", params=SECTORS, ids=[s[0] for s in SECTORS])
def built(request):
    name, (S, nphi, nel, nu, nsu, J, K), kw = request.param
    B = blqh_amd.Basis(nphi, nel, nu, J, K, nspecies=S, nel_su=nsu)
    H = blqh_amd.Hamiltonian(B, blqh_amd.params(nphi, **kw))
    print(f"sector {name} n {H.n}", flush=True)
    rp, col, val = H.export()
    return name, B, H, sp.csr_matrix((val, col, rp), shape=(H.n, H.n))


@pytest.mark.parametrize("plan", PLANS, ids=[f"t{p[2]}_np{p[4]}" for p in PLANS])
def test_product(built, plan):
    name, B, H, A = built
    print(f"{name} n={H.n} plan {plan}", flush=True)
    H.set_spmv(*plan)
    rng = np.random.default_rng(1)
    x = rng.normal(size=H.n) + 1j * rng.normal(size=H.n)
    scale = np.abs(A).max() * np.abs(x).max() * np.diff(A.indptr).max()
    np.testing.assert_allclose(H.spmv(x), A @ x, rtol=0, atol=2e-15 * scale)
    assert H.get_spmv()[0] == 6


def test_default_matches_csr_solver(built):
    """The default plan's ground state is the CSR kernel's: the values are the same bits,
    only the order of a row's sum differs."""
    name, B, H, A = built
    if H.n < 8:
        pytest.skip("too few states for a set number of steps")
    print(f"{name} n={H.n} Lanczos", flush=True)
    H.set_spmv(-1)
    a = H.lanczos(lam=120, seed=5)
    assert H.get_spmv()[0] == 6
    H.set_spmv(0, 16)
    b = H.lanczos(lam=120, seed=5)
    assert a["E0"] == pytest.approx(b["E0"], rel=1e-10, abs=1e-12)
    assert a["E_rq"] == pytest.approx(b["E_rq"], rel=1e-10, abs=1e-12)


def test_refused_plans(built):
    name, B, H, A = built
    for bad in ((6, 32, 512, 0, 2), (6, 64, 128, 0, 1), (6, 64, 256, 0, 8), (6, 64, 512, 0, 3), (6, 64, 512, 0, 0)):
        with pytest.raises(blqh_amd.BlqhError):
            H.set_spmv(*bad)


# Batches of one-panel members take x through LDS by column tiles; a member of more than
# 65536 rows moves the whole batch to the gathering kernel.
BATCHES = {
    "tiny": [(2, 4, 4, 2, -1, 0, 0), (2, 6, 6, 3, -1, 1, 2), (2, 8, 8, 4, -1, 4, 4)],
    "mixed_kinds": [(2, 8, 8, -1, -1, 1, 3), (2, 10, 10, 5, -1, 0, 0), (4, 6, 6, 3, 3, 0, 1)],
    "one_and_many_tiles": [(2, 12, 12, -1, -1, 0, 0), (2, 6, 6, 3, -1, 0, 0), (2, 13, 13, -1, -1, 1, 0)],
    "several_panels": [(2, 14, 14, -1, -1, 0, 0), (2, 8, 8, 4, -1, 4, 4)],
}


@pytest.mark.parametrize("name", BATCHES)
def test_batch_against_panel_kernel(name):
    """lanes = 64 (coded layout) against lanes = 16 (CSR-valued panels): a set number of
    steps, so that both run the same recurrence; energies to 1e-11 of the scale."""
    hams = []
    for S, nphi, nel, nu, nsu, J, K in BATCHES[name]:
        B = blqh_amd.Basis(nphi, nel, nu, J, K, nspecies=S, nel_su=nsu)
        hams.append(blqh_amd.Hamiltonian(B, blqh_amd.params(nphi, d=0.9, delta_sas=0.05 if nu < 0 else 0.0)))
    print(f"{name} rows {[h.n for h in hams]}", flush=True)
    seeds = list(range(3, 3 + len(hams)))
    batch = blqh_amd.Batch(hams)
    assert batch.lanes == 64
    steps = dict(lam=8, seeds=seeds, tol=0.0, res_tol=0.0, check_every=3)
    a = batch.lanczos(**steps)
    batch.lanes = 16
    b = batch.lanczos(**steps)
    for h, u, v in zip(hams, a, b):
        assert u["E0"] == pytest.approx(v["E0"], rel=1e-11, abs=1e-11)
        if h.n > 8:  # with fewer states than steps the recurrence has run out of vectors
            np.testing.assert_allclose(u["psi"], v["psi"], rtol=0, atol=1e-9)


@pytest.mark.parametrize("G", [1, 2, 3, 4])
@pytest.mark.parametrize("sector", [(12, 0, 6), (12, 1, 5), (8, 1, 3)], ids=["real_tiles", "complex_tiles", "one_tile"])
def test_shared_scales_against_combined(sector, G):
    """G scales on one base and tunnelling part against the G combined matrices, eight steps."""
    nphi, J, K = sector
    scales = [0.05, 0.1, 0.2, 0.0][:G]
    B = blqh_amd.Basis(nphi, nphi, -1, J, K)
    par = blqh_amd.params(nphi, d=0.6)
    h0, t = blqh_amd.Hamiltonian(B, par, terms=1), blqh_amd.Hamiltonian(B, par, terms=2)
    print(f"sector {sector} n {h0.n} G {G}", flush=True)
    steps = dict(lam=8, tol=0.0, res_tol=0.0)
    r = blqh_amd.Batch.scaled([h0], [t], scales).lanczos(seeds=[7] * G, check_every=3, **steps)
    for s, u in zip(scales, r):
        one = blqh_amd.Hamiltonian.combine(h0, t, s).lanczos(seed=7, **steps)
        assert u["E0"] == pytest.approx(one["E0"], rel=1e-11, abs=1e-11)
        np.testing.assert_allclose(u["psi"], one["psi"], rtol=0, atol=1e-9)


@pytest.mark.parametrize("case", [(2, 4, 4, 2, -1, 0, 0), (2, 6, 6, 3, -1, 1, 2), (2, 8, 8, 4, -1, 4, 4),
                                  (2, 8, 8, -1, -1, 1, 3), (1, 18, 6, -1, -1, 3, 1), (4, 6, 6, 3, 3, 0, 1),
                                  (2, 9, 9, -1, -1, 0, 0), (2, 9, 9, -1, -1, 2, 1), (2, 10, 10, 5, -1, 3, 2)],
                         ids=lambda c: "_".join(map(str, c)))
def test_one_workgroup_steps_equal_kernel_steps(case):
    """Up to 1,024 rows one workgroup runs the steps (Krylov vectors kept); the three kernels
    run them when the vectors are replayed.  Same order of sums: the same bits."""
    S, nphi, nel, nu, nsu, J, K = case
    B = blqh_amd.Basis(nphi, nel, nu, J, K, nspecies=S, nel_su=nsu)
    par = blqh_amd.params(nphi) if S == 1 else blqh_amd.params(nphi, d=0.8, delta_sas=0.05)
    H = blqh_amd.Hamiltonian(B, par)
    print(f"{case} n {H.n}", flush=True)
    for chk in (1, 5, 70):
        steps = dict(lam=min(100, H.n), tol=0.0, res_tol=0.0, seed=3, check_every=chk)
        a, b = H.lanczos(store_basis=1, **steps), H.lanczos(store_basis=0, **steps)
        assert a["iterations"] == b["iterations"]
        np.testing.assert_array_equal(a["alpha"], b["alpha"])
        np.testing.assert_array_equal(a["beta"], b["beta"])
        assert a["E0"] == b["E0"]


@pytest.mark.parametrize("copies", [2, 90, 130])
@pytest.mark.parametrize("K", [0, 2], ids=["real", "complex"])
def test_batch_teams_against_single_solves(copies, K):
    """One, two and four wavefronts to a slice (by the number of members: 604 rows are three
    256-row, two 512-row units or one of 1,024), beside members with fewer slices than a unit:
    eight steps against the single solver's."""
    par = blqh_amd.params(9, d=0.7, delta_sas=0.05)
    big = blqh_amd.Hamiltonian(blqh_amd.Basis(9, 9, -1, 3, K), par)
    tiny = blqh_amd.Hamiltonian(blqh_amd.Basis(8, 8, 4, 4, 4), blqh_amd.params(8, d=3.0))
    hams = [big] * (copies - 1) + [tiny]
    print(f"rows {big.n} and {tiny.n}, {copies} members", flush=True)
    steps = dict(lam=8, tol=0.0, res_tol=0.0)
    r = blqh_amd.Batch(hams).lanczos(seeds=list(range(copies)), check_every=3, **steps)
    for p in (0, copies // 2, copies - 2, copies - 1):
        one = hams[p].lanczos(seed=p, **steps)
        assert r[p]["E0"] == pytest.approx(one["E0"], rel=1e-11, abs=1e-11)
        np.testing.assert_allclose(r[p]["psi"], one["psi"], rtol=0, atol=1e-9)


@pytest.mark.parametrize("G", [1, 4])
@pytest.mark.parametrize("copies", [1, 90, 130])
def test_shared_scale_teams_against_combined(copies, G):
    """The same for shared-scale groups: sums of one, two and four wavefronts for up to four vectors."""
    par = blqh_amd.params(9, d=0.7)
    B = blqh_amd.Basis(9, 9, -1, 3, 2)
    h0, t = blqh_amd.Hamiltonian(B, par, terms=1), blqh_amd.Hamiltonian(B, par, terms=2)
    scales = [0.05, 0.1, 0.2, 0.0][:G]
    print(f"rows {h0.n}, {copies} sectors, {G} scales", flush=True)
    steps = dict(lam=8, tol=0.0, res_tol=0.0)
    r = blqh_amd.Batch.scaled([h0] * copies, [t] * copies, scales).lanczos(seeds=list(range(copies * G)), check_every=3,
                                                                           **steps)
    for p in {0, G - 1, copies * G // 2, copies * G - 1}:
        one = blqh_amd.Hamiltonian.combine(h0, t, scales[p % G]).lanczos(seed=p, **steps)
        assert r[p]["E0"] == pytest.approx(one["E0"], rel=1e-11, abs=1e-11)
        np.testing.assert_allclose(r[p]["psi"], one["psi"], rtol=0, atol=1e-9)


@pytest.mark.parametrize("store", [0, 1], ids=["replay", "kept"])
def test_coefficients_for_every_test_interval(store):
    """Coefficients reach the host in groups, one for each convergence test and one for half a
    mailbox (32 steps): the same bits whatever the interval, also past the mailbox's 64 entries."""
    B = blqh_amd.Basis(9, 9, -1, 2, 1)
    H = blqh_amd.Hamiltonian(B, blqh_amd.params(9, d=0.8, delta_sas=0.05))
    steps = dict(lam=150, tol=0.0, res_tol=0.0, seed=3, store_basis=store)
    first = H.lanczos(check_every=1, **steps)
    assert first["iterations"] == 150
    for chk in (2, 31, 32, 33, 63, 64, 65, 149, 150, 1000):
        print(f"interval {chk}", flush=True)
        r = H.lanczos(check_every=chk, **steps)
        np.testing.assert_array_equal(r["alpha"], first["alpha"])
        np.testing.assert_array_equal(r["beta"], first["beta"])
        np.testing.assert_array_equal(r["psi"], first["psi"])


@pytest.mark.parametrize("bad", [np.nan, np.inf], ids=["nan", "inf"])
def test_non_finite_entries_reach_their_rows_only(built, bad):
    """A NaN or an infinity in x shows in the rows that hold its column and in no other: the lanes
    past their row's end multiply nothing.  Tried at the first internal row of every panel, which
    those lanes read, and at others."""
    from tests import hostmirror
    name, B, H, A = built
    pos = hostmirror.internal_order(B.sector, B.id)
    at = np.argsort(pos) if pos is not None else np.arange(H.n)  # reference row of an internal one
    cols = A.tocsc()
    rng = np.random.default_rng(2)
    x = rng.normal(size=H.n) + 1j * rng.normal(size=H.n)
    rows = list(at[::65536]) + list(rng.integers(0, H.n, 2))
    for plan in ((-1, 0, 0, 0, 0), (6, 64, 512, 0, 1), (6, 64, 512, 0, 8), (6, 64, 1024, 0, 16)):
        H.set_spmv(*plan)
        good = H.spmv(x)
        for i in rows:
            print(f"{name} plan {plan} entry {i}", flush=True)
            z = x.copy()
            z[i] = bad
            y = H.spmv(z)
            hit = np.zeros(H.n, bool)
            hit[cols.indices[cols.indptr[i]:cols.indptr[i + 1]]] = True
            np.testing.assert_array_equal(np.isfinite(y), ~hit)
            np.testing.assert_array_equal(y[~hit], good[~hit])


@pytest.mark.parametrize("name", ["tiny", "mixed_kinds", "scaled", "single"])
def test_event_timing_runs_the_same_kernels(name):
    """With the kernel timing on, solves run the kernels that they run without it: the same bits,
    the steps of one workgroup among them, and every step counted."""
    steps = dict(lam=30, tol=0.0, res_tol=0.0)
    if name == "single":
        H = blqh_amd.Hamiltonian(blqh_amd.Basis(8, 8, 4, 4, 4), blqh_amd.params(8, d=3.0))
        count = 1

        def solve():
            return [H.lanczos(seed=1, **steps)]
    elif name == "scaled":
        B = blqh_amd.Basis(8, 8, -1, 1, 3)
        par = blqh_amd.params(8, d=0.6)
        h0, t = blqh_amd.Hamiltonian(B, par, terms=1), blqh_amd.Hamiltonian(B, par, terms=2)
        batch = blqh_amd.Batch.scaled([h0], [t], [0.05, 0.1])
        count = 2

        def solve():
            return batch.lanczos(seeds=[1, 2], check_every=3, **steps)
    else:
        hams = []
        for S, nphi, nel, nu, nsu, J, K in BATCHES[name]:
            B = blqh_amd.Basis(nphi, nel, nu, J, K, nspecies=S, nel_su=nsu)
            hams.append(blqh_amd.Hamiltonian(B, blqh_amd.params(nphi, d=0.9, delta_sas=0.05 if nu < 0 else 0.0)))
        batch = blqh_amd.Batch(hams)
        count = len(hams)

        def solve():
            return batch.lanczos(seeds=list(range(count)), check_every=3, **steps)
    print(name, flush=True)
    plain = solve()
    blqh_amd.profile_reset()
    blqh_amd.profile_enable(True)
    try:
        timed = solve()
        launches, ms, nbytes = blqh_amd.profile_read()
    finally:
        blqh_amd.profile_enable(False)
    for u, v in zip(plain, timed):
        assert u["E0"] == v["E0"] and u["iterations"] == v["iterations"] and u["residual"] == v["residual"]
        np.testing.assert_array_equal(u["psi"], v["psi"])
    assert launches >= max(r["iterations"] for r in timed) and ms > 0 and nbytes > 0


@pytest.mark.parametrize("case,kw", [((2, 2, 1, 1, -1, 0, 0), {}), ((2, 2, 1, -1, -1, 1, 1), dict(delta_sas=0.1)),
                                     ((1, 4, 1, -1, -1, 0, 0), None), ((2, 3, 2, -1, -1, 1, 2), dict(delta_sas=0.1)),
                                     ((2, 5, 5, -1, -1, 1, 2), dict(theta_x=0.31, theta_y=0.17, delta_sas=0.1)),
                                     ((4, 2, 2, -1, -1, 0, 1), dict(delta_sas=0.1))], ids=lambda c: str(c))
def test_layouts_of_a_few_rows(case, kw):
    """Layouts whose parts are empty or tiny (no entry beside the diagonal, no value met twice, no
    rest): the product against scipy's, for real and complex."""
    S, nphi, nel, nu, nsu, J, K = case
    B = blqh_amd.Basis(nphi, nel, nu, J, K, nspecies=S, nel_su=nsu)
    H = blqh_amd.Hamiltonian(B, blqh_amd.params(nphi) if S == 1 else blqh_amd.params(nphi, d=0.7, **kw))
    rp, col, val = H.export()
    A = sp.csr_matrix((val, col, rp), shape=(H.n, H.n))
    x = np.arange(1, H.n + 1) * (1 - 0.5j)
    for plan in ((6, 64, 512, 0, 8), (6, 64, 256, 0, 1)):
        print(f"{case} n {H.n} entries {H.nnz} plan {plan}", flush=True)
        H.set_spmv(*plan)
        scale = max(np.abs(val).max(initial=0) * np.abs(x).max() * np.diff(rp).max(initial=1), 1e-300)
        np.testing.assert_allclose(H.spmv(x), A @ x, rtol=0, atol=2e-15 * scale)


def test_default_states_match_csr_solver(built):
    """Eight steps from one start (before rounding can pick another state of a level): the default
    plan's state and coefficients are the CSR kernel's up to the order of the sums."""
    name, B, H, A = built
    if H.n < 16:
        pytest.skip("too few states for a set number of steps")
    print(f"{name} n={H.n}", flush=True)
    steps = dict(lam=8, seed=5, tol=0.0, res_tol=0.0)
    H.set_spmv(-1)
    a = H.lanczos(**steps)
    H.set_spmv(0, 16)
    b = H.lanczos(**steps)
    # a row sum's rounding, grown by at most the spread of the spectrum over beta in each step
    top = np.abs(a["alpha"]).max() + 2 * a["beta"].max()
    grown = 2.0 ** -52 * np.diff(A.indptr).max() * (top / a["beta"][1:].min()) ** 8
    tol = min(max(grown, 1e-13), 1e-6)
    np.testing.assert_allclose(a["alpha"], b["alpha"], rtol=0, atol=tol * top)
    np.testing.assert_allclose(a["beta"], b["beta"], rtol=0, atol=tol * top)
    np.testing.assert_allclose(a["psi"], b["psi"], rtol=0, atol=tol)
