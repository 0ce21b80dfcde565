"""The work that a user of the engine has it do, case by case, through the public
classes of blqh_amd: ground states of one sector (Hamiltonian resident, rebuilt for
a new parameter point, or from the basis on), batched ground states of all sectors,
shared-scale sweeps, the warm-start network's loss and gradient, and observables.

Sizes: the README run, the two-species sectors at N_phi = 12, 14 and 16, the spinful
sectors at N_phi = 8 and the monolayer sectors at N_phi = 18, as bench.py and the
tests use them.  The layer distance d (for the monolayer, the aspect ratio) and the
start vectors come from the seed.
"""
import math

import numpy as np

import blqh_amd

# Lanczos steps to the stopping rule (|dE| < 1e-10 and residual < 1e-7) that work()
# charges; solves take 20 (79 states) to 160.
STEPS = 100


def listed():
    # psi=True: the state is wanted and the sector's ground level is not degenerate, so that
    # the state is as well defined as the energy
    return [
        # the README's run: the smallest sector anyone solves; latency and launches count
        dict(name="solve_nphi8_readme", kind="solve", S=2, nphi=8, nel=8, nel_up=4, J=4, K=4, d=3.0, dsas=0.0, chk=1,
             lam=200, converge=True, psi=True),
        # one complex sector of the N_phi = 12 sweep, 18.8k states
        dict(name="solve_nphi12_complex", kind="solve", S=2, nphi=12, nel=12, nel_up=-1, J=3, K=8, d=1.0, dsas=0.05,
             chk=1, lam=200, converge=True, psi=True),
        # a real sector at N_phi = 14, 205k states
        dict(name="solve_nphi14_real", kind="solve", S=2, nphi=14, nel=14, nel_up=-1, J=7, K=7, d=1.0, dsas=0.05,
             chk=1, lam=200, converge=True, psi=True),
        # the largest: 2.35M states, 831M entries (bench.py's default, its check interval)
        dict(name="solve_nphi16_all", kind="solve", S=2, nphi=16, nel=16, nel_up=-1, J=0, K=0, d=1.0, dsas=0.02,
             chk=5, lam=200, converge=True, psi=True),
        # the next parameter point of one sector: Hamiltonian, then its ground state
        dict(name="point_nphi12", kind="point", S=2, nphi=12, nel=12, nel_up=-1, J=5, K=6, d=1.0, dsas=0.05, chk=1,
             lam=200, converge=True, psi=True),
        dict(name="point_nphi16_u8", kind="point", S=2, nphi=16, nel=16, nel_up=8, J=0, K=0, d=1.0, dsas=0.0, chk=5,
             lam=200, converge=True, psi=True),
        # what the command line does: basis, Hamiltonian and ground state of a new sector
        dict(name="cold_nphi14", kind="cold", S=2, nphi=14, nel=14, nel_up=-1, J=3, K=5, d=1.0, dsas=0.05, chk=1,
             lam=200, converge=True, psi=True),
        # the energies of all 64 spinful sectors of one parameter point in one batch
        dict(name="batch_spin_nphi8", kind="batch", S=4, nphi=8, nel=8, nel_up=4, nel_su=4, d=1.0, dsas=0.05, chk=2),
        # many tiny problems: the K-resolved monolayer spectrum, 108 sectors of about 175 states
        dict(name="batch_mono_nphi18", kind="batch", S=1, nphi=18, nel=6, nel_up=-1, nel_su=-1, d=0.0, dsas=0.0,
             chk=2),
        # one d of the N_phi = 12 sweep: 144 sectors times three tunnelling strengths
        dict(name="sweep_nphi12", kind="sweep", nphi=12, nel=12, d=0.4, scales=3, chk=2),
        # forward and backward of the warm-start network on one training minibatch
        dict(name="mlp_grad_28", kind="mlp", nbits=28, count=4096),
        # observables of a state of 205k components
        dict(name="observables_nphi14", kind="obs", S=2, nphi=14, nel=14, nel_up=-1, nel_su=-1, J=0, K=0),
    ]


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "point", "cold", "batch", "sweep", "mlp", "obs"])
    d, chk = round(rng.uniform(0.2, 3.0), 3), rng.choice([1, 1, 2, 5])
    if kind == "mlp":
        return dict(kind=kind, nbits=rng.randint(12, 64), count=int(round(math.exp(rng.uniform(math.log(16), math.log(65536))))))
    if kind == "sweep":
        n = rng.randint(6, 10)
        return dict(kind=kind, nphi=n, nel=n, d=d, scales=rng.randint(1, 4), chk=chk)
    if kind == "batch":
        if rng.random() < 0.3:
            nel = rng.choice([4, 5, 6])
            return dict(kind=kind, S=1, nphi=nel * rng.choice([2, 3]), nel=nel, nel_up=-1, nel_su=-1, d=0.0, dsas=0.0, chk=chk)
        if rng.random() < 0.4:
            n = rng.choice([4, 6])
            return dict(kind=kind, S=4, nphi=n, nel=n, nel_up=n // 2, nel_su=n // 2, d=d, dsas=0.05, chk=chk)
        n = rng.randint(6, 10)
        return dict(kind=kind, S=2, nphi=n, nel=n, nel_up=-1, nel_su=-1, d=d, dsas=rng.choice([0.0, 0.05, 0.1]), chk=chk)
    # one sector: the dimension grows about 3.6-fold with each flux quantum, so an even
    # choice of N_phi spreads the size over its logarithm
    n = rng.randint(7, 15 if kind != "cold" else 14)
    fixed = rng.random() < 0.3
    c = dict(kind=kind, S=2, nphi=n, nel=n, nel_up=n // 2 if fixed else -1, J=rng.randrange(n), K=rng.randrange(n))
    if kind == "obs":
        return dict(c, nel_su=-1)
    c.update(d=d, dsas=0.0 if fixed else rng.choice([0.0, 0.05, 0.1]), chk=chk)
    # any sector, its ground level degenerate or not: to the stopping rule for the energy, or a
    # set number of steps (the reference's way), short of convergence, for the state as well
    if rng.random() < 0.5:
        return dict(c, lam=200, converge=True, psi=False)
    return dict(c, d=round(rng.uniform(0.2, 2.0), 3), lam=rng.randint(7, 12), converge=False, psi=True)


def _rng(seed):
    return np.random.default_rng(1000003 * int(seed) + 17)


def _d(case, seed):
    return case["d"] + 0.05 * float(_rng(seed).random())


def _params(case, seed):
    if case["S"] == 1:
        return blqh_amd.params(case["nphi"], gamma=1.0 + 0.05 * float(_rng(seed).random()))
    if case["S"] == 4:
        return blqh_amd.params(case["nphi"], d=_d(case, seed), delta_sas=case["dsas"], delta_v=0.02, delta_z=0.01)
    return blqh_amd.params(case["nphi"], d=_d(case, seed), delta_sas=case["dsas"])


def _basis(case, J=None, K=None):
    return blqh_amd.Basis(case["nphi"], case["nel"], case.get("nel_up", -1), case["J"] if J is None else J,
                          case["K"] if K is None else K, nspecies=case.get("S", 2), nel_su=case.get("nel_su", -1))


def _sectors(case):
    nphi, nel = case["nphi"], case["nel"]
    nk = math.gcd(nphi, nel) if case.get("S") == 1 else nphi
    return [(J, K) for J in range(nphi) for K in range(nk)]


def prepare(case, seed):
    kind, rng = case["kind"], _rng(seed)
    state = dict(case=case, seed=int(rng.integers(1, 1 << 31)))
    if kind == "mlp":
        nbits, n = case["nbits"], case["count"]
        net = blqh_amd.Mlp(nbits, seed=state["seed"])
        net.params = net.params + rng.normal(0, 0.05, net.nparams).astype(np.float32)
        state.update(net=net, data=_minibatch(rng, nbits, n))
    elif kind == "obs":
        B = _basis(case)
        psi = (rng.normal(size=B.n) + 1j * rng.normal(size=B.n)) * np.exp(rng.normal(0, 2, B.n))
        state.update(basis=B, psi=psi / np.linalg.norm(psi))
    elif kind == "batch":
        par = _params(case, seed)
        state["hams"] = [blqh_amd.Hamiltonian(_basis(case, J, K), par) for J, K in _sectors(case)]
        state["batch"] = blqh_amd.Batch(state["hams"])
        state["seeds"] = rng.integers(0, 1 << 31, len(state["hams"])).astype(np.uint32)
    elif kind == "sweep":
        par = blqh_amd.params(case["nphi"], d=_d(case, seed))
        bases = [_basis(dict(case, nel_up=-1), J, K) for J, K in _sectors(case)]
        h0 = [blqh_amd.Hamiltonian(B, par, terms=1) for B in bases]
        t = [blqh_amd.Hamiltonian(B, par, terms=2) for B in bases]
        scales = [0.0, 0.05, 0.1, 0.15][:case["scales"]]
        state["batch"] = blqh_amd.Batch.scaled(h0, t, scales)
        state["seeds"] = rng.integers(0, 1 << 31, len(bases) * len(scales)).astype(np.uint32)
    else:
        state["par"] = _params(case, seed)
        if kind != "cold":
            state["basis"] = _basis(case)
        if kind == "solve":
            state["ham"] = blqh_amd.Hamiltonian(state["basis"], state["par"])
    return state


def _minibatch(rng, nbits, n):
    words = rng.integers(0, (1 << nbits) - 1, size=n, dtype=np.uint64, endpoint=True)
    return (words, rng.uniform(0, 3, n).astype(np.float32), rng.choice([0.0, 0.05, 0.1], n).astype(np.float32),
            rng.normal(-4, 2, n).astype(np.float32), rng.integers(0, 2, n).astype(np.float32))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "mlp":
        loss, grad = state["net"].loss_grad(*state["data"])
        return {"loss": loss, "grad": grad}
    if kind == "obs":
        o = blqh_amd.observables(state["basis"], state["psi"])
        return {"occupation": o["occupation"], "sz": o["pseudospin_sz"], "sx": o["pseudospin_sx"]}
    if kind in ("batch", "sweep"):
        r = state["batch"].lanczos(lam=200, seeds=state["seeds"], check_every=case["chk"], want_psi=False)
        return {"E0": np.array([x["E0"] for x in r]), "E_rq": np.array([x["E_rq"] for x in r])}
    basis = _basis(case) if kind == "cold" else state["basis"]
    ham = state["ham"] if kind == "solve" else blqh_amd.Hamiltonian(basis, state["par"])
    r = ham.lanczos(lam=case["lam"], seed=state["seed"], check_every=case["chk"], want_psi=case["psi"],
                    tol=1e-10 if case["converge"] else 0.0)
    out = {"E0": np.array(r["E0"])}
    if case["psi"]:
        out.update(E_rq=np.array(r["E_rq"]), psi=r["psi"])
    if not case["converge"]:
        out.update(alpha=r["alpha"], beta=r["beta"])
    if kind == "cold":
        out.update(id=basis.id.view(np.int64), period=basis.period)
    return out


def _words(case):
    """Sector words of one J (all J equal), orbits, and entries of a row, about."""
    S, nphi, nel, up = case.get("S", 2), case["nphi"], case["nel"], case.get("nel_up", -1)
    bits = S * nphi
    if S == 1:
        words = math.comb(bits, nel)
    elif up >= 0:
        words = math.comb(bits // 2, up) * math.comb(bits // 2, nel - up)
        if S == 4:  # spin-up count fixed too: about the share of the most likely one
            words *= 0.3
    else:
        words = math.comb(bits, nel)
    empty = 1 - nel / bits
    row = 0.75 * nel * (nel - 1) / 2 * nphi * empty * empty * (0.6 if S == 1 else 1.3 if S == 4 else 1)
    order = math.gcd(nphi, nel) if S == 1 else nphi
    return words / nphi, max(1.0, words / nphi / order), max(1.0, row)


def work(case):
    """A solve reads every entry (value, 8 bytes in the real sectors and 16 in the complex
    ones, and a 2-byte column) once a step, and the vectors of the recurrence (48 bytes a
    row): no step can begin before the last one has ended.  A build writes 20 bytes an
    entry; a basis writes a 4-byte table entry a word."""
    kind = case["kind"]
    if kind == "mlp":
        p = (case["nbits"] + 2) * 64 + 64 + 4096 + 64 + 130
        return {"bytes": 24.0 * case["count"] + 8.0 * p, "flops": 6.0 * p * case["count"]}
    words, n, row = _words(case)
    nnz = n * row
    if kind == "obs":
        # every translation of a row tries one hop per orbital
        return {"bytes": 26.0 * n + 16.0 * n, "flops": 8.0 * n * case["nphi"] ** 2}
    steps = 35 if case.get("S") == 1 else 20 if n < 100 else STEPS
    if not case.get("converge", True):
        steps = case["lam"]
    if kind in ("batch", "sweep"):
        P, G = len(_sectors(case)), case.get("scales", 1)
        return {"bytes": P * steps * (18.0 * nnz + 48.0 * n * G), "flops": P * G * steps * 8.0 * nnz}
    real = 2 * case["K"] % case["nphi"] == 0
    b = steps * ((10.0 if real else 18.0) * nnz + 48.0 * n)
    if kind != "solve":
        b += 20.0 * nnz
    if kind == "cold":
        b += 4.0 * words
    return {"bytes": b, "flops": steps * (4.0 if real else 8.0) * nnz}


# ---- 64-bit values, in plain numpy ------------------------------------------------


def _start(n, seed):
    """std::mt19937(seed): draw 2i is the imaginary, 2i + 1 the real part of entry i."""
    g = np.random.MT19937()
    g._legacy_seeding(int(seed))
    u = g.random_raw(2 * n).astype(np.float64) / 4294967295.0 - 0.5
    v = u[1::2] + 1j * u[0::2]
    return v / np.linalg.norm(v)


def _ground(csr, seed, steps=0):
    """Ground state from the same start: Lanczos with full reorthogonalisation, `steps` steps or
    to convergence.  (E0, E_rq, psi, alpha, beta)"""
    rowptr, col, val = csr
    n = len(rowptr) - 1
    real = np.all(val.imag == 0)
    val = val.real.copy() if real else val
    mul = lambda x: np.add.reduceat(val * x[col], rowptr[:-1])  # noqa: E731  (no row is empty: the diagonal)
    V = np.empty(((steps or min(n, 200)) + 1, n), np.complex128)
    V[0] = _start(n, seed)
    a, b = [], []
    for j in range(len(V) - 1):
        w = mul(V[j])
        a.append(float(np.vdot(V[j], w).real))
        for _ in range(2):
            w = w - V[:j + 1].T @ (V[:j + 1].conj() @ w)
        b.append(float(np.linalg.norm(w)))
        e, s = np.linalg.eigh(np.diag(a) + np.diag(b[:-1], 1) + np.diag(b[:-1], -1))
        if not steps and abs(b[-1] * s[-1, 0]) < 1e-10:  # further on, rounding brings in other states of a degenerate level
            break
        V[j + 1] = w / b[-1]
    u = s[:, 0] @ V[:len(a)]
    u *= np.exp(-1j * np.angle(np.vdot(V[0], u))) / np.linalg.norm(u)
    psi = u.conj()
    return e[0], float(np.vdot(psi, mul(psi)).real), psi, np.array(a), np.array([1.0] + b)


def exact(case, seed):
    """Solves of a resident matrix: the matrix is what the program has in hand.  The other
    single sectors build theirs inside the pass (seconds to minutes in numpy): None."""
    kind = case["kind"]
    if kind == "mlp":
        return _exact_mlp(prepare(case, seed), case["nbits"])
    if kind == "obs":
        return _exact_obs(prepare(case, seed))
    if kind == "solve" and _words(case)[1] < 20000:
        s = prepare(case, seed)
        r = _ground(s["ham"].export(), s["seed"], 0 if case["converge"] else case["lam"])
        out = dict(zip(("E0", "E_rq", "psi", "alpha", "beta"), map(np.asarray, r)))
        keep = {"E0"} | ({"E_rq", "psi"} if case["psi"] else set())
        return {k: v for k, v in out.items() if k in keep or not case["converge"]}
    if kind == "batch" and len(_sectors(case)) * _words(case)[1] < 25000:
        s = prepare(case, seed)
        r = [_ground(H.export(), q) for H, q in zip(s["hams"], s["seeds"])]
        return {"E0": np.array([x[0] for x in r]), "E_rq": np.array([x[1] for x in r])}
    return None


def _exact_obs(state):
    c, B = state["case"], state["basis"]
    nphi, p = c["nphi"], np.abs(state["psi"]) ** 2
    bits = (B.id[:, None] >> np.arange(2 * nphi, dtype=np.uint64)) & np.uint64(1)
    layer = bits.reshape(-1, 2, nphi).astype(np.float64)
    D = B.period.astype(np.int64)
    occ = np.zeros((2, nphi))
    for q in range(nphi):
        w = np.where(q < D, p / D, 0.0)
        occ += np.tensordot(w, np.roll(layer, q, axis=2), axes=(0, 0))
    return {"occupation": occ, "sz": (2 * float(p @ layer[:, 0].sum(1)) - c["nel"]) / (2 * c["nel"]), "sx": None}


def _exact_mlp(state, nbits):
    words, d, dsas, ya, ys = state["data"]
    t, nin, o, parts = state["net"].params.astype(np.float64), nbits + 2, 0, []
    for shape in ((nin, 64), (64,), (64, 64), (64,), (64, 2), (2,)):
        parts.append(t[o:o + math.prod(shape)].reshape(shape))
        o += math.prod(shape)
    W1, b1, W2, b2, W3, b3 = parts
    bit = ((words[:, None] >> np.arange(nbits, dtype=np.uint64)) & np.uint64(1)).astype(np.float64)
    X = np.concatenate([2 * bit - 1, d.astype(np.float64)[:, None] / 3, 10 * dsas.astype(np.float64)[:, None]], 1)
    h1 = np.tanh(X @ W1 + b1)
    h2 = np.tanh(h1 @ W2 + b2)
    z = h2 @ W3 + b3
    n, ya, ys = len(words), ya.astype(np.float64), ys.astype(np.float64)
    loss = float(np.mean((z[:, 0] - ya) ** 2 + np.logaddexp(0.0, z[:, 1]) - ys * z[:, 1]))
    g = np.stack([2 * (z[:, 0] - ya), 1 / (1 + np.exp(-z[:, 1])) - ys], 1) / n
    d2 = (g @ W3.T) * (1 - h2 ** 2)
    d1 = (d2 @ W2.T) * (1 - h1 ** 2)
    return {"loss": loss, "grad": np.concatenate([(X.T @ d1).ravel(), d1.sum(0), (h1.T @ d2).ravel(), d2.sum(0),
                                                  (h2.T @ g).ravel(), g.sum(0)])}
