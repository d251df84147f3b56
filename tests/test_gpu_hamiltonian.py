"""GPU parity of the CN step with the full NRQCD Hamiltonian (c2..c4 terms,
nrq_hamiltonian.hip) against the sparse restatement
oracle/hamiltonian_oracle.py with exact solves.

Bar: the GPU solves to FP64 true relative residual 1e-12, the oracle solves
exactly, the system is within a few per cent of the identity: propagators
within 1e-10 relative to their largest entry."""
import numpy as np
import pytest

from oracle import gaugefix_oracle as gf
from oracle import hamiltonian_oracle as ho

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


@pytest.fixture()
def cn(nrq, lattice):
    state = {"on": False}

    def init(ext, spacing, tol=1e-12):
        lattice(ext, spacing)
        nrq.nrqcd_init(2.0, [1, 0, 0, 0], 1.0, tol)
        state["on"] = True

    yield init
    if state["on"]:
        nrq.nrqcd_finalize()


def _setup(nrq, oracle, cn, ext, sp, seed=4, steps=3, precision=None):
    cn(ext, sp)
    oracle.lattice_init(ext, sp)
    lat = gf.Lattice(ext, sp, oracle.generators())
    U, E = oracle.box_init(seed, 0.7, 1.0, 1.0)
    oracle.leapfrog(U, E, 1.0, steps)
    g = nrq.GaugeConfiguration(precision) if precision else nrq.GaugeConfiguration()
    g.upload(U, E)
    if precision:
        U, E = g.download()  # the oracle sees the stored (rounded) fields
        U, E = np.asfortranarray(U), np.asfortranarray(E)
    return lat, g, U, E


def _pauli(oracle):
    return [oracle.pauli(k) for k in (1, 2, 3)]


@pytest.mark.parametrize("c", [[1, 1, 1, 1], [0.8 + 0.1j, 0.5 - 0.2j, -0.3, 0.7j], [1, 0, 0, 1.5]])
def test_full_hamiltonian_point_source(nrq, oracle, cn, c):
    ext, sp = (4, 3, 5), (0.05, 1.0, 0.9, 1.2)
    _say(f"full Hamiltonian CN 2 steps 4x3x5, c = {c}")
    lat, g, U, E = _setup(nrq, oracle, cn, ext, sp)
    h = nrq.NRQCDField()
    h.InitSinglePoint(1, 1)
    Q, A = oracle.point_prop(1), oracle.point_prop(1)
    for _ in range(2):
        st = h.Update(g, 2.0, c, 1.0)
        assert st.max_true_relres <= 1e-12 and st.solves == 12
        ho.cn_update(lat, U, E, Q, A, 2.0, c, 1.0, _pauli(oracle))
    Qg, Ag = h.download()
    assert np.max(np.abs(Qg - Q)) < 1e-10 * np.max(np.abs(Q))
    assert np.max(np.abs(Ag - A)) < 1e-10 * np.max(np.abs(A))
    for gconjg in (False, True):
        corr = h.correlators(gconjg)
        for k, v in oracle.correlators(Q, A, gconjg).items():
            assert abs(corr[k] - v) < 1e-9 * max(1.0, abs(v)), k


def test_full_hamiltonian_general_propagators_fp32_links(nrq, oracle, cn):
    ext, sp = (3, 4, 4), (0.1, 1.0, 1.0, 0.8)
    _say("full Hamiltonian, random propagators, FP32 link storage")
    lat, g, U, E = _setup(nrq, oracle, cn, ext, sp, seed=7, precision=nrq.NRQ_PRECISION_FP32)
    rng = np.random.default_rng(9)
    v = lat.vol
    Q = np.asfortranarray(rng.normal(size=(6, 6, v)) + 1j * rng.normal(size=(6, 6, v)))
    A = np.asfortranarray(rng.normal(size=(6, 6, v)) + 1j * rng.normal(size=(6, 6, v)))
    c = [0.9, 1.1 + 0.3j, 0.6, -0.8]
    h = nrq.NRQCDField()
    h.upload(Q, A)
    h.Update(g, 1.4, c, 0.7)
    ho.cn_update(lat, U, E, Q, A, 1.4, c, 0.7, _pauli(oracle))
    Qg, Ag = h.download()
    # FP32-rounded links are unitary only to ~1e-7, and the principal logarithm
    # of the plaquettes (GPU: Hermitian-pencil eigenvectors; oracle: general
    # eigen-decomposition) is defined only to that order: 1e-7 here
    assert np.max(np.abs(Qg - Q)) < 1e-7 * np.max(np.abs(Q))
    assert np.max(np.abs(Ag - A)) < 1e-7 * np.max(np.abs(A))


def test_spin_orbit_fills_the_other_spin_row(nrq, oracle, cn):
    """A single spin-colour source: without c4 the other spin rows stay exactly
    zero, with c4 they fill, as in the oracle."""
    ext, sp = (3, 3, 4), (0.05, 1.0, 1.0, 1.0)
    _say("single-dof source with and without c4")
    lat, g, U, E = _setup(nrq, oracle, cn, ext, sp, seed=2)
    for c in ([1, 1, 1, 0], [1, 1, 1, 1]):
        h = nrq.NRQCDField()
        h.InitSinglePointSingleDoF(1, 2, 5, 2, 3, 7)
        Q, A = [np.asfortranarray(x) for x in h.download()]
        h.Update(g, 2.0, c, 1.0)
        ho.cn_update(lat, U, E, Q, A, 2.0, c, 1.0, _pauli(oracle))
        Qg, Ag = h.download()
        assert np.max(np.abs(Qg - Q)) < 1e-10 * np.max(np.abs(Q))
        assert np.max(np.abs(Ag - A)) < 1e-10 * np.max(np.abs(A))
        mixed = max(np.abs(Qg[d, j]).max() for j in range(6) for d in range(6) if d % 2 != j % 2)
        assert (mixed == 0.0) if c[3] == 0 else (mixed > 1e-8)


def test_full_hamiltonian_reports_nonconvergence(nrq, oracle, cn):
    """The columns of a step are solved together: with an iteration cap below
    what they need, the step reports NRQ_ERR_NOCONV instead of returning the
    unconverged fields as converged; with the cap lifted, the next step
    converges every column again."""
    ext, sp = (4, 3, 5), (0.05, 1.0, 0.9, 1.2)
    _say("full Hamiltonian, iteration cap 2")
    lat, g, U, E = _setup(nrq, oracle, cn, ext, sp)
    h = nrq.NRQCDField()
    h.InitSinglePoint(1, 1)
    nrq.nrqcd_set_solver(nrq.NRQ_SOLVER_GMRES_FP64, 30, 2)
    try:
        with pytest.raises(nrq.NRQError) as err:
            h.Update(g, 2.0, [1, 1, 1, 1], 1.0)
        assert err.value.code == -5  # NRQ_ERR_NOCONV
    finally:
        nrq.nrqcd_set_solver(nrq.NRQ_SOLVER_GMRES_FP64, 30, 10000)
    Q, A = h.download()
    assert np.all(np.isfinite(Q)) and np.all(np.isfinite(A))
    st = h.Update(g, 2.0, [1, 1, 1, 1], 1.0)
    assert st.max_true_relres <= 1e-12 and st.solves == 12


def test_full_hamiltonian_column_batches_are_bit_identical(nrq, oracle, cn, monkeypatch):
    """A Krylov-storage budget of five columns (NRQ_HAM_BATCH_BYTES) solves the
    12 columns of a step in batches of 5, 5 and 2: the same fields, bit for
    bit, as all 12 together, since every column takes the same operations in
    either case."""
    ext, sp = (4, 3, 5), (0.05, 1.0, 0.9, 1.2)
    _say("full Hamiltonian, column batches of 5 against 12")
    lat, g, U, E = _setup(nrq, oracle, cn, ext, sp)
    c = [1, 1, 1, 1]
    whole = nrq.NRQCDField()
    whole.InitSinglePoint(1, 1)
    st = whole.Update(g, 2.0, c, 1.0)
    assert st.solves == 12
    per_col = 16 * (30 + 3) * 6 * lat.vol
    monkeypatch.setenv("NRQ_HAM_BATCH_BYTES", str(5 * per_col + 1))
    parts = nrq.NRQCDField()
    parts.InitSinglePoint(1, 1)
    st = parts.Update(g, 2.0, c, 1.0)
    assert st.solves == 12 and st.max_true_relres <= 1e-12
    Qa, Aa = whole.download()
    Qb, Ab = parts.download()
    assert np.array_equal(Qa, Qb) and np.array_equal(Aa, Ab)


@pytest.mark.parametrize("ext", [(4, 4, 4), (5, 13, 2), (3, 7, 9)])
def test_full_hamiltonian_at_the_edges_of_wavefronts(nrq, oracle, cn, ext):
    """Volumes of one whole, two and a fraction, and three minus a few
    wavefronts of sites, with an odd number of columns on each propagator (a
    thread of the operator takes two)."""
    sp = (0.05, 1.0, 0.9, 1.2)
    _say(f"full Hamiltonian, {ext}")
    lat, g, U, E = _setup(nrq, oracle, cn, ext, sp, seed=5)
    rng = np.random.default_rng(12)
    v = lat.vol
    Q = np.asfortranarray(rng.normal(size=(6, 6, v)) + 1j * rng.normal(size=(6, 6, v)))
    A = np.asfortranarray(rng.normal(size=(6, 6, v)) + 1j * rng.normal(size=(6, 6, v)))
    Q[:, 3] = 0.0
    A[:, 1:4] = 0.0
    c = [0.9, 1.1 + 0.3j, 0.6, -0.8]
    h = nrq.NRQCDField()
    h.upload(Q, A)
    st = h.Update(g, 1.4, c, 0.7)
    assert st.solves == 8 and st.max_true_relres <= 1e-12
    ho.cn_update(lat, U, E, Q, A, 1.4, c, 0.7, _pauli(oracle))
    Qg, Ag = h.download()
    assert np.max(np.abs(Qg - Q)) < 1e-10 * np.max(np.abs(Q))
    assert np.max(np.abs(Ag - A)) < 1e-10 * np.max(np.abs(A))
