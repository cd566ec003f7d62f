"""The dense-propagator kernels: the exact exponential (one wave per vector) at
the edges of its row and column classes, against the oracle: site counts on
both sides of every class boundary, windows of one and two steps, one sample
and a sample count that leaves no full workgroup pattern.  Tolerance 1e-5
relative L2 as for every exact-exponential result (FP32 state, FP64
exponential)."""
import numpy as np
import pytest

from nise_2017_amd import abi, synth

from test_gpu_multi import rel, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,ns,sr", [(1, 3, 2), (2, 1, 1), (23, 5, 9)])
def test_class_edges(orc, T, ns, sr):
    Ns = [1, 7, 8, 9, 16, 17, 24, 25, 32, 33, 40, 41, 48, 49, 56, 57, 63, 64]
    systems = [system(N, 0, 700 + N, T=T, ns=ns, sr=sr) for N in Ns]
    print(f"[dense] T={T} ns={ns} every {sr}", flush=True)
    out, _ = abi.absorption_multi(systems)
    for (non, H, mu, Cr), (re, im) in zip(systems, out):
        o_re, o_im = orc.absorption(non, H, mu, C_rec=Cr)
        e = rel(re + 1j * im, o_re + 1j * o_im)
        assert e < 1e-5, (non.singles, e)
    assert np.isfinite(out[-1][0]).all()


def lattice_case(N, T, ns, sr, seed, ts=1, begin=0, **kw):
    """N sites of a dipole lattice, Full records."""
    L = int(np.ceil(np.sqrt(N)))
    rng, mus, coup = synth.lattice_static(L, seed=seed)
    nfr = (begin + ns - 1) * sr + T + 2
    H = synth.full_records(synth.lattice_diag(rng, nfr, L * L), coup)
    a, b = np.triu_indices(L * L)
    keep = (a < N) & (b < N)
    H = np.ascontiguousarray(np.concatenate([H[:, :1], H[:, 1:][:, keep]], axis=1))
    mu = synth.dipole_records(mus[:N], nfr)
    lo, hi = synth.shifted_center(H, N)
    non = abi.make_non(singles=N, tmax1=T, sample=sr, begin=begin, end=begin + ns, ts=ts, propagation=1, deltat=2.0,
                       min1=lo, max1=hi, **kw)
    non.shifte = np.float32((np.float32(hi) + np.float32(lo)) / np.float32(2))
    return non, H, mu


def both(non, H, mu, C=None):
    """The default plan (checked to run one workgroup per sample) and the row
    conveyor on the same records."""
    p = abi.AbsPlan(non, H, H.shape[1], mu, mu.shape[1], H.shape[0], C)
    try:
        assert p.info()["nwg"] == non.end - non.begin
        dense = p.execute()
        graph = [p.execute(flags=2) for _ in range(3)]
        p.set_rows(0)
        rows = p.execute()
    finally:
        p.close()
    for g in graph:
        assert np.array_equal(g[0], dense[0]) and np.array_equal(g[1], dense[1])
    return dense[0] + 1j * dense[1], rows[0] + 1j * rows[1]


@pytest.mark.parametrize("N,T,ns,sr,ts,begin", [
    (65, 40, 9, 3, 1, 0), (95, 33, 4, 5, 2, 1), (96, 24, 5, 30, 1, 0), (97, 40, 7, 4, 1, 2), (127, 30, 3, 2, 1, 0),
    (128, 41, 8, 3, 2, 0), (64, 64, 10, 4, 1, 3), (33, 50, 7, 5, 2, 0), (5, 64, 6, 7, 1, 0), (66, 2, 3, 1, 1, 0)])
def test_trotter_propagators_against_conveyor(orc, N, T, ns, sr, ts, begin):
    """The Trotter scheme through per-frame propagators against the row
    conveyor and the oracle: both sides of every row class, odd N, Trotter
    substeps, samples that do not start at frame 0, windows with gaps, graph
    replays.  1e-5 as for the conveyor: the distance between the two grows with
    the sweeps (tmax times substeps), at most 7.1e-6 after 128 (test_longest_runs
    has the largest)."""
    non, H, mu = lattice_case(N, T, ns, sr, seed=800 + N, ts=ts, begin=begin)
    print(f"[dense] Trotter N={N} T={T}", flush=True)
    d, r = both(non, H, mu)
    assert rel(d, r) < 1e-5
    o_re, o_im = orc.absorption(non, H, mu)
    assert rel(d, o_re + 1j * o_im) < 1e-5


@pytest.mark.parametrize("N,T,ts", [(25, 256, 1), (25, 32, 8), (77, 256, 1), (77, 128, 2), (77, 64, 4)])
def test_longest_runs(orc, N, T, ts):
    """The most sweeps that go through propagators (256): within 1.5e-5 of the
    reference's rounding, oracle and conveyor (twice the 7.1e-6 measured after
    128 sweeps: each sweep's rounding is biased the same way), and nearer to
    64 bits than it."""
    non, H, mu = lattice_case(N, T, 8, 5, seed=840 + N + ts, ts=ts)
    print(f"[dense] 256 sweeps: N={N} T={T} ts={ts}", flush=True)
    d, r = both(non, H, mu)
    assert not np.array_equal(d, r)
    o_re, o_im = orc.absorption(non, H, mu)
    assert rel(d, r) < 1.5e-5 and rel(d, o_re + 1j * o_im) < 1.5e-5
    x_re, x_im = orc.absorption(non, H, mu, f64=True)
    x = x_re + 1j * x_im
    assert rel(d, x) < rel(r, x)


@pytest.mark.parametrize("N,T,ts", [(25, 129, 2), (77, 128, 3), (77, 33, 8)])
def test_runs_of_more_sweeps_keep_the_conveyor(N, T, ts):
    """Substeps count: past 256 sweeps the default is the conveyor, bit for bit."""
    non, H, mu = lattice_case(N, T, 8, 5, seed=850 + N, ts=ts)
    print(f"[dense] {T * ts} sweeps: N={N} T={T} ts={ts}", flush=True)
    p = abi.AbsPlan(non, H, H.shape[1], mu, mu.shape[1], H.shape[0])
    default = p.execute()
    p.set_rows(0)
    rows = p.execute()
    p.close()
    assert np.array_equal(default[0], rows[0]) and np.array_equal(default[1], rows[1])


def test_trotter_propagators_coupling_type_and_shifts():
    """Coupling type with static dipoles, single-site shifts, host and device records."""
    import torch
    N, T, ns = 70, 30, 6
    non, H, mu = lattice_case(N, T, ns, 4, seed=870, hamiltonian="Coupling", couplingcut=0.2,
                              single_shift=[(3, 1.0, 25.0), (69, 0.9, -4.0)])
    a, b = np.triu_indices(N)
    Hc = np.ascontiguousarray(np.concatenate([H[:, :1], H[:, 1:][:, a == b]], axis=1))
    Cr, muc = np.ascontiguousarray(H[0]), np.ascontiguousarray(mu[:1])
    d, r = both(non, Hc, muc, Cr)
    assert rel(d, r) < 1e-5
    x = [torch.from_numpy(v).cuda() for v in (Hc, muc, Cr)]
    torch.cuda.synchronize()
    p = abi.AbsPlan(non, x[0], Hc.shape[1], x[1], muc.shape[1], Hc.shape[0], x[2], where=abi.NISE_DEVICE)
    re, im = p.execute()
    p.close()
    assert np.array_equal(re + 1j * im, d)


@pytest.mark.parametrize("N,T,ns,sr", [(40, 60, 200, 14), (90, 60, 90, 14), (126, 256, 3, 90)])
def test_noalloc_windows_match_plan(N, T, ns, sr):
    """A run whose propagators exceed the fixed scratch array: windows of
    samples, and segments of a sample's steps where one window is too large,
    bit for bit the plan's result."""
    import ctypes as C

    import torch
    non, H, mu = lattice_case(N, T, ns, sr, seed=880 + N)
    Hd, mud = torch.from_numpy(H).cuda(), torch.from_numpy(mu).cuda()
    torch.cuda.synchronize()
    p = abi.AbsPlan(non, Hd, H.shape[1], mud, mu.shape[1], H.shape[0], where=abi.NISE_DEVICE)
    assert p.info()["nwg"] == ns
    re, im = p.execute()
    p.close()
    r1, i1 = np.zeros(T, np.float32), np.zeros(T, np.float32)
    abi.check(abi.lib().nise_absorption_batched_noalloc(C.byref(non), abi.ptr(Hd), H.shape[1], abi.ptr(mud), mu.shape[1],
                                                        H.shape[0], None, r1, i1))
    assert np.array_equal(re, r1) and np.array_equal(im, i1)


def test_gradient_from_propagator_checkpoints(orc):
    """The adjoint from checkpoints that the propagator kernels wrote (N <= 64
    and above), against the conveyor's."""
    from nise_2017_amd import adjoint
    for N in (20, 70):
        non, H, mu = lattice_case(N, 40, 6, 5, seed=890 + N)
        g = np.linspace(1.0, -0.5, 40)
        got = []
        for rows in (None, 4):
            m = adjoint.AdjointAbsorption(non, H, mu, every=7, rows=rows)
            m.forward(np.full(N, 0.5, np.float32), 1.02)
            gd, gc = m.backward(g, g[::-1].copy())
            got.append(np.concatenate([gd, [gc]]))
            m.close()
        assert rel(got[0], got[1]) < 1e-4
