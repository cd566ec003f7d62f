"""The basis-vector path of nise_2dir_batched (t1 windows of 16 steps and
more) at the edges of its lane and column classes, against the oracle's item
loop: one site, both sides of every lanes-per-vector class, the largest N,
t1 windows of 64, 65 and 130 steps, one t3 step (without the EA pathway: at
t3 = 0 the three pathways of harmonic transitions sum to zero), Trotter substeps, every
technique, per-frame anharmonicities, the Coupling type, samples that do not
start at frame 0.  Large N and short t3 windows take the pathways apart: their
sum there is a difference of about 1e-3 of its terms, in which the FP32
oracle is itself 2e-4 to 1.4e-3 off the 64-bit result (test_large_n_sum
compares both with it).  Tolerance as in test_gpu_2dir.py."""
import numpy as np
import pytest

from nise_2017_amd import abi, synth

from test_gpu_2dir import TOL, mk, rel

pytestmark = pytest.mark.gpu


def check(orc, make, H, mu, **rec):
    ref = orc.twodir(make(), H, mu, acc64=True, **{k: v for k, v in (("A_rec", rec.get("anh")), ("over_rec", rec.get("over")),
                                                              ("C_rec", rec.get("C"))) if v is not None})
    R = abi.twodir_batched(make(), H, mu, coupling_rec=rec.get("C"), anh_rec=rec.get("anh"), over_rec=rec.get("over"))
    assert rel(R, ref) < TOL


@pytest.mark.parametrize("N,T1,T3,ts,tech", [
    (1, 16, 3, 1, "2DIR"), (2, 17, 5, 2, "2DIR"), (3, 16, 1, 1, "noEAIR"), (7, 16, 4, 1, "2DUVvis"),
    (8, 16, 4, 1, "2DIR"), (9, 20, 3, 1, "2DUVvis"), (16, 16, 4, 1, "2DIR"), (17, 18, 3, 2, "2DIR"),
    (32, 16, 3, 1, "2DUVvis"), (33, 16, 3, 1, "EAIR"), (45, 16, 2, 1, "EAIR"), (61, 22, 2, 1, "EAIR"), (61, 22, 2, 1, "noEAIR"),
    (5, 64, 3, 1, "2DIR"), (5, 65, 2, 1, "2DUVvis"), (4, 130, 2, 1, "2DIR"),
    (4, 16, 5, 1, "GBIR"), (4, 16, 5, 1, "SEIR"), (4, 16, 5, 1, "EAIR"), (4, 16, 5, 1, "noEAUVvis")])
def test_edges_vs_oracle(orc, N, T1, T3, ts, tech):
    print(f"[basis] N={N} T1={T1} T3={T3} ts={ts} {tech}", flush=True)
    H, mu = synth.ring_2dir(N=N, nframes=T1 + T3 + 30, seed=900 + N + T1)
    check(orc, lambda: mk(N, T1, T3, 7, 1, 4, H, ts=ts, technique=tech, lifetime=400.0), H, mu)


@pytest.mark.parametrize("coupled", [True, False])
def test_records_vs_oracle(orc, coupled):
    """Per-frame anharmonicities and overtone dipoles, with and without couplings."""
    N, T1, T3 = 5, 19, 6
    H, mu, anh, over = synth.twodir_system(N=N, nframes=80, seed=951, coupled=coupled)
    check(orc, lambda: mk(N, T1, T3, 5, 0, 6, H, anharmonicity=0.0), H, mu, anh=anh, over=over)


def test_dense_coupling_type_vs_oracle(orc):
    """Every pair coupled (Coupling type, static dipoles), host and device records alike."""
    import torch
    N, T1, T3 = 12, 16, 4
    rng, mus, coup = synth.lattice_static(4, seed=961, cut=0.0)
    n = np.arange(N)
    Hf = synth.full_records(synth.lattice_diag(rng, 60, 16), coup)
    a, b = np.triu_indices(16)
    keep = np.isin(a, n) & np.isin(b, n)
    Hf = np.ascontiguousarray(np.concatenate([Hf[:, :1], Hf[:, 1:][:, keep]], axis=1))
    a, b = np.triu_indices(N)
    Hc = np.ascontiguousarray(np.concatenate([Hf[:, :1], Hf[:, 1:][:, a == b]], axis=1))
    Cr, mur = np.ascontiguousarray(Hf[0]), synth.dipole_records(mus[:N], 1)
    make = lambda: mk(N, T1, T3, 6, 0, 5, Hf, hamiltonian="Coupling", technique="EAIR")  # noqa: E731
    check(orc, make, Hc, mur, C=Cr)
    R = abi.twodir_batched(make(), Hc, mur, coupling_rec=Cr)
    dev = [torch.from_numpy(x).cuda() for x in (Hc, mur, Cr)]
    torch.cuda.synchronize()
    assert np.array_equal(R, abi.twodir_batched(make(), dev[0], dev[1], coupling_rec=dev[2]))


@pytest.mark.parametrize("N,T1,T3,S", [(33, 16, 3, 4), (45, 16, 2, 4), (61, 22, 2, 3), (40, 30, 20, 3)])
def test_large_n_sum_vs_64_bits(orc, N, T1, T3, S):
    """The sum of the three pathways above N = 32 against direct propagation in
    64 bits: no further off than the reference's FP32 arithmetic (the oracle; 1.5
    for the chance of two roundings of the same size)."""
    from perf import cases
    case = dict(kind="2dir", N=N, t1=T1, t3=T3, samples=S, every=9, anh=16.0)
    print(f"[basis] 64 bits: N={N} T1={T1} T3={T3}", flush=True)
    s = cases.prepare(case, 77)
    R = cases.run(s)
    exact = cases.exact(case, 77)
    s = cases.inputs(case, 77)
    ref = orc.twodir(s["non"], s["H"].cpu().numpy(), s["mu"].cpu().numpy(), acc64=True)
    e, e_ref = rel(R, exact), rel(ref, exact)
    print(f"[basis] {e:.1e}, oracle {e_ref:.1e}", flush=True)
    assert e < 1.5 * e_ref
