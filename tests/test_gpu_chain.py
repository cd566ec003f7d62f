"""Nearest-neighbour chains: the systolic kernels (chain.hip) against the row
conveyor with one row, whose operations they run in the same order."""
import numpy as np
import pytest

from nise_2017_amd import abi, synth

pytestmark = pytest.mark.gpu


def chain_case(N, T, ns, sr, ts=1, begin=0, seed=900):
    """Nearest-neighbour couplings; from N = 6 on one of them absent."""
    H, mu = synth.chain_absorption(N=N, nframes=(ns - 1) * sr + begin * sr + T + 2, seed=seed + N)
    if N >= 6:
        H[:, 1 + 2 * N] = 0  # pair (2, 3) of the upper triangle
    lo, hi = synth.shifted_center(H, N)
    non = abi.make_non(singles=N, tmax1=T, sample=sr, begin=begin, end=begin + ns, ts=ts, propagation=1, deltat=2.0,
                       min1=lo, max1=hi)
    non.shifte = np.float32((np.float32(hi) + np.float32(lo)) / np.float32(2))
    return non, H, mu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)


# one sample and many, remainders of 12, 6 and 3 vectors per wave, T below, at
# and above the lanes per vector, substeps, gaps between samples
@pytest.mark.parametrize("N,T,ns,sr,ts,begin", [
    (2, 1, 1, 1, 1, 0), (2, 40, 5, 3, 1, 0), (3, 2, 3, 1, 1, 1), (6, 23, 7, 30, 1, 0), (11, 64, 9, 4, 2, 0),
    (20, 21, 5, 6, 1, 0), (21, 22, 11, 2, 3, 0), (42, 43, 5, 3, 1, 2), (43, 65, 4, 9, 1, 0), (64, 30, 90, 5, 1, 0),
    (128, 48, 3, 7, 2, 0), (200, 44, 2, 3, 1, 0)])
def test_chain_kernels_against_row_conveyor(N, T, ns, sr, ts, begin):
    """Forward bit for bit, also on graph replays; the gradient to 1e-5 (the
    conveyor adds each frame's terms of a site over the vectors in FP32)."""
    non, H, mu = chain_case(N, T, ns, sr, ts, begin)
    print(f"[chain] N={N} T={T} ns={ns} every {sr} ts={ts}", flush=True)
    rng = np.random.default_rng(5)
    g_re, g_im = (rng.standard_normal(T).astype(np.float32) for _ in range(2))
    delta = rng.standard_normal(N).astype(np.float32)
    p = abi.AbsPlan(non, H, H.shape[1], mu, mu.shape[1], H.shape[0])
    try:
        plain = p.execute()
        graph = [p.execute(flags=2) for _ in range(3)]
        p.enable_adjoint(5)
        p.set_params(delta, 0.9)
        fwd = p.execute()
        gd, gc = p.adjoint(g_re, g_im)
        p.set_rows(1)
        p.set_params(delta, 0.9)
        rfwd = p.execute()
        if N > 155:  # one row's adjoint does not fit the LDS
            p.set_rows(2)
            p.execute()
        rd, rc = p.adjoint(g_re, g_im)
        p.set_rows(1)
        p.set_params()
        rplain = p.execute()
    finally:
        p.close()
    for a in (plain, *graph):
        assert np.array_equal(a[0], rplain[0]) and np.array_equal(a[1], rplain[1])
    assert np.array_equal(fwd[0], rfwd[0]) and np.array_equal(fwd[1], rfwd[1])
    assert rel(np.append(gd, gc), np.append(rd, rc)) < 1e-5


@pytest.mark.parametrize("N,T,ns,sr", [(9, 40, 30, 3), (50, 300, 60, 40), (100, 64, 400, 30)])
def test_chain_batch_and_noalloc_match_plan(N, T, ns, sr):
    """The batch of systems (beside a system that is no chain) and the run in
    the fixed array, in one window or several: bit for bit the plan's result."""
    import ctypes as C

    import torch

    from test_gpu_multi import system
    non, H, mu = chain_case(N, T, ns, sr)
    print(f"[chain] batch, noalloc: N={N} T={T} ns={ns} every {sr}", flush=True)
    Hd, mud = torch.from_numpy(H).cuda(), torch.from_numpy(mu).cuda()
    torch.cuda.synchronize()
    p = abi.AbsPlan(non, Hd, H.shape[1], mud, mu.shape[1], H.shape[0], where=abi.NISE_DEVICE)
    re, im = p.execute()
    p.close()
    r1, i1 = np.zeros(T, np.float32), np.zeros(T, np.float32)
    abi.check(abi.lib().nise_absorption_batched_noalloc(C.byref(non), abi.ptr(Hd), H.shape[1], abi.ptr(mud), mu.shape[1],
                                                        H.shape[0], None, r1, i1))
    assert np.array_equal(re, r1) and np.array_equal(im, i1)
    out, done = abi.absorption_multi([(non, H, mu, None), system(23, 1, 3), (non, H, mu, None)])
    for k in (0, 2):
        assert np.array_equal(re, out[k][0]) and np.array_equal(im, out[k][1])
    assert np.all(done > 0)


def test_batch_runs_its_chains_together():
    """Equal chains of a batch share one launch: they end at about the same
    time.  One after the other, the last of 24 would end 24 times as late as the
    first."""
    case = chain_case(64, 200, 60, 10)
    system = (*case, None)
    print("[chain] 24 equal chains", flush=True)
    abi.absorption_multi([system] * 24)
    out, done = abi.absorption_multi([system] * 24)
    assert max(done) < 4 * min(done), done
    for re, im in out:
        assert np.array_equal(re, out[0][0]) and np.array_equal(im, out[0][1])


def test_batch_of_uneven_chains_matches_plans():
    """Chains of every lanes-per-vector count, with substeps, beside a lattice
    and an exact-exponential system: bit for bit their plans' results."""
    from test_gpu_multi import system
    cases = [chain_case(N, T, ns, sr, ts, begin)
             for N, T, ns, sr, ts, begin in [(3, 17, 4, 2, 1, 0), (9, 40, 30, 3, 2, 1), (21, 33, 5, 7, 1, 0),
                                             (70, 50, 12, 4, 3, 2), (130, 24, 3, 30, 1, 0), (2, 1, 1, 1, 1, 0)]]
    batch = [(*c, None) for c in cases] + [system(23, 1, 3), system(20, 0, 4)]
    print("[chain] uneven batch", flush=True)
    out, done = abi.absorption_multi(batch)
    for (non, H, mu), (re, im) in zip(cases, out):
        p = abi.AbsPlan(non, H, H.shape[1], mu, mu.shape[1], H.shape[0])
        r, i = p.execute()
        p.close()
        assert np.array_equal(re, r) and np.array_equal(im, i), non.singles
    assert np.all(done > 0)


def test_chain_plan_holds_only_its_own_tables():
    """A chain plan's device memory is its records (32 bytes per site and frame)
    and the partial sums; the conveyor's tables come when the plan leaves the
    chain kernels."""
    import torch
    N, T, ns, sr = 100, 64, 3000, 4
    non, H, mu = chain_case(N, T, ns, sr)
    Hd, mud = torch.from_numpy(H).cuda(), torch.from_numpy(mu).cuda()
    torch.cuda.synchronize()
    abi.AbsPlan(non, Hd, H.shape[1], mud, mu.shape[1], H.shape[0], where=abi.NISE_DEVICE).close()
    free = torch.cuda.mem_get_info()[0]
    p = abi.AbsPlan(non, Hd, H.shape[1], mud, mu.shape[1], H.shape[0], where=abi.NISE_DEVICE)
    try:
        chain = p.execute()
        used = free - torch.cuda.mem_get_info()[0]
        frames = (ns - 1) * sr + T
        rec, partial, tables = 32 * N * frames, 3 * ns * T * 16, 16 * N * frames
        print(f"[chain] plan of {rec >> 20} + {partial >> 20} MiB holds {used >> 20}", flush=True)
        assert used < rec + partial + tables // 2
        p.set_rows(0)
        rows = p.execute()
        assert np.array_equal(chain[0], rows[0]) and np.array_equal(chain[1], rows[1])
        p.set_shape(16, 5)
        slots = p.execute()
        assert rel(slots[0] + 1j * slots[1], rows[0] + 1j * rows[1]) < 1e-6
    finally:
        p.close()
