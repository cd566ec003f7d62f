"""The dense-propagator kernel (one wave per vector, exact exponential) at
the edges of its row and column classes, against the oracle: site counts on
both sides of every class boundary, windows of one and two steps, one sample
and a sample count that leaves no full workgroup pattern.  Tolerance 1e-5
relative L2 as for every exact-exponential result (FP32 state, FP64
exponential)."""
import numpy as np
import pytest

from nise_2017_amd import abi

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
