"""The relay-matrix builder where few tiles give grid points and image slices
workgroups of their own: one tile, one past a tile, the first sizes of each
form, with and without a long image list, every grid point through
alpha_SCS."""
import numpy as np
import pytest

from mbd_amd import engine, generators, io
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,box", [(5, 8.0), (17, 9.0), (112, 13.0), (113, 13.0), (130, 14.0),
                                   (17, None), (113, None)])
def test_few_tiles(n, box):
    if box:
        geo, st = generators.random_periodic(n, box, seed=n)
        st.mbd_scs_dip_cutoff = 3.0 * box - 0.5  # 7 x 7 x 7 images
    else:
        geo, st = generators.chain_molecule(np.random.default_rng(n), n - 2), io.Settings()
    xyz, lat = geo.to_bohr()
    sy = O.system_from(geo.names, xyz, geo.hirshfeld, lat, geo.periodic, st)
    with engine.MbdEngine(0) as eng:
        eng.set_geometry(geo, st)
        for k in (0, 20):
            want = O.relay_matrix(sy, k)
            assert np.allclose(eng.relay_matrix(k), want, rtol=1e-12, atol=1e-14 * np.abs(want).max())
            got = eng.relay_matrix(k, mode="mixed")
            assert np.allclose(got, want, rtol=2e-6, atol=2e-7 * np.abs(want).max())
        a, pol, _, c6, _, d = eng.scs("fp64")
    wa, wpol, wc6, _, info = O.scs_all(sy)
    assert d["info_scs"] == info == 0
    # condition numbers below 1e3 over entries right to 1e-13
    assert np.allclose(a, wa, rtol=1e-10, atol=0) and np.allclose(pol, wpol, rtol=1e-10, atol=0)
    assert np.allclose(c6, wc6, rtol=2e-10, atol=0)
