"""The library's host code (device bookkeeping, transfers, graphs, plans) on the
CPU, against a stand-in for the HIP runtime (fakehip/fakehip.c)."""
import pytest

from tests import fakehip


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return fakehip.compile_fake(tmp_path_factory.mktemp("fakehip"))


def test_read_backs_and_uploads_run_on_the_contexts_device(so):
    """Uploads and read-backs of a lattice of device 1 while device 0 is
    current: buffers, events and kernels are those of device 1, and device 0 is
    current again afterwards."""
    fakehip.run(so, """
        fake.hipSetDevice(1)
        made = [Lattice(12, 10, 8, ncomp=c, precision=p) for c in (2, 3) for p in (0, 1)]
        batch = Batch([(8, 6, 6), (6, 6, 6)], ncomp=3)
        fake.hipSetDevice(0)
        home = Lattice(12, 10, 8, ncomp=2)
        for g in [home] + made:
            g.upload_sites(np.zeros((10, 12, 14, g.site_doubles)))
            g.populations(), g.density(), g.momentum(), g.download_sites()
        batch.populations(1)
        d = ctypes.c_int(-1)
        fake.hipGetDevice(ctypes.byref(d))
        assert d.value == 0
        assert len(log()) > 10
    """)
