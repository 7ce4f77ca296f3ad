"""Host functions called from several threads, each with its own array."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_host_functions_from_several_threads():
    # lattices of several sizes and forms (a wave per quadrant, quadrants, tiles): every call has its own
    # workspace, so each thread gets the numbers it gets alone
    import flue_lat_amd as FL
    fc = FL.compiled.flue_c
    dims = [(4, 4, 4, 4), (10, 9, 11, 13), (2, 16, 16, 16), (5, 25, 27, 29)]
    arrays = [np.asfortranarray(FL.GaugeField.random(d, 40 + c, 0.4).to_complex().cpu().numpy())
              for c, d in enumerate(dims)]

    def measure(U):
        return (fc.magnetic_c(U), fc.plaquette_c(U, 1, 4, 4)[0], fc.wmunu_c(U, 2, 3, 2, 1),
                fc.plaquette_c(U, 2, 4, 4)[0])

    alone = [measure(U) for U in arrays]
    got = [[] for _ in arrays]

    def work(c):
        for _ in range(6):
            got[c].append(measure(arrays[c]))

    threads = [threading.Thread(target=work, args=(c,)) for c in range(len(arrays))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for c in range(len(arrays)):
        assert got[c] == [alone[c]] * 6, dims[c]
