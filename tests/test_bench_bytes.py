"""The benchmark charges each kernel class with the bytes of the sequence that has run, which the FFT
launches per step tell, and refuses launches of any other."""
import pytest

import bench
import crava_amd as C

W = dict(nxp=576, nyp=576, nzp=320)
G, NR = 289 * 576 * 320 * 8, 576 * 576 * 320 * 4


def _launches(x, y, z):
    return {C.K_FFT_X: x, C.K_FFT_Y: y, C.K_FFT_Z: z}


@pytest.mark.parametrize("R", [0, 1, 2])
def test_bytes_follow_the_launches(R):
    n, B = 11 + 3 * R, 128 * 289 * 576 * 8
    band = bench.kernel_bytes(W, 5, R, 128, _launches(n, n, 11))
    assert band[C.K_FFT_Z] == 8 * (NR + B) + 3 * (B + 2 * NR)
    assert band[C.K_FFT_Y] == 22 * B + 6 * R * G and band[C.K_POSTERIOR] == 11 * B + 6 * G
    split = bench.kernel_bytes(W, 5, R, 128, _launches(n, n, 0))
    assert split[C.K_FFT_Z] == 0 and split[C.K_FFT_X] == n * (NR + G) and split[C.K_POSTERIOR] == 17 * G
    for bad in (_launches(n, n, 12), _launches(n, n, 5), _launches(4, 4, 4)):
        with pytest.raises(ValueError):
            bench.kernel_bytes(W, 5, R, 128, bad)
