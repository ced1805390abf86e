"""make_macrhs and make_s0mac where their chunks of planes and blocks of
threads depend on the domain: one plane a chunk, two from profiles in memory,
several from profiles in LDS or too long for it, the last chunk short; chunks of
16 planes in blocks of 512 and 1024 threads.  Bit for bit against the oracle."""
import pytest

from . import test_gpu_inputs_profiles as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,box,bins,interp,dpdt", [
    ((15, 10, 20), 5, 5, 3, 0.5),        # one plane
    ((90, 90, 90), 9, 5, 3, 0.5),        # two planes, profiles in memory: 2, 2, 2, 2, 1
    ((108, 108, 108), 9, 5, 2, -1.0),    # two planes, profiles in LDS
    ((150, 150, 150), 10, 5, 3, 0.5),    # four: 4, 4, 2
    ((150, 150, 150), 10, 20, 3, 0.5),   # the same, profiles too long for LDS
])
def test_macrhs_chunks(gpu, oracle_lib, n, box, bins, interp, dpdt):
    T.test_macrhs_profiles_bitwise(gpu, oracle_lib, n, box, bins, interp, dpdt, "normal")


@pytest.mark.parametrize("n,box,bins,interp", [
    ((10, 15, 20), 5, 5, 3),      # one plane
    ((60, 60, 60), 20, 5, 2),     # two, the last chunk one
    ((90, 60, 60), 10, 5, 3),     # six, six, one
    ((160, 160, 160), 40, 2, 3),  # 16, blocks of 1024: 16, 16, 11
    ((160, 160, 160), 20, 2, 3),  # the same planes, blocks of 512
])
def test_s0mac_chunks(gpu, oracle_lib, n, box, bins, interp):
    T.test_s0mac_profiles_bitwise(gpu, oracle_lib, n, box, bins, interp, "normal")
