"""How a training step's next samples are split over the workgroups of its last launch (no GPU)."""
import ctypes as C
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SUM_BLOCKS = (4481 + 31) // 32 + 1  # the sum's workgroups: 32 of 4,481 columns each, and the losses'


@pytest.mark.parametrize("cus", [32, 64, 128, SUM_BLOCKS, SUM_BLOCKS + 1, 160, 256, 304])
def test_samples_fill_the_compute_units_that_the_sum_leaves(cus):
    """A batch that fits the idle CUs at 1,024 samples each is spread over all of them in whole waves;
    any other, and every one where the sum leaves no CU, takes 640 a workgroup."""
    gen_per = C.CDLL(os.path.join(ROOT, "radrhd_solver_amd", "librhllc_hip.so"))["_ZN9rhllc_mlp7gen_perEii"]
    gen_per.restype, gen_per.argtypes = C.c_int, [C.c_int, C.c_int]
    idle = cus - SUM_BLOCKS
    for n in (256, 1024, 7168, 7424, 65536, 116736, 116992, 1 << 20):
        per = gen_per(n, cus)
        if idle > 0 and n <= 1024 * idle:
            assert per % 64 == 0 and per <= 1024
            assert -(-n // per) <= idle and (per == 64 or -(-n // (per - 64)) > idle)
        else:
            assert per == 640
