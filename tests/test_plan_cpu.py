"""The forward's choice of kernel (csrc/tfgfa_plan.h), on the CPU: the shapes that the GPU tests name
reach the kernels they name, and the choice stays with the measured times."""
import pytest

from custom_flash_attn import _C

import test_gpu_plans as shapes

CUS = 256


def _plan(heads, Nq, Nk, D, causal):
    return _C.fwd_plan(heads, CUS, Nq, Nk, D, causal)


@pytest.mark.parametrize("D,plans", [(8, shapes.NARROW_PLANS), (64, shapes.NARROW_PLANS),
                                     (72, shapes.WIDE_PLANS), (128, shapes.WIDE_PLANS)])
def test_shapes_of_the_gpu_tests_reach_their_kernels(D, plans):
    for plan, group in plans.items():
        for B, H, Nq, Nk, causal in group:
            assert _plan(B * H, Nq, Nk, D, causal) == plan, (H, Nq, Nk, causal)
    assert set(plans) == {"kWhole", "kHalves", "kGroups2", "kPairs"} | ({"kGroups4"} if D <= 64 else set())


# (head dim, heads, N_q, N_k, causal): us of each kernel, bf16, in graph replays on 256 CUs.  Problems on
# which a rule by the causal flag and the longest chain alone took up to 1.6 times the faster of the
# whole-block and split-key kernels.
MEASURED = {
    (64, 192, 128, 128, True): dict(kWhole=5.6, kHalves=6.5, kGroups2=6.1, kPairs=5.9, kGroups4=8.7),
    (64, 32, 768, 192, True): dict(kWhole=6.2, kHalves=7.2, kGroups2=7.3, kPairs=7.6, kGroups4=10.3),
    (64, 12, 4096, 2048, True): dict(kWhole=28.6, kHalves=41.5, kGroups2=34.3, kPairs=30.6, kGroups4=34.0),
    (64, 29, 1408, 704, True): dict(kWhole=13.5, kHalves=20.9, kGroups2=17.9, kPairs=15.9, kGroups4=22.1),
    (64, 37, 448, 448, True): dict(kWhole=8.3, kHalves=6.7, kGroups2=8.2, kPairs=7.2, kGroups4=8.7),
    (64, 8, 2048, 2048, True): dict(kWhole=24.7, kHalves=15.8, kGroups2=20.7, kPairs=16.0, kGroups4=13.9),
    (64, 12, 2048, 2048, True): dict(kWhole=24.6, kHalves=18.5, kGroups2=20.7, kPairs=16.5, kGroups4=15.6),
    (64, 21, 1152, 1152, True): dict(kWhole=16.2, kHalves=14.4, kGroups2=14.0, kPairs=11.7, kGroups4=13.4),
    (64, 20, 2048, 2048, True): dict(kWhole=25.4, kHalves=26.7, kGroups2=21.0, kPairs=18.4, kGroups4=24.6),
    (64, 16, 1280, 352, False): dict(kWhole=7.8, kHalves=10.1, kGroups2=8.3, kPairs=8.2, kGroups4=12.0),
    (64, 16, 2048, 1312, False): dict(kWhole=17.6, kHalves=26.4, kGroups2=16.1, kPairs=17.0, kGroups4=20.8),
    (128, 8, 2176, 704, False): dict(kWhole=15.7, kHalves=32.1, kGroups2=16.0, kPairs=24.5),
    (128, 16, 1536, 1152, False): dict(kWhole=22.5, kHalves=44.3, kGroups2=21.3, kPairs=31.5),
    (128, 75, 249, 811, False): dict(kWhole=20.1, kHalves=49.1, kGroups2=19.9, kPairs=34.4),
    (96, 160, 83, 1113, False): dict(kWhole=24.6, kHalves=33.4, kGroups2=20.9, kPairs=33.1),
    (80, 40, 287, 46, False): dict(kWhole=5.5, kHalves=9.0, kGroups2=6.7, kPairs=6.3),
    (128, 21, 1152, 1152, True): dict(kWhole=24.9, kHalves=32.8, kGroups2=22.5, kPairs=22.5),
    (128, 12, 1312, 1312, True): dict(kWhole=24.8, kHalves=22.5, kGroups2=22.4, kPairs=18.7),
    (128, 18, 448, 448, True): dict(kWhole=12.0, kHalves=9.5, kGroups2=12.2, kPairs=11.3),
}


@pytest.mark.parametrize("problem", MEASURED, ids=str)
def test_choice_is_within_a_few_percent_of_the_fastest(problem):
    """Within 1.05 of the best kernel's time: twice what repeated runs differ by."""
    D, heads, Nq, Nk, causal = problem
    times = MEASURED[problem]
    assert times[_plan(heads, Nq, Nk, D, causal)] <= 1.05 * min(times.values())


@pytest.mark.parametrize("cus", [64, 228, 256, 304])
def test_choice_is_compiled_for_its_head_dim(cus):
    """Every size gets a kernel that its head dim has: key groups of four up to 64 dims only."""
    for D in (8, 64, 72, 128):
        for heads in (1, 5, 16, 100, 300, 1 << 20):
            for Nq in (1, 33, 129, 700, 4096):
                for Nk in (1, 65, 900, 4096):
                    for causal in (False, True):
                        plan = _C.fwd_plan(heads, cus, Nq, Nk, D, causal)
                        assert plan != "kGroups4" or D <= 64
