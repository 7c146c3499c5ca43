"""The rules by which the library chooses kernels, on the CPU: what they need is a matrix's format and sizes."""
import random

import pytest

FORMATS = ("B32S4", "B32S8", "Q_G_4", "Q_G_8", "Q_8", "Q_G_3", "Q_G_2", "SB256A3", "SB256A2", "Q_4", "Q_G_6")


@pytest.mark.parametrize("fmt", FORMATS)
def test_the_faster_plan_among_those_of_as_many_launches(rules, fmt):
    """What the host takes for a call is its launches' alone, so no plan of as many is faster on the GPU than the one that is taken,
    nor one of fewer: products of 5 to 300 rows of one matrix and of a pair, with any scratch, some and none."""
    rng = random.Random(FORMATS.index(fmt))
    for _ in range(400):
        N, K, M = rng.randint(64, 6144), 256 * rng.randint(1, 60), rng.randint(5, 300)
        for f32 in (False, True):
            for scratch in (rules.ANY, rng.randint(0, 1 << 22), 0):
                for matrices in (1, 2) if fmt not in ("Q_4", "Q_G_6") else (1,):
                    every, taken = rules.plans(fmt, N, K, f32, M, scratch, matrices)
                    fewer = [p for p in every if p.launches <= taken.launches]
                    assert min(p.us for p in fewer) == taken.us, (N, K, M, f32, scratch, matrices, taken.shape, taken.ksplit)


@pytest.mark.parametrize("fmt,N,K,f32,M,launches", [
    ("B32S8", 289, 3840, False, 29, 2),    # us a call, and in a graph: one launch 8.8 and 8.7, two 7.9 and 7.0
    ("Q_G_3", 444, 1792, True, 82, 2),     # 8.9 and 8.9, 8.4 and 8.0
    ("Q_G_2", 1472, 2560, False, 20, 2),   # 9.2 and 9.2, 7.9 and 7.4
    ("Q_4", 306, 2048, False, 71, 2),      # 9.0 and 9.0, 7.9 and 7.3
    ("Q_8", 256, 4096, False, 21, 2),      # 9.3 and 9.2, 8.0 and 6.8
    ("B32S4", 1075, 1792, True, 20, 1),    # 7.7 and 7.7, 8.1 and 6.8
    ("B32S4", 320, 1024, False, 20, 1),    # 5.2 and 5.1, 7.8 and 6.2
    ("SB256A2", 1536, 1792, False, 18, 1),  # 7.7 and 7.7, 7.7 and 7.3
])
def test_a_second_launch_where_it_saves_the_call_time(rules, fmt, N, K, f32, M, launches):
    """A second launch is taken where it makes the call shorter: two take the host 7.6 to 8.0 us."""
    assert rules.plans(fmt, N, K, f32, M)[1].launches == launches


@pytest.mark.parametrize("fmt,N,K,f32,B,tiles", [
    ("SB256A2", 1318, 2304, True, 5, True),    # us in a graph: decode kernels 10.1, integer tile kernel 7.3
    ("SB256A3", 1152, 1280, True, 8, True),    # 9.4, 7.1
    ("Q_G_3", 1088, 3840, False, 11, True),    # 9.4, 7.5
    ("Q_4", 1536, 1024, True, 8, True),        # 9.0, 6.6
    ("Q_G_3", 1466, 1536, True, 6, True),      # 8.2, 7.7
    ("Q_G_3", 1152, 1536, True, 7, True),      # 8.7, 7.3
    ("Q_G_2", 1216, 2304, False, 10, True),    # 8.2, 7.3
    ("B32S8", 512, 6400, True, 8, True),       # 9.4, 8.0
    ("B32S4", 1024, 8192, True, 7, True),      # 9.0, 7.8
    ("B32S4", 432, 8448, True, 7, False),      # 8.0, 8.9
    ("Q_8", 384, 8448, True, 7, False),        # 8.8, 9.4
    ("B32S4", 576, 8960, True, 5, False),      # 8.1, 9.0
    ("SB256A3", 14336, 4096, False, 8, False),  # 13, 18
    ("Q_G_4", 14336, 4096, True, 16, True),    # 25, 22
])
def test_five_to_sixteen_rows_by_the_gpu_time_of_both_kernels(rules, fmt, N, K, f32, B, tiles):
    """The decode kernels and the integer tile kernel are compared by their times on the GPU, whatever the launches: seen by the
    scratch that is asked for, which is what the kernel that serves uses."""
    need, decode = rules.rows_scratch(fmt, N, K, f32, B)
    plan = rules.plans(fmt, N, K, f32, B)[1]
    parts = 4 * plan.ksplit * B * N if plan.ksplit > 1 else 0
    assert parts != decode  # (else the scratch would not tell)
    assert need == (max(decode, parts) if tiles else decode)
