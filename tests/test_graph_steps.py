"""Decode steps per graph of a generate call (draco_graph_steps), on the CPU:
against the measured costs of a captured kernel (1.8 us) and of a graph launch
(what several steps a graph save per token), the choice is never far from the
best one, however short or long the generation."""
import ctypes as ct

import pytest

CAPTURE = 1.8                        # us a captured and instantiated kernel
SAVED = {1: 0.0, 4: 5.0, 16: 6.5}    # us a token


def _steps(hip, nodes, n_gen, prompt):
    f = hip._Z17draco_graph_stepsiib
    f.restype, f.argtypes = ct.c_int, [ct.c_int, ct.c_int, ct.c_bool]
    return f(nodes, n_gen, prompt)


def _cost(nodes, n_gen, s):
    tokens = n_gen - n_gen % s if s > 1 else 0
    return (CAPTURE * nodes * s if s > 1 else 0.0) - SAVED[s] * tokens


@pytest.mark.parametrize("nodes", [8, 14, 26, 60, 98, 128])
def test_steps_cost_no_more_than_the_best_choice(hip, nodes):
    for n_gen in list(range(1, 40)) + [64, 100, 150, 200, 256, 400, 512, 1024, 2048, 4096]:
        s = _steps(hip, nodes, n_gen, False)
        assert s in SAVED and s <= max(n_gen, 1)
        best = min(_cost(nodes, n_gen, k) for k in SAVED if k <= n_gen)
        # slack: 40 us and one percent of the smallest step (45 us) a token
        assert _cost(nodes, n_gen, s) <= best + 40 + 0.5 * n_gen, (n_gen, s)


def test_steps_of_many_kernels_and_behind_a_prompt(hip):
    assert [_steps(hip, 130, n, p) for n in (4, 64, 100000) for p in (False, True)] == [1] * 6
    assert [_steps(hip, 98, n, True) for n in (1, 8, 15, 16, 32, 200)] == [1, 1, 1, 4, 4, 4]
    assert [_steps(hip, 98, n, False) for n in (1, 4, 16, 64, 146)] == [1] * 5
