"""The launch-shape tuner on the CPU, against an evaluator that reports a kernel
and a table of times: the waves are left at the widest where the kernel that
runs has workgroups of its own, whatever the noise, and chosen by time where
the segment kernel runs."""
import pytest

from acehip import autotune

NOISE = {4: 0.95, 8: 1.0, 16: 1.02}  # the narrowest looks 7 % faster


class _Ev:
    npool, nAA, nA = 100, 10, 10

    def __init__(self, kernel_of, time_of):
        self.kernel_of, self.time_of = kernel_of, time_of
        self.W, self.P, self.seen = 8, 0, []

    def set_tile(self, W):
        self.W = W

    def set_parts(self, P):
        self.P = P

    def set_pool_shape(self, ch, epw):
        pass

    def last_dag_shape(self):
        return 1, 0, 0

    def last_dag_kernel(self):
        return self.kernel_of(self.P)

    def energy_forces(self, b):
        self.seen.append((self.W, self.P))


@pytest.fixture
def tuned(monkeypatch):
    monkeypatch.setattr(autotune, "_CACHE", {})
    monkeypatch.setattr(autotune, "tune_pool", lambda *a: ((16, 0), {}))
    monkeypatch.setattr(autotune.torch.cuda, "synchronize", lambda: None)

    def run(kernel_of, time_of):
        ev = _Ev(kernel_of, time_of)
        monkeypatch.setattr(autotune, "_time_call", lambda fn, reps: (fn(), time_of(ev.W, ev.P))[1])
        (W, P), results, _ = autotune.tune(ev, type("B", (), {"nenv": 5})())
        assert (ev.W, ev.P) == (W, P)
        return W, P, results

    return run


def test_pair_kernel_keeps_the_widest(tuned):
    W, P, results = tuned(lambda P: "pairs", lambda W, P: NOISE[W] * {0: 1.0, 1: 0.95, 2: 1.1, 3: 1.2, 4: 1.3}[P])
    assert (W, P) == (16, 1) and {w for w, _ in results} == {16}


def test_pair_kernel_takes_the_fastest_parts(tuned):
    W, P, _ = tuned(lambda P: "pairs", lambda W, P: {0: 1.009, 1: 1.0, 2: 1.02, 3: 1.1, 4: 1.2}[P])
    assert (W, P) == (16, 1)


def test_slot_kernel_keeps_its_own_parts(tuned):
    # parts that the caller sets are the segment kernel's, slower here
    W, P, results = tuned(lambda P: "slots" if P == 0 else "segments", lambda W, P: NOISE[W] * (1.0 if P == 0 else 1.5))
    assert (W, P) == (16, 0) and (4, 0) not in results and (4, 2) in results


def test_segment_kernel_by_time(tuned):
    W, P, results = tuned(lambda P: "segments", lambda W, P: {4: 1.0, 8: 0.9, 16: 1.1}[W] * (1.0 if P == 2 else 1.05))
    assert (W, P) == (8, 2) and len(results) == 15


def test_segment_kernel_keeps_the_librarys_choice_within_one_percent(tuned):
    W, P, _ = tuned(lambda P: "segments", lambda W, P: 1.009 if (W, P) == (16, 0) else 1.0)
    assert (W, P) == (16, 0)
