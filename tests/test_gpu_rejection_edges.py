"""The rejection structure's direct fill and the sectioned draws at their
edges: runs that begin and end around a wave's 64 slots, neighbouring runs
long enough to be cut into tasks, shares of a section's samples smaller than a
wave."""
import numpy as np
import pytest

import atg
from test_gpu_rejection_fill import bits, expected_accept

pytestmark = pytest.mark.gpu


def spikes(n, at):
    w = np.full(n, 1e-9)
    w[at] = 1.0
    return w


CASES = {
    "one_slot_each_63": lambda: np.full(63, 1.0 - 1e-12) + np.arange(63) * 1e-14,
    "uniform_64": lambda: np.linspace(0.5, 1.5, 64),
    "uniform_65": lambda: np.linspace(0.5, 1.5, 65),
    "wave_and_one": lambda: np.linspace(0.1, 1.9, 1025),
    "block_and_one": lambda: np.linspace(1.9, 0.1, 4097),
    "runs_of_64": lambda: spikes(640, np.arange(0, 640, 64)),
    "runs_of_63_and_65": lambda: spikes(640, np.array([0, 63, 64, 127, 128, 191, 639])),
    "tasks_in_one_round": lambda: spikes(20_000, np.array([100, 101, 102, 120, 127, 128])),
    "tasks_at_both_ends": lambda: spikes(20_000, np.array([0, 1023, 1024, 19_999])),
    "one_run": lambda: spikes(9_000, np.array([8_999])),
}


@pytest.mark.parametrize("case", list(CASES))
def test_edges_match_oracle(gpu, oracle, case):
    torch = gpu
    w = CASES[case]()
    t = atg.Table(len(w))
    t.set_weights(w)
    t.rejection_build()
    W = t.rejection_weight_sum()
    incl, A = oracle.rejection_build(w, W)
    np.testing.assert_array_equal(t.rejection_array(), A)
    assert np.array_equal(bits(t.rejection_accept()), bits(expected_accept(w, W, incl)))
    for count in (1, 16, 17, 1023, 1025, 40_000):
        out = torch.full((count,), -1, dtype=torch.int32, device="cuda")
        t.rejection_sample_sectioned(count, seed=count, section_slots=1024, out=out)
        exp = oracle.sample_rejection_sectioned(A, w, W, 1024, count, count)
        np.testing.assert_array_equal(out.cpu().numpy(), exp, err_msg=f"count={count}")


def test_items_whose_count_overflows_have_no_slots(gpu):
    # N w is infinite for three items (W is not): the others keep theirs.
    n, big = 5000, [100, 127, 1500]
    w = np.ones(n)
    w[big] = 5e304
    t = atg.Table(n)
    t.set_weights(w)
    t.rejection_build()
    np.testing.assert_array_equal(t.rejection_array(), np.delete(np.arange(n), big))
