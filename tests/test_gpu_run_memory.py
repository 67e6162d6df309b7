"""A run or batch that is closed gives its pinned host arrays back: the process holds as many mappings
after forty as after four."""
import pytest

from spheral_amd import abi

pytestmark = pytest.mark.gpu


def mappings():
    with open("/proc/self/maps") as f:
        return sum(1 for _ in f)


def test_closed_runs_leave_no_mappings(gpu):
    cfg = abi.default_config(2)
    held = []
    for count in (4, 36):
        print(f"[case] {count} runs", flush=True)
        for _ in range(count):
            gpu.Run(cfg, 64).close()
        held.append(mappings())
    assert held[1] - held[0] < 36            # less than one per run
