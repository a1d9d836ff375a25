"""The library short of device memory (memory_scenarios.py): what it takes for itself gives way, what
does without it goes on without it, and what fails leaves nothing that a step could read."""
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

HERE = Path(__file__).resolve().parent


@pytest.mark.parametrize("name", ["labels_cut_short", "sets_do_not_fit", "sets_take_back", "others_give_way",
                                  "epsilon_on_the_host", "position_gradient_on_the_host",
                                  "force_set_again", "labels_set_again", "short_runs_step_singly",
                                  "current_device_stays", "run_from_another_device",
                                  "kept_memory_is_bounded", "gradient_cut_short",
                                  "launch_errors_are_reported", "second_array_refused",
                                  "threads_short_of_memory"])
def test_scenario(name):
    assert (HERE / "cpp" / "_build" / "alloc_limit.so").exists(), "build it with __graft_entry__.build()"
    print(f"[memory] {name}", flush=True)
    r = subprocess.run([sys.executable, "-u", str(HERE / "memory_scenarios.py"), name], capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and f"done {name}" in r.stdout, r.stdout + r.stderr
