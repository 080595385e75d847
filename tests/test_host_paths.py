"""Host paths of libpbf.so that a GPU run reaches only when something fails or
would fault when it is wrong: tests/cpp/pbf_host_paths.cpp runs the built library
on a HIP runtime of its own (device memory is host memory, kernels do not run)
and checks every pointer that a launch or a copy hands over. No GPU needed."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
BUILD = ROOT / "physika-old_amd" / "_build"
CLANGXX = "/opt/rocm/llvm/bin/clang++"


@pytest.fixture(scope="module")
def host_paths(tmp_path_factory):
    if not shutil.which(CLANGXX):
        pytest.skip("clang++ not available")
    if not (BUILD / "libpbf.so").exists():
        pytest.skip("libpbf.so not built")
    exe = tmp_path_factory.mktemp("host_paths") / "pbf_host_paths"
    subprocess.run([CLANGXX, "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", str(ROOT / "tests" / "cpp" / "pbf_host_paths.cpp"), "-rdynamic",
                    f"-L{BUILD}", "-lpbf", f"-Wl,-rpath,{BUILD}", "-Wl,-rpath-link,/opt/rocm/lib", "-o", str(exe)],
                   check=True)
    return exe


def run(exe, scenario):
    r = subprocess.run([str(exe), scenario], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "VIOLATION" not in r.stdout, (r.returncode, (r.stdout + r.stderr)[-3000:])


def test_failed_list_reservation(host_paths):
    """Each allocation of a growing context fails once: the calls after it run
    without lists (bit masks, re-tests), and no kernel is handed a null list,
    whose first chunks a lane pair reads ahead of the wave's words."""
    run(host_paths, "list_reservation")


def test_failed_tape_slots(host_paths):
    """Each allocation of a rollout and its reverse fails once, in both
    precisions: a slot that got only some of its arrays is not used, neither by
    a reverse that is tried again nor by the next forward, which records into
    the slots."""
    run(host_paths, "tape_slots")


@pytest.mark.parametrize("scenario", ["last_search", "failed_rollout"])
def test_lists_of_the_last_search(host_paths, scenario):
    """step_neighbors exports the last search, whole and from one set of arrays:
    a recorded forward's last step, also after a call was captured and not yet
    replayed; and none, or whole ones, after a rollout call that failed midway."""
    run(host_paths, scenario)


def test_row_starts_are_there_when_the_export_returns(host_paths):
    """A second export of one search takes the row starts counted by the first;
    the caller's copy of them is waited for all the same."""
    run(host_paths, "blocking_export")


def test_viscosity_weights(host_paths):
    """The weights kept over a viscosity solve: up to 192 MiB and no more, reserved by
    pbf_reserve and pbf_set_params, and not asked for in every step once an
    allocation has failed."""
    run(host_paths, "viscosity_weights")


def test_pass_block_that_the_caller_sets(host_paths):
    """pbf_tuning.pass_block is what the PBD passes run, lane pairs included; only the
    default settings leave it to the library (64 for lane pairs)."""
    run(host_paths, "pass_blocks")


def test_forward_without_a_reverse_records_nothing(host_paths):
    """With pbf_rollout_record off a forward records no step, whatever reverses ran
    before; its lists are exported and a reverse still follows it."""
    run(host_paths, "unrecorded_forward")


def test_unknown_capture_state(host_paths):
    """Where HIP cannot say whether the call's stream is being captured, the context is
    not taken for a captured one for good (it would never record again)."""
    run(host_paths, "unknown_capture")


def test_replayed_frames_of_a_scene_that_turns_uneven(host_paths):
    """A graph captured while the scene was even is captured again once it is uneven:
    its frames then choose the block order by the counts, as the others do."""
    run(host_paths, "replays_of_uneven_scenes")
