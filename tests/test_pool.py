"""The rules of the allocation pool (csrc/pool.h) on the host: tests/c/pool_test.cpp compiles it against a runtime of its own and runs one case per process."""
import pathlib, subprocess
import pytest

ROOT = pathlib.Path(__file__).resolve().parent

@pytest.fixture(scope="module")
def program(tmp_path_factory):
  exe = tmp_path_factory.mktemp("pool") / "pool_test"
  r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", str(ROOT / "c" / "pool_test.cpp"), "-o", str(exe)], capture_output=True, text=True)
  assert r.returncode == 0, r.stderr
  return exe

@pytest.mark.parametrize("case", ["freed_twice", "waits_before_handing_out", "capture_opened_elsewhere", "capture_of_another_thread", "a_free_that_fails", "capture_of_its_own", "classes_hold_little_more", "no_host_memory", "full_of_other_blocks", "pinned_freed_in_a_capture", "pinned_of_someone_else"])
def test_pool(program, case):
  r = subprocess.run([str(program), case], capture_output=True, text=True, timeout=60)
  assert r.returncode == 0, r.stdout + r.stderr
