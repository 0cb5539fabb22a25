"""Host side of a march (``csrc/march_launch.h``) compiled against a model of the HIP
runtime with two devices (``fake_hip/``): the device a march belongs to, the order of
marches, and the status when the device cannot hold one."""

import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "prince_amd", "csrc")

SOURCE = r"""
#include "march_launch.h"
namespace prh_internal {
int32_t error(const std::string&) { return 1; }
int32_t check(hipError_t e, const char*) { return e == hipSuccess ? 0 : 1; }
}
static FakeStream streams[2] = {{0}, {1}};
static int kernel;
// stream: 0, 1, or -1 for the null stream
extern "C" int launch(int stream, unsigned blocks, unsigned lds) {
  uint32_t sync = 0;
  prh_internal::MarchLaunch m{&kernel, &kernel, &kernel, blocks, 1024, lds, &sync, &kernel};
  return prh_internal::launch_march(m, stream < 0 ? nullptr : &streams[stream]);
}
extern "C" void set_current(int d) { fake::current = d; }
extern "C" int current() { return fake::current; }
extern "C" int pending() { return fake::last; }
extern "C" void device(unsigned max_blocks, int lds_max, int per_cu, int coop) {
  fake::max_blocks = max_blocks;
  fake::lds_max = lds_max;
  fake::per_cu = per_cu;
  fake::coop = coop;
}
extern "C" const char* calls() {
  static std::string s;
  s = fake::log;
  fake::log.clear();
  return s.c_str();
}
"""


@pytest.fixture()
def lib(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    (tmp_path / "launch.cpp").write_text(SOURCE)
    so = str(tmp_path / "launch.so")
    subprocess.run([cxx, "-std=c++17", "-shared", "-fPIC", "-fno-gnu-unique", "-I" + CSRC,
                    "-I" + os.path.join(HERE, "fake_hip"), "-o", so, str(tmp_path / "launch.cpp")],
                   check=True)
    lib = ctypes.CDLL(so)
    lib.calls.restype = ctypes.c_char_p
    return lib


LDS = 160 * 1024 - 64


def test_a_march_belongs_to_its_streams_device(lib):
    lib.set_current(0)
    for stream, device in ((1, 1), (0, 0), (-1, 0)):
        assert lib.launch(stream, 256, LDS) == 0
        assert lib.current() == 0
        assert f"march{device} " in lib.calls().decode()
    lib.set_current(1)
    assert lib.launch(0, 256, LDS) == 0 and lib.current() == 1
    assert lib.calls().decode().split() == ["wait0", "kernel0", "march0", "kernel0", "record0"]


def test_marches_of_one_device_follow_each_other(lib):
    lib.set_current(0)
    for stream in (0, 1, -1, 1):
        assert lib.launch(stream, 256, LDS) == 0
    got = [c for c in lib.calls().decode().split() if not c.startswith("kernel")]
    assert got == ["march0", "record0", "march1", "record1", "wait0", "march0", "record0",
                   "wait1", "march1", "record1"]


@pytest.mark.parametrize("blocks,device", [
    (257, (256, 163840, 1, 1)),   # more workgroups than the chip holds
    (256, (256, 163840, 0, 1)),   # none fits a CU
    (256, (256, 65536, 1, 1)),    # less LDS
    (256, (256, 163840, 1, 0)),   # no cooperative launches
    (256, (128, 163840, 1, 1)),   # refused by the launch itself
])
def test_a_march_that_does_not_fit_steps_aside_without_an_error(lib, blocks, device):
    lib.device(*device)
    assert lib.launch(0, blocks, LDS) == 2
    assert lib.pending() == 0
    assert "march" not in lib.calls().decode()
    lib.device(256, 163840, 1, 1)
    assert lib.launch(0, 256, LDS) == 0
