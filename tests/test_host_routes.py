"""Which kernels the runtime compiles and launches, and the memory it takes for them, on the CPU: the host sources
with the double of the device layer behind hooks (tests/host/route_driver.cpp, a scenario per run), under the
sanitizers."""
import os
import subprocess

import pytest

from tests.host import build as host_build


@pytest.fixture(scope="module")
def driver():
    host_build.build()
    objs = [os.path.join(host_build.OUT, s + ".o") for s in host_build.HOST]
    from map_amd import build as B
    exe = os.path.join(host_build.OUT, "route_driver")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-Wno-unused-function"] + host_build.SAN +
                   ["-I" + B.BUILD, "-I" + host_build.CSRC, os.path.join(host_build.HERE, "route_driver.cpp")] + objs +
                   ["-o", exe, "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["compile", "served plan", "no bits", "served flow", "zone records", "zone records, small device"])
def test_routes(driver, scenario):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0", UBSAN_OPTIONS="print_stacktrace=1:halt_on_error=1")
    r = subprocess.run([driver, scenario], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300, env=env, cwd="/tmp")
    assert r.returncode == 0 and "route driver: ok" in r.stdout, r.stdout[-3000:]
