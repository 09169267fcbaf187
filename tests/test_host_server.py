"""The request loop without a GPU (tests/host): a server that is destroyed
while its worker has not come back from the last request, and requests of
several threads at once."""
import subprocess

import pytest

import hostlib


@pytest.fixture(scope="module")
def build(tmp_path_factory):
    return str(tmp_path_factory.mktemp("host"))


@pytest.mark.parametrize("requests", [0, 1, 3])
def test_destroyed_right_after_a_request(build, requests):
    exe = hostlib.program(build, "server_stop.cpp")
    r = subprocess.run([exe, str(requests)], capture_output=True, text=True, timeout=20)
    assert r.returncode == 0 and r.stdout == "stopped\n", (r.returncode, r.stdout, r.stderr)


def test_requests_of_several_threads(build):
    exe = hostlib.program(build, "server_submit.cpp")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=20)
    assert r.returncode == 0 and r.stdout == "distinct\n", (r.returncode, r.stdout, r.stderr)
