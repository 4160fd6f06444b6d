"""Runs tests/host/test_device_pool.cpp: the pool of device memory and context parts against a runtime whose calls fail."""
import os
import subprocess

HOST = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


def test_pool_on_a_runtime_that_fails():
    subprocess.check_call(["make", "-C", HOST, "test_device_pool"])
    p = subprocess.run([os.path.join(HOST, "test_device_pool")], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=60, text=True)
    print(p.stdout, flush=True)
    assert p.returncode == 0 and "0 failed" in p.stdout, p.stdout
