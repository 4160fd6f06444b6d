"""Runs tests/host/test_plan_rules.cpp: the rules of the plan that are arithmetic alone."""
import os
import subprocess

HOST = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


def test_rules_of_the_plan():
    subprocess.check_call(["make", "-C", HOST, "test_plan_rules"])
    p = subprocess.run([os.path.join(HOST, "test_plan_rules")], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=60, text=True)
    assert p.returncode == 0 and "0 failed" in p.stdout, p.stdout
