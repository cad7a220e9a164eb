"""How many host threads widen results: no more than the process's CPU quota
leaves (beedrill_amd/csrc/bd_cpus.h, compiled here; no GPU needed)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "beedrill_amd",
                    "csrc")
MAIN = """
#include "bd_cpus.h"
#include <stdlib.h>
int main(int, char **a) {
    printf("%d", bd::quota_cpus(atoi(a[1]), a[2], a[3]));
    return bd::usable_cpus() >= 1 ? 0 : 1;
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("cpus")
    (d / "main.cc").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", CSRC, "-o", str(d / "main"),
                    str(d / "main.cc")], check=True)
    return str(d / "main")


@pytest.mark.parametrize("groups,files,want", [
    (None, {}, 64),
    ("", {}, 64),
    ("no colons\n0::/gone\n", {}, 64),
    ("0::/\n", {"cpu.max": "max 100000\n"}, 64),
    ("0::/\n", {"cpu.max": "100000 100000\n"}, 1),
    ("0::/\n", {"cpu.max": "30000 100000\n"}, 1),
    ("0::/\n", {"cpu.max": "399999 100000\n"}, 3),
    ("0::/\n", {"cpu.max": "9900000 100000\n"}, 64),
    ("0::/\n", {"cpu.max": "garbage\n"}, 64),
    ("0::/\n", {"cpu.max": ""}, 64),
    ("0::/a/b\n", {"a/b/cpu.max": "max 100000\n", "a/cpu.max": "200000 100000\n"}, 2),
    ("0::/a/b\n", {"a/b/cpu.max": "500000 100000\n", "a/cpu.max": "800000 100000\n"}, 5),
    ("0::/a/b\n", {"cpu.max": "700000 50000\n"}, 14),
    ("4:memory:/m\n3:cpu,cpuacct:/job\n", {"cpu/job/cpu.cfs_quota_us": "250000\n",
                                           "cpu/job/cpu.cfs_period_us": "100000\n"}, 2),
    ("3:cpu,cpuacct:/\n", {"cpu/cpu.cfs_quota_us": "-1\n", "cpu/cpu.cfs_period_us": "100000\n"}, 64),
    ("3:cpuset:/\n", {"cpu/cpu.cfs_quota_us": "100000\n", "cpu/cpu.cfs_period_us": "100000\n"}, 64),
    ("3:cpu:/j\n0::/j\n", {"cpu/j/cpu.cfs_quota_us": "600000\n",
                           "cpu/j/cpu.cfs_period_us": "100000\n"}, 6),
])
def test_cpus_left_by_quotas(exe, tmp_path, groups, files, want):
    if groups is not None:
        (tmp_path / "groups").write_text(groups)
    for name, text in files.items():
        p = tmp_path / "tree" / name
        p.parent.mkdir(parents=True, exist_ok=True)
        p.write_text(text)
    r = subprocess.run([exe, "64", str(tmp_path / "groups"), str(tmp_path / "tree")],
                       capture_output=True, text=True)
    assert r.returncode == 0 and int(r.stdout) == want
