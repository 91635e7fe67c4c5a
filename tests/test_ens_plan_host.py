"""The ensemble's automatic chunk on the CPU (tests/ens_plan_check.cpp): the
rule ends for every ensemble that a capacity of 2^28 particles allows, keeps a
launch at 2^22 workgroups, and leaves the state to the 256-star items (chunk 0)
where one chunk per cluster has more."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
MOST = 1 << 22


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    cc = shutil.which("g++")
    if cc is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("plan") / "ens_plan_check")
    subprocess.run([cc, "-O2", "-std=c++17", "-I", os.path.join(ROOT, "pn_amd", "csrc"),
                    os.path.join(HERE, "ens_plan_check.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True)

    def run(*cases):
        out = subprocess.run([exe], input="\n".join(f"{a} {b}" for a, b in cases), timeout=60,
                             check=True, capture_output=True, text=True).stdout
        return [tuple(int(t) for t in line.split()[2:]) for line in out.splitlines()]

    return run


@pytest.mark.parametrize("clusters,stars", [
    (MOST + 1, 1), (MOST + 1, 64), (MOST // 2 + 1, 65), (1 << 24, 3), (1 << 27, 1)])
def test_more_rows_than_a_launch(check, clusters, stars):
    assert check((clusters, stars)) == [(0, -1)]


@pytest.mark.parametrize("clusters,stars", [
    (1, 0), (1, 1), (4, 0), (MOST, 0), (MOST, 1), (MOST, 64), (MOST // 2, 65), (MOST // 64, 4000),
    (1, (1 << 28) - 1), (100, 2000000), (300, 70000)])
def test_launch_fits(check, clusters, stars):
    [(L, parts)] = check((clusters, stars))
    assert L >= 64 and parts <= MOST
    rows = clusters * -(-stars // 64)
    assert parts == rows * -(-stars // L)
    if L > 4096:                    # doubled only as far as needed
        assert rows * -(-stars // (L // 2)) > MOST


@pytest.mark.parametrize("clusters,stars", [(256, 8192), (256, 512), (12, 9000), (40, 1000), (8, 300)])
def test_ordinary_ensembles(check, clusters, stars):
    """4096, halved to 512 below 6000 workgroups and to 64 below 1024."""
    parts = lambda L: clusters * -(-stars // 64) * -(-stars // L)      # noqa: E731
    L = 4096
    while L > 512 and parts(L) < 6000:
        L //= 2
    while L > 64 and parts(L) < 1024:
        L //= 2
    assert check((clusters, stars)) == [(L, parts(L))]
