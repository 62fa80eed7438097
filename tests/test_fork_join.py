"""The fork and join around work on side streams (csrc/fork_join.h), compiled for the host: whatever fails, every
stream that was forked is joined, nothing runs on one that was not, and the first error comes back."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "fork_join.h"
int main(int, char** a)
{
    const int nst = atoi(a[1]), n = atoi(a[2]), bad_fork = atoi(a[3]), bad_work = atoi(a[4]), bad_join = atoi(a[5]);
    const int rc = mft::fork_join(
        nst, n, [&](int k) { return std::printf("f%d ", k), k == bad_fork ? 10 : 0; },
        [&](int g, int k) { return std::printf("w%d@%d ", g, k), g == bad_work ? 20 : 0; },
        [&](int k) { return std::printf("j%d ", k), k == bad_join ? 30 : 0; });
    std::printf("%d\n", rc);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("fork_join")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "matilda.ft_amd", "csrc"), "-o", str(d / "main"),
                    str(d / "main.cpp")], check=True)
    return str(d / "main")


@pytest.mark.parametrize("args, want", [
    ((0, 0, -1, -1, -1), "0"), ((1, 1, -1, -1, -1), "w0@0 0"),
    ((3, 5, -1, -1, -1), "f1 f2 w0@0 w1@1 w2@2 w3@0 w4@1 j1 j2 0"),
    ((3, 5, -1, 1, -1), "f1 f2 w0@0 w1@1 j1 j2 20"),       # a group's launch fails after the fork
    ((3, 5, -1, 0, 1), "f1 f2 w0@0 j1 j2 20"),             # the first error is the one that is reported
    ((4, 4, 2, -1, -1), "f1 f2 j1 10"),                    # no work on, and no join of, a stream that is not forked
    ((3, 3, -1, -1, 1), "f1 f2 w0@0 w1@1 w2@2 j1 j2 30"),  # a join that fails keeps no other from being joined
])
def test_every_forked_stream_is_joined(program, args, want):
    r = subprocess.run([program] + [str(a) for a in args], capture_output=True, text=True, timeout=60, check=True)
    assert r.stdout.split() == want.split()
