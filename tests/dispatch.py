"""Asks the compiled dispatch rules (dispatch_rules.cpp) which kernel a call takes."""
import functools
import os
import shutil
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@functools.lru_cache(maxsize=1)
def _program():
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    exe = os.path.join(tempfile.mkdtemp(prefix="dispatch"), "dispatch_rules")
    subprocess.run([gxx, "-O1", "-std=c++17", "-o", exe, os.path.join(HERE, "dispatch_rules.cpp")], check=True)
    return exe


def ask(*lines):
    """The answers to query lines such as "tiled 640 2560 256 819456 512 20 1"."""
    r = subprocess.run([_program()], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True)
    out = r.stdout.split("\n")[:-1]
    assert len(out) == len(lines), out
    return out


def tiled(n, k, w_off, s_off, n_experts, max_n, exact):
    return ask(f"tiled {n} {k} {w_off} {s_off} {n_experts} {max_n} {int(exact)}")[0]


def counted(n, k, wide, exact, counts, max_n=None):
    """Which kernel the device takes where both are launched."""
    return ask(f"counted {n} {k} {int(wide)} {int(exact)} {max_n or max(counts)} {len(counts)} "
               + " ".join(map(str, counts)))[0]


def step(T, E, k, hidden, inter):
    return ask(f"step {T} {E} {k} {hidden} {inter}")[0]
