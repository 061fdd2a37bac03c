"""Group accesses promise one element's alignment (csrc/sr_group_access.h), compiled for the host.

Views that start anywhere take the same accesses as aligned ones, so the
compiler must not be told of any alignment past the element's.  The attribute
is lost where the type passes through a template argument, with nothing to
see at run time on a GPU that takes any alignment.
"""

from __future__ import annotations

import os
import re
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
CLANG = [str(Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "llvm" / "bin" / "clang++"), "-O2", "-std=c++17",
         "-I", str(ROOT / "stochastic-rounding-pytorch_amd" / "csrc"),
         str(ROOT / "tests" / "native" / "group_access.cpp")]


def test_groups_move_from_any_element(tmp_path):
    binary = tmp_path / "group_access"
    subprocess.run([*CLANG, "-o", str(binary)], check=True)
    result = subprocess.run([str(binary)], capture_output=True, text=True, timeout=60)
    assert result.returncode == 0 and result.stdout == "0 failures\n", (result.returncode, result.stdout)


def test_no_access_promises_more_than_an_element(tmp_path):
    listing = tmp_path / "group_access.ll"
    subprocess.run([*CLANG, "-S", "-emit-llvm", "-o", str(listing)], check=True)
    # The bodies of load<BYTES, kCached> and store<BYTES> hold one access of the group's memory each.
    promised = {}
    for kind, body in re.findall(r"^define [^\n]*@_ZN\S*?(4loadILi\d+ELb[01]E|5storeILi\d+E)\S*\([^\n]*\{\n(.*?)^\}",
                                 listing.read_text(), re.M | re.S):
        kept = r"load" if kind.startswith("4load") else r"store"
        promised[kind] = [int(n) for n in re.findall(rf"^.*\b{kept} (?:<\d x i32>|i32).*align (\d+)", body, re.M)]
    assert promised == {"4loadILi16ELb0E": [4], "4loadILi16ELb1E": [4], "4loadILi8ELb0E": [2], "4loadILi4ELb0E": [1],
                        "5storeILi16E": [4], "5storeILi8E": [2], "5storeILi4E": [1]}
