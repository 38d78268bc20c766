"""Exhaustive CPU check of the trit kernel's operand tables: builds
tests/pair_tables.cpp against ternel_amd/csrc/tq1_bytes.h with the host
compiler and runs it over all byte values, legal and illegal."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_every_byte_value_gives_its_operand_pairs(tmp_path) -> None:
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    target = tmp_path / "pair_tables"
    subprocess.run([compiler, "-std=c++17", "-O1", "-Wall", "-Werror", "-Wno-unknown-pragmas", "-Wno-format-extra-args",
                    "-D__host__=", "-D__device__=", f"-I{ROOT / 'ternel_amd' / 'csrc'}",
                    str(ROOT / "tests" / "pair_tables.cpp"), "-o", str(target)],
                   check=True, capture_output=True, text=True)
    result = subprocess.run([str(target)], capture_output=True, text=True, timeout=60)
    assert result.returncode == 0 and result.stdout.splitlines()[-1] == "ok", result.stdout + result.stderr
