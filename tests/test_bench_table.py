"""The benchmark's kernel table on the host: rows of an operator that could not be
set up are left out instead of timed on another one."""
from __future__ import annotations

import sys
from pathlib import Path

import pytest

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))

import bench  # noqa: E402


class Sim:
    N = 1 << 20

    def __init__(self, upload):
        self.upload = upload

    def csr(self):
        raise RuntimeError("not assembled")

    def ell(self):
        return None, None

    def set_ell(self, col, val):
        if not self.upload:
            raise RuntimeError("no memory")

    def time_kernel(self, what, reps):
        return 0.1


@pytest.mark.parametrize("upload", [True, False])
def test_stored_rows_need_the_stored_operator(upload):
    rows = bench.kernel_table(Sim(upload), 20)
    assert {n for n in rows if n.endswith("_stored")} == (
        {"spmv_stored", "spmv_dot_stored", "bicg_iter_stored"} if upload else set())
    assert "spmv_fp64" in rows and "spmv_csr" not in rows
