"""The byte range of a strided operand (lucid_amd/csrc/lq_extent.h), which bounds the int8 GEMM's
LDS-DMA copies: compiled for the host with g++ and checked copy by copy (no GPU), and every
descriptor of a GEMM operand is made from it."""

from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "lucid_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_copies_stay_in_the_operand(tmp_path):
    exe = tmp_path / "extent_check"
    src = os.path.join(ROOT, "tests", "native", "extent_check.cpp")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, src, "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    assert out.stdout.strip() == "ok"


@pytest.mark.parametrize("kernel,operands", [("gemm_i8_dma_kernel", "AB"), ("gemm_i8_decode_partial_kernel", "A")])
def test_gemm_kernels_bound_their_operands_by_it(kernel, operands):
    text = open(os.path.join(CSRC, "lq_gemm.hip")).read()
    body = text[text.index(f"void {kernel}"):]
    body = body[:body.index("__global__")]
    made = dict(re.findall(r"const v4i (r[ab]) = operand_rsrc\(a\.([AB]), ", body))
    assert made == {"r" + o.lower(): o for o in operands}
