"""The kernels that the GEMM and few-row tests name at their sizes are those the
launchers choose there (the host-only rules, compiled from the library's header)."""

from __future__ import annotations

import subprocess

import pytest

import helpers
import test_gpu_gemm_split as gemm
import test_gpu_skinny as skinny

CUS = 256  # of an MI355X


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    exe = tmp_path_factory.mktemp("choices") / "choices"
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{helpers.PKG_DIR / 'csrc' / 'kernels'}",
                    str(helpers.REPO / "tests" / "cpp" / "choices.cpp"), "-o", str(exe)], check=True)

    def run(lines):
        out = subprocess.run([str(exe), str(CUS)], input="\n".join(lines) + "\n", text=True,
                             capture_output=True, check=True).stdout.splitlines()
        assert len(out) == len(lines)
        return out

    return run


@pytest.mark.parametrize("cases", [gemm.FLOAT64, gemm.SPECIAL, gemm.FORMS],
                         ids=["float64", "special", "forms"])
def test_matmul_cases_take_the_kernel_they_name(choose, cases):
    lines = ["gemm {} {} {} {} {}".format(*(c if len(c) == 5 else (*c, "f32", "kn"))) for c in cases]
    assert dict(zip(cases, choose(lines))) == cases


def test_every_tile_and_form_is_among_the_cases():
    kinds = set(gemm.FLOAT64.values())
    for tile in ("256x128", "128x128", "128x64", "64x64"):
        assert any(k.startswith(tile) and k.endswith("split") for k in kinds), tile
        for form in ("ALIGNED", "ANY", "SHIFT"):
            assert any(k.startswith(f"{tile} {form}") for k in kinds), (tile, form)


@pytest.mark.parametrize("cases", [skinny.ONE_LAUNCH, skinny.ONE_LAUNCH_TAILS],
                         ids=["one launch", "tails"])
def test_few_row_cases_take_the_kernel_they_name(choose, cases):
    assert dict(zip(cases, choose([f"few {n} {k}" for n, k in cases]))) == cases


def test_a_k_that_the_split_kernel_cannot_count_goes_to_the_fp32_instruction(choose):
    last = 2**31 - 1 - 1024
    assert choose([f"gemm 17 1 {k} f32 kn" for k in (last, last + 1, 2**31 - 1)]) == [
        "64x64 SHIFT split", "fp32 staged", "fp32 staged"]
