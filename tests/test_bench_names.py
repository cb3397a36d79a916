"""The kernel record of bench.py names the kernels that run: its element counts
are the sources' dispatch lines."""
import importlib.util
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "dg-mpi_amd", "csrc")


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def ints(text):
    return tuple(int(x) for x in re.findall(r"\d+", text))


def test_lines_are_the_sources(bench):
    k = open(os.path.join(SRC, "dg_kernels.hip")).read()
    lim = re.search(r"lim\[2\]\[PMAX\] = \{\{([^}]*)\}, \{([^}]*)\}\}", k)
    assert (ints(lim[1]), ints(lim[2])) == (bench.TWO_PASS_FROM["f64"], bench.TWO_PASS_FROM["fp32"])
    halves = re.search(r"int halves_team\(unsigned E\) \{(.*?)\n\}", k, re.S)[1]
    assert tuple(max(int(x) for x in re.findall(r"E <= (\d+)", line))
                 for line in halves.strip().split("\n")) == bench.HALVES_TO[:3]
    q = open(os.path.join(SRC, "dg_kernels_2d.inc")).read()
    assert ints(re.search(r"unsigned lim\[PMAX\] = \{([^}]*)\}", q)[1]) == bench.QUADS_FROM


@pytest.mark.parametrize("args,name,launches", [
    ((3, 64 ** 3, 3, 0.0, None), "face_flux_kernel<3,Roe>+element_kernel<3>", 2),
    ((3, 64 ** 3, 3, 0.0, "FP32"), "face_flux_kernel<3,Roe,fp32>+element_kernel<3,fp32>", 2),
    ((3, 64 ** 3, 3, 0.0, "BF16x3"), "stage_kernel<3,Roe,fp32,bf16x3>", 1),
    ((2, 512, 3, 0.0, None), "stage_halves_kernel<2,Roe>", 1),
    ((4, 1000, 3, 0.0, None), "stage_kernel<4,Roe>", 1),
    ((3, 8000, 3, 0.1, None), "stage_kernel<3,Roe,mapped>", 1),
    ((3, 1024 ** 2, 2, 0.0, None), "stage2d_box_kernel<3,Roe>", 1),
    ((3, 1024, 2, 0.0, None), "stage2d_kernel<3,Roe>", 1)])
def test_names(bench, args, name, launches):
    assert bench.stage_kernels(*args) == (name, launches)
