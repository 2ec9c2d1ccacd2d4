"""Builds tests/cpp/_build/libfacade_check.so: the C++ façade check
(facade_check.cpp over include/dgmr.hpp) that tests/test_gpu_facade.py loads,
libreach_check.so, the host build of the blends' tile-reach test that
tests/test_tile_reach.py checks, libsection_check.so, the host build of the
marcher's section list that tests/test_section_list.py checks, and
libraster_check.so, the host build of the rasteriser's scalar terms that
tests/test_raster_terms.py checks.  Run by __graft_entry__.build() after the
library itself."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
LIB_DIR = os.path.join(ROOT, "differentiable_gaussian_mixture_renderer_amd", "_lib")
OUT = os.path.join(HERE, "_build", "libfacade_check.so")


REACH_OUT = os.path.join(HERE, "_build", "libreach_check.so")


SECTION_OUT = os.path.join(HERE, "_build", "libsection_check.so")


RASTER_OUT = os.path.join(HERE, "_build", "libraster_check.so")


def _build_host(source: str, out: str) -> str:
    """A device header built for the host (g++, no contraction, as the
    kernels compile)."""
    os.makedirs(os.path.dirname(out), exist_ok=True)
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", os.path.join(HERE, source), "-o", out + ".tmp"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed:\n{res.stdout}{res.stderr}")
    os.replace(out + ".tmp", out)
    return out


def build_reach() -> str:
    """The tile-reach test of the blends, for a CPU brute-force check."""
    return _build_host("reach_check.cpp", REACH_OUT)


def build_sections() -> str:
    """The marcher's section list, for a CPU check against the restatement."""
    return _build_host("section_check.cpp", SECTION_OUT)


def build_raster() -> str:
    """The rasteriser's scalar terms, for a CPU check against double."""
    return _build_host("raster_check.cpp", RASTER_OUT)


def build() -> str:
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    cmd = ["hipcc", "-O2", "-std=c++17", "-fPIC", "-shared", "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "facade_check.cpp"),
           "-L", LIB_DIR, "-ldgmr_hip", "-Wl,-rpath,$ORIGIN/../../../differentiable_gaussian_mixture_renderer_amd/_lib", "-o", OUT + ".tmp"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed:\n{res.stdout}{res.stderr}")
    os.replace(OUT + ".tmp", OUT)
    return OUT


if __name__ == "__main__":
    print(build_reach())
    print(build_sections())
    print(build_raster())
    print(build())
