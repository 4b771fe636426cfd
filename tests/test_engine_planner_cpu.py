"""The native engines' GEMM plans (engine_util.h GemmPlanner) against the Python ones
(ops/gemm.py resolve): one measured table, one estimate, so the same tile for every size, with the
library GEMM's entries read (CAKE_GEMM_LIB=1) and without."""
import json
import shutil
import subprocess

import pytest

from cake_amd import build as B
from cake_amd.ops import gemm as G

pytestmark = pytest.mark.skipif(not B.GEMM_LIB.exists() or shutil.which(B.CXX) is None,
                                reason="native libraries not built")

PROBE = r"""
#include "engine_util.h"
#include <cstdio>
#include <iostream>
int main(int, char** argv) {
  cake::GemmPlanner p;
  p.load(argv[1]);
  long long M, Nv, K;
  int id, big, mfma;
  std::string epi;
  while (std::cin >> M >> Nv >> K >> epi >> id >> big >> mfma) {
    const auto r = p.resolve(M, Nv, K, epi, id, big != 0, mfma != 0);
    std::printf("%d %d\n", r.first, r.second);
  }
}
"""


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    d = tmp_path_factory.mktemp("planner")
    (d / "probe.cpp").write_text(PROBE)
    rt = B.CSRC / "runtime"
    subprocess.run([B.CXX, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{B.CSRC / 'engine'}", str(d / "probe.cpp"), str(rt / "json.cpp"),
                    str(rt / "net.cpp"), str(rt / "proto.cpp"), str(B.GEMM_LIB), f"-Wl,-rpath,{B.LIB}",
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-ldl", "-lpthread",
                    "-o", str(d / "probe")], check=True)
    return d / "probe"


@pytest.mark.parametrize("lib", ["0", "1"])
def test_engines_plan_as_python_does(probe, tmp_path, monkeypatch, lib):
    table = tmp_path / "table.json"
    entry = {"M": 2048, "Nv": 4096, "K": 4096, "epi": "store"}
    table.write_text(json.dumps({"entries": [
        {**entry, "cfg": G.LIB, "splits": 1}, {**entry, "cfg": 27, "splits": 1},
        {**entry, "M": 512, "cfg": G.LIB, "splits": 1}, {**entry, "M": 300, "cfg": 13, "splits": 2}]}))
    monkeypatch.setenv("CAKE_GEMM_LIB", lib)
    monkeypatch.setenv("CAKE_GEMM_TABLE", str(table))
    monkeypatch.setattr(G, "_TUNED", G._load_tuned())
    monkeypatch.setattr(G, "_resolved", {})
    monkeypatch.setattr(G, "_plans", {})
    ask = [(M, Nv, K, epi, big, mfma) for M in (65, 300, 512, 777, 2048) for Nv, K in
           ((4096, 4096), (28672, 4096), (640, 72)) for epi in ("store", "resid32", "swiglu")
           for big in (0, 1) for mfma in (0, 1)]
    text = "".join(f"{M} {Nv} {K} {epi} {G.EPI[epi]} {big} {mfma}\n" for M, Nv, K, epi, big, mfma in ask)
    out = subprocess.run([probe, str(table)], input=text, capture_output=True, text=True, check=True)
    got = [tuple(map(int, line.split())) for line in out.stdout.splitlines()]
    want = [G.resolve(M, Nv, K, epi, bool(big), bool(mfma)) for M, Nv, K, epi, big, mfma in ask]
    assert got == want
    named = {a[:4] for a, p in zip(ask, got) if p[0] == G.LIB}
    assert named == ({(2048, 4096, 4096, "store"), (512, 4096, 4096, "store")} if lib == "1" else set())
