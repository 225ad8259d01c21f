"""The operations that the kernels execute, counted by flops.executed, against the matrix products that the profiler
counts an atom at the benchmark's header and 57 neighbours (profiles/fe16k_lmax6_sq_counters.txt)."""
import importlib

from helpers import PKG

flops = importlib.import_module("magace_amd.flops")


def test_executed_products_of_the_benchmark_header():
    ex = flops.executed(PKG.potgen.H2000, 31272, 57.3)
    assert ex["density"] == 2048 * 434
    assert ex["forces"] == 2048 * 528
    assert ex["adjoint"] == 8 * 31272
