"""The names under which autotune reports and the bench show launch variants say
what the kernels of the precision do."""
import pytest


@pytest.mark.parametrize("precision,names", [
    ("fp64", {-1: "default", 8: "64x64", 16: "48x64", 83: "by_shape"}),
    ("fp32", {-1: "default", 8: "64x64", 16: "128x64", 83: "by_shape"}),
    ("i8x5", {-1: "default", 200: "int8", 83: "bk8_w3"}),
    ("i8x4", {-1: "default", 200: "int8", 201: "int8x5", 83: "bk8_w3"}),
    ("bf16x3", {-1: "default", 0: "64x64", 9: "64x64_astat", 13: "128x192_presplit_w8"}),
])
def test_variant_names(ggpu, precision, names):
    k = object.__new__(ggpu.GwKernel)
    k.precision = precision
    assert {v: k.variant_name(v) for v in names} == names
    assert k.variant_name(84) == "84"          # no kernel has this id
