"""The Python binding's configuration defaults are the library's, as the C header states them."""
import inspect
import os
import re

from gpugi_amd import rt

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "gpugi_rt.h")


def defaults(fn):
    return {p.name: p.default for p in inspect.signature(fn).parameters.values()}


def test_wide_and_batch_configuration():
    text = open(HEADER).read()
    leaf, stack, refill, wait = map(int, re.search(r"Default \((\d+), (\d+), (\d+), (\d+)\)", text).groups())
    d = defaults(rt.Context.set_wide_config)
    assert (d["refill_lanes"], d["wait_lanes"]) == (refill, wait)
    grab, grid, depth = map(int, re.search(r"Defaults: WIDE, (\d+), (\d+), (\d+)\.", text).groups())
    d = defaults(rt.Batch.config)
    assert (d["kernel"], d["tiles_per_grab"], d["grid_multiplier"], d["stack_depth"]) == \
        (rt.KERNEL_WIDE, grab, grid, depth)
