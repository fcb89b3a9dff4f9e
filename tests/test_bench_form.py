"""bench.py's --fused: what it asks of the context and what it reports, for a
context that starts in a form of its own choice."""
import argparse

import pytest

import bench


class Engine:
    fused = 2  # as a large box starts

    def set_fused(self, on):
        self.fused = on

    def set_launch(self, waves):
        pass


class Run:
    def advance(self, steps):
        pass


@pytest.mark.parametrize("flag,form,name", [("off", 0, "separate"), ("last", 1, "last"),
                                            ("x", 2, "x")])
def test_bench_runs_the_form_it_reports(flag, form, name):
    eng = Engine()
    a = argparse.Namespace(fused=flag, sweep_waves=4, warmup=1)
    tuned, fused = bench.tune(a, eng, Run())
    assert eng.fused == fused == form
    assert tuned["fused_sweep"] == name
