"""bench.py's CPU figures where the compiled reference (oracle/_ref/libmossref.so) is absent, as on
every host without the reference checkout: each is None and the run goes on to its result line."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CALLS = {
    "cpu_baseline": (b"", (None,) * 4, 2, 1),
    "cpu_gemv": (1,),
    "cpu_attention": (),
    "cpu_prefill": (b"", 1),
    "cpu_codec": (b"", 1),
    "cpu_streams": (b"", 1, 1),
}


@pytest.fixture
def bench(monkeypatch, tmp_path):
    monkeypatch.syspath_prepend(ROOT)
    import bench
    import oracle
    missing = str(tmp_path / "libmossref.so")
    monkeypatch.setattr(oracle, "REF_SO", missing)
    monkeypatch.setattr(oracle.RefCpu.__init__, "__defaults__", (missing, "decode"))
    yield bench
    sys.modules.pop("bench", None)


@pytest.mark.parametrize("name", sorted(CALLS))
def test_without_the_reference_a_cpu_figure_is_none(bench, name):
    assert getattr(bench, name)(*CALLS[name]) is None


def test_every_cpu_figure_is_covered(bench):
    assert {n for n in dir(bench) if n.startswith("cpu_")} == set(CALLS)
    assert np.isfinite(bench.host_cpu()["cpu_share"])
