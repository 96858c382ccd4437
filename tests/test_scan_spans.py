"""The spans the autotuner tries (mdet_amd/csrc/scan_spans.h): the span an untuned
context takes is the first of them at every size, so tuning cannot settle for
less."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_the_default_span_is_tried_at_every_size(tmp_path):
    exe = str(tmp_path / "model")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-o", exe, os.path.join(HERE, "scan_spans_model.cpp")],
                   check=True)
    lines = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines()
    assert lines.pop() == "0 1"  # a percent is noise, a tenth is not
    seen = set()
    for line in lines:
        n, default, *spans = map(int, line.split())
        seen.add(default)
        assert spans[0] == default and len(set(spans)) == len(spans)
        assert {512, 1024, 2048, 4096} <= set(spans)
        assert all(s % 256 == 0 and 256 <= s <= max(4096, default) for s in spans), n
    assert seen == {512, 1024, 2048, 4096, 8192, 16384}
