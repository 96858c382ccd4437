"""The lists of an edge-list call that the device fills before the host knows
their lengths, on a host model built from the library's own rule
(mdet_amd/csrc/pass_lists.h): whatever the capacities, no candidate record is
read that no kernel wrote, and the passes that a call may take are enough for
every list to be sized from its own length."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("lists") / "model")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-o", exe, os.path.join(HERE, "pass_lists_model.cpp")],
                   check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    print(out, flush=True)
    return [dict(zip(w[::2], map(int, w[1::2]))) for w in (line.split() for line in out.splitlines())]


def test_no_unwritten_record_is_read(model):
    r = model[1]
    assert r["gaps"] > 1000 and r["reads"] > 1000  # the sweep reaches both sides
    assert r["unwritten_read"] == 0
    assert r["refused_whole"] == 0  # and what is whole is read


def test_every_list_is_sized_within_the_passes_of_a_call(model):
    r = model[0]
    assert r["failed"] == 0 and r["failed_full_rows"] == 0
    # lists, survivors and candidates, then all fits; the full rows' lists come behind those
    assert r["most"] == 3 and r["most_full_rows"] == r["limit"]
