"""The encoder's page claim (fp_page_claim.hpp), every interleaving on the CPU.

Record sizes are the format's: 22528 dense bytes and a variable region of 48
to 2048 bytes in steps of 16.  Any two records exceed any one, which is what
keeps claims by a plain add from overlapping; sizes without that property do
overlap, so the search can see it.
"""

from __future__ import annotations

import subprocess

import pytest

SMALL, LARGE = 22528 + 48, 22528 + 2048


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    from pathlib import Path

    exe = tmp_path_factory.mktemp("claim") / "model"
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), str(Path(__file__).with_name("page_claim_model.cpp"))],
                   check=True)

    def run(page, fill, needs, polls=0):
        out = subprocess.run([str(exe), str(page), str(fill), str(polls), *map(str, needs)], capture_output=True,
                             text=True, timeout=100)
        return out.stdout.strip()

    return run


@pytest.mark.parametrize("page,fill,needs", [
    (LARGE, 0, [SMALL, LARGE, LARGE - 16]),  # one record's room
    (SMALL + 16, 0, [LARGE, SMALL, SMALL + 32, SMALL + 16]),  # some fit, some never do
    (SMALL - 16, 0, [SMALL, LARGE, SMALL + 512]),  # none fits
    (3 * LARGE, LARGE + 32, [SMALL, LARGE, LARGE, SMALL + 512]),  # room for two behind earlier records
    (2 * SMALL + 64, 0, [LARGE, SMALL, SMALL + 16, SMALL + 48]),  # a pending add leaves the fill inside the page
])
def test_every_interleaving_keeps_records_apart(model, page, fill, needs):
    assert model(page, fill, needs).startswith("ok")


def test_sizes_without_the_property_overlap(model):
    assert model(100, 40, [70, 20, 30]) in ("records overlap", "the fill is not what the placed records make it")


@pytest.mark.parametrize("polls", [1, 3])
@pytest.mark.parametrize("over", [16, LARGE])
def test_a_fill_that_rests_past_the_page_ends_the_wait(model, polls, over):
    # no pending add explains it: every record spills after its polls, and the fill is left as it was
    assert model(2 * LARGE, 2 * LARGE + over, [SMALL, LARGE], polls=polls).startswith("ok")
