"""The kernel names bench.py looks up in the profiles are those the profiler
prints: for the default launch shapes of each traced call, every name occurs in
the tracked trace of that call."""
import pathlib
import sys

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))
import bench  # noqa: E402

SLOTS = ("sound_column", "sound_div", "sound_momentum", "waf_vertical", "waf_horizontal",
         "adv_stagger_in", "adv_stagger_out", "tail")

# call: (column_j, wafv_group, form, kz, crm, lrotllr)
CALLS = {
    "small-24x20x10": (16, 1, "fp64", 10, 0, 0),
    "hill-64x64x23": (16, 1, "fp64", 23, 0, 0),
    "periodic-100x50x30-mixed": (16, 1, "mixed", 30, 1, 0),
    "lbc-151x127x35": (32, 2, "fp64", 35, 0, 1),
    "split-97x83x30-tracers": (16, 1, "fp64", 30, 0, 0),
    "domain-256x256x41": (32, 4, "fp64", 41, 0, 0),
    "domain-256x256x41-mixed": (32, 4, "mixed", 41, 0, 0),
    "periodic-500x100x60": (32, 2, "fp64", 60, 1, 0),
    "domain-512x512x41-mixed": (32, 4, "mixed", 41, 0, 0),
    "ensemble-8x128x128x30": (32, 4, "fp64", 30, 0, 0),
}


def traced(call):
    text = (ROOT / "profiles" / "kernel_trace_cases.md").read_text()
    part = text.split(f"## {call}\n", 1)[1].split("\n## ", 1)[0]
    return {line.split("|")[1].replace(" ", "") for line in part.splitlines()
            if line.startswith("| ")}


@pytest.mark.parametrize("call", CALLS)
def test_names_occur_in_the_trace(call):
    column_j, group, form, kz, crm, rot = CALLS[call]
    variants = dict(column=2, column_j=column_j, waf_h=0, waf_group=4, wafv_group=group,
                    waf_tile=8, waf_hgroup=0, mixed_merge=1)
    names = traced(call)
    for slot in SLOTS:
        assert bench.kernel_struct(slot, variants, form, kz, crm, rot) in names, slot


@pytest.mark.parametrize("column,column_j,kz,name", [
    (2, 64, 41, "SoundColumnChunk<double,64,4,11>"), (2, 64, 43, "SoundColumnChunk<double,32,8,6>"),
    (2, 32, 64, "SoundColumnChunk<double,32,8,8>"), (2, 32, 65, "SoundColumnChunk<double,16,16,8>"),
    (0, 32, 70, "SoundColumnChunk<double,16,16,8>"), (0, 32, 63, "SoundColumn<double>"),
    (2, 16, 129, "SoundColumnStream<double>"), (1, 32, 41, "SoundColumnStream<double>")])
def test_column_names_follow_the_height(column, column_j, kz, name):
    """The column solve falls back to a form that holds the column."""
    assert bench.kernel_struct("sound_column", dict(column=column, column_j=column_j), "fp64",
                               kz) == name
