"""The shipped launch-shape table against the class table it was measured with."""
import json
import os
import re

from barbu_amd import build


def _classes():
    src = open(os.path.join(build.CSRC, "ftl_classes.h")).read()
    rows = re.findall(r"X\((\d+), (\d+), (\d+), (true|false), (\d+), (\d+)\)", src)
    return {int(i): (int(m), int(g), gu == "true", int(w), int(c)) for i, m, g, gu, w, c in rows}


def test_shipped_table_is_of_these_classes():
    table = json.load(open(os.path.join(build.HERE, "tuned_gfx950.json")))
    classes = _classes()
    assert len(classes) == build.NCLASSES
    for t in table["timings_us"]:
        m, g, guarded, waves, chunk = classes[t["class"]]
        assert not guarded and m * g == t["npoints"]
        assert (t["lanes"], t["waves"], t["chunk"]) == (g, waves, min(chunk, m)), t
    for n, c in list(table["class"].items()) + list(table["class_wind"].items()):
        assert classes[c][0] * classes[c][1] == int(n)
    for n, g in table["lanes"].items():
        assert classes[table["class"][n]][1] == g
