"""The names of the native libraries: a change to anything that is compiled into one gives it another name, so that what was
built before is not loaded."""

import shutil

import pytest

from distie_amd.csrc import build

# headers that each library is compiled with, also those that only other headers include
HEADERS = {"ops": {"common.h", "lds_load.h", "no_alloc.h", "packed.h", "vector_values.h"}, "attn_d128": {"common.h", "lds_load.h"},
           "attn_d48": {"common.h", "lds_load.h"}, "mixattn_d64": {"common.h"}, "library": {"common.h"}, "core": set()}


@pytest.fixture
def sources(tmp_path, monkeypatch):
    for path in build.SRC.iterdir():
        if path.is_file():
            shutil.copy(path, tmp_path)
    monkeypatch.setattr(build, "SRC", tmp_path)
    return tmp_path


@pytest.mark.parametrize("changed", sorted(set().union(*HEADERS.values())))
def test_a_changed_header_renames_the_libraries_that_hold_it(sources, changed):
    before = {name: build.file_name(name) for name in HEADERS}
    assert before == {name: build.file_name(name) for name in HEADERS}
    path = sources / changed
    path.write_text(path.read_text() + "\n")
    assert {name for name in HEADERS if build.file_name(name) != before[name]} == {n for n, held in HEADERS.items() if changed in held}


def test_headers_are_followed_through_headers(sources):
    (sources / "inner.h").write_text("#pragma once\n")
    (sources / "outer.h").write_text('#pragma once\n  #  include "inner.h"\n#include "outer.h"\n#include <vector>\n')
    path = sources / "attention.hip"
    path.write_text('#include "outer.h"\n' + path.read_text())
    before = build.file_name("attn_d64")
    (sources / "inner.h").write_text("#pragma once\nint changed;\n")
    assert build.file_name("attn_d64") != before
