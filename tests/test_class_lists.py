"""The class lists of the dispatcher (X-macros of openqp_amd/csrc/dispatch.hip) are the
ones the build compiles kernels for (openqp_amd/build.py): a class only in the build is
compiled and never launched, a class only in the dispatcher is an undefined symbol when
the library is loaded.  CPU only."""
import os
import re

import pytest

from helpers import ROOT
from openqp_amd import build as B

LISTS = {"OQPH_JK_CLASSES": B.CLASSES + B.F_JK,
         "OQPH_GRAD_CLASSES": [c for c in B.CLASSES + B.F_GRAD if c not in B.GRAD_HL],
         "OQPH_JKC_CLASSES": B.JKC, "OQPH_GRC_CLASSES": B.GRC}


@pytest.fixture(scope="module")
def macros():
    txt = open(os.path.join(ROOT, "openqp_amd", "csrc", "dispatch.hip")).read().replace("\\\n", " ")
    return {m[1]: [tuple(int(x) for x in t) for t in re.findall(r"X\((\d), (\d), (\d), (\d)\)", m[2])]
            for m in re.finditer(r"#define (OQPH_\w+_CLASSES)\(X\)(.*)", txt)}


@pytest.mark.parametrize("name", sorted(LISTS))
def test_dispatcher_and_build_agree(macros, name):
    assert len(macros[name]) == len(set(macros[name]))
    assert sorted(macros[name]) == sorted(LISTS[name])
