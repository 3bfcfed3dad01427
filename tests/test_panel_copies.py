"""The panel kernel keeps its producers and its count reader inline (as functions
its registers are laid out worse); the sampled product's panel form has them as
functions.  Both must stay one text: the plan's layout and the counted waits
are the same."""
import os
import re

from conftest import ROOT


def _source():
    with open(os.path.join(ROOT, "spmm_amd", "csrc", "panel_kernel.hpp")) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    return re.sub(r"\s+", " ", text)


def _both(first, until_a, until_b):
    s = _source()
    a = s.index(first)
    b = s.index(first, a + 1)
    assert s.find(first, b + 1) < 0
    return s[a:s.index(until_a, a)].rstrip(" }"), s[b:s.index(until_b, b)].rstrip(" }")


def test_producers_are_the_same_text():
    a, b = _both("const int piece = lane % (G::kRowBytes / 16);", "return;", "template <int kRor>")
    assert len(a) > 2000 and "s_waitcnt vmcnt" in a
    assert a == b


def test_count_readers_are_the_same_text():
    a, b = _both("pn_static_for<0, kPnCntUsed / 4>", "};", "__device__")
    a, b = (re.sub(r"[^;]*$", "", x) for x in (a, b))
    assert "rem == 3" in a and a == b
