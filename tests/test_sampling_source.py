"""What the sampler's kernel promises the compiler about its pointers, from its source.  No GPU."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mamba_rs_amd", "csrc")


def _text(name):
    return re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, name)).read())


def test_slot_arrays_that_the_launch_writes_are_not_restrict():
    """A generation's launch takes `active` and `seen` of its slots as parameters and moves the same slots on through GenSlots.  With __restrict__ on
    such a parameter the compiler may read it behind the barrier that stands in front of the write, and waves of a row would part ways."""
    sampling = _text("sampling.hip")
    slots = re.search(r"struct GenSlots \{(.*?)\};", _text("common.hpp"), re.S).group(1)
    members = set(re.findall(r"\*?\s*(\w+)\s*[,;]", re.sub(r"/\*.*?\*/", "", slots)))
    advance = re.search(r"void advance_slot\((.*?)\n\}", sampling, re.S).group(1)
    written = {m for m in members if re.search(rf"\bg\.{m}\[[^\]]*(?:\[[^\]]*\][^\]]*)?\]\s*(?:=[^=]|\+=)", advance)}
    assert {"active", "seen", "out_len", "finished", "prompt_pos"} <= written, written
    params = re.search(r"void sample_rows_kernel\((.*?)\)\s*\{", sampling, re.S).group(1)
    params = {re.search(r"(\w+)\s*$", p).group(1): p for p in params.split(",")}
    shared = written & set(params)
    assert shared == {"active", "seen"}
    for name in shared:
        assert "__restrict__" not in params[name], params[name].strip()
