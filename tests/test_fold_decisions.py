"""The kernels that fold a solver's sums themselves also record the loop's new state, by the scene's
first workgroup, while waves of other workgroups may not have started. A wave that read there what is
being written could take another way through the fold's barriers than the rest of its workgroup. So in
their folding form no word of the record is read that the same launch writes. Checked on the source.
"""
import os
import re

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mps_cuda_amd", "csrc", "sph.hip")


def _block(text: str, start: int) -> str:
    """The braces' content that opens at or after `start`."""
    a = text.index("{", start)
    depth = 0
    for k in range(a, len(text)):
        depth += {"{": 1, "}": -1}.get(text[k], 0)
        if depth == 0:
            return text[a + 1:k]
    raise AssertionError("unbalanced braces")


def _function(text: str, name: str) -> str:
    return _block(text, re.search(rf"\b{name}\([^;]*?\)\s*{{", text, re.S).start())


def _writes(body: str) -> set:
    return set(re.findall(r"(?:st\[sid\]\.|st->|sd->)(\w+)(?:\[[^]]*\])?\s*=(?!=)", body))


@pytest.mark.parametrize("kernel,record", [("k_pressure_apply", "record_pressure"), ("k_cg_apply", "record_cg"),
                                           ("k_cg_update3", None)])
def test_no_word_is_read_that_the_launch_writes(kernel, record):
    with open(SRC) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    body = _function(text, kernel)
    # what runs with FOLD: everything but the `else` of `if constexpr (FOLD)`
    m = re.search(r"if constexpr \(FOLD\)", body)
    fold = _block(body, m.end())
    before, after = body[:m.start()], body[m.end():].lstrip()[len(fold) + 2:]
    if after.lstrip().startswith("else"):
        after = after[after.index(_block(after, 0)) + len(_block(after, 0)):]
    if kernel == "k_cg_apply":  # (its statements after the folding branch, which always returns, are the other form's)
        assert fold.rstrip().endswith(";") and "return" in fold.rstrip().rsplit("\n", 1)[-1]
        after = ""
    writes = _writes(before + fold)
    if record:
        assert record in fold
        writes |= _writes(_function(text, record))
    assert writes  # the parts were found
    reads = set()
    for part in (before, fold, after):
        reads |= set(re.findall(r"st\[sid\]\.(\w+)(?!\w|\s*=[^=])", part))
    assert reads and not reads & writes, (reads, writes)
