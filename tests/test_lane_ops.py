"""Exchanges between the lanes of a wavefront in the kernels' source: none stands behind `||`, `&&` or
`?`, which switch off the lanes that need no second operand, and a lane that reads one that is
switched off gets an undefined value."""

import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "athenak_amd",
                    "csrc")
FILES = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.hpp")))
EXCHANGE = re.compile(r"\b(__shfl\w*|__ballot|__any|__all|WaveScan|WaveInclScan|CoopSum|"
                      r"__builtin_amdgcn_(ds_bpermute|readlane|readfirstlane|update_dpp|mov_dpp))\(")


def open_part(text):
    """text without its closed parentheses: what still encloses its end."""
    while True:
        cut = re.sub(r"\([^()]*\)", " ", text)
        if cut == text:
            return text
        text = cut


def offending(text):
    text = re.sub(r"//[^\n]*|/\*.*?\*/", " ", text, flags=re.S)
    return [" ".join(statement.split()) for statement in re.split(r"[;{}]", text)
            if any(re.search(r"\|\||&&|\?", open_part(statement[:m.start()]))
                   for m in EXCHANGE.finditer(statement))]


@pytest.mark.parametrize("path", FILES, ids=os.path.basename)
def test_no_exchange_behind_a_short_circuit(path):
    with open(path) as f:
        assert offending(f.read()) == []


def test_the_check_sees_one():
    assert offending("const bool head = lane == 0 || __shfl_up(at, 1, 64) != at;")
    assert offending("heads = __ballot(lane == 0 || __shfl_up(at, 1, 64) != at);")
    assert not offending("const long long prev = __shfl_up(at, 1, 64); f(lane == 0 || prev != at);")
    assert not offending("const int a = WaveScan(on ? n : 0), e = WaveScan((on && n) ? 1 : 0);")
