"""Host rules of the prefill launcher (csrc/tpa_prefill.hip), compiled here from its own text, without a GPU: how the workgroups
over dense tiles are ordered on an XCD."""

import ctypes
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensor-product-attention-jax_amd", "csrc")


def function(name, file):
    """the text of the function of that name, up to the brace that closes it"""
    text = open(os.path.join(CSRC, file)).read()
    found = re.search(r"^[^\n/]*\b%s\(" % name, text, re.M)
    depth, at = 0, text.index("{", found.end())
    for i in range(at, len(text)):
        depth += {"{": 1, "}": -1}.get(text[i], 0)
        if depth == 0:
            return text[found.start() : i + 1] + "\n"
    raise AssertionError(name)


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    src = tmp_path_factory.mktemp("rules") / "rules.cc"
    src.write_text(
        "#include <algorithm>\n#include <cstdint>\nusing std::min; using std::max;\n#define __device__\n#define __forceinline__ inline\n"
        + "".join(function(n, "tpa_common.h") for n in ("pair_in_group", "pair_group_workgroups", "pair_groups"))
        + function("dense_pair_groups", "tpa_prefill.hip")
        + """
extern "C" int groups(int npairs, int nqb, int four, int causal) { return dense_pair_groups(npairs, nqb, four, causal); }
extern "C" int place(int id, int npairs, int groups, int nblk, int* pair, int* rank) { return pair_in_group(id, npairs, groups, nblk, *pair, *rank); }
"""
    )
    lib = src.with_suffix(".so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", str(src), "-o", str(lib)], check=True)
    return ctypes.CDLL(str(lib))


@pytest.mark.parametrize(
    "pairs,rows,four",
    [(64, 4096, 1), (16, 8192, 1), (128, 1536, 1), (64, 3200, 1), (32, 1920, 1), (48, 1777, 1), (64, 4096, 0), (64, 2048, 0)],
)
def test_no_group_of_pairs_starts_its_heavy_blocks_late(rules, pairs, rows, four):
    """Causal blocks taken up in their order by the workgroups an XCD holds at once (two per compute unit of four waves, one of
    eight): the last one ends within a tenth of the mean, or of the heaviest block where that is longer."""
    block, resident = (128, 64) if four else (256, 32)
    nblk = -(-rows // block)
    groups = rules.groups(pairs, nblk, four, 1)
    worst = 0.0
    for xcd in range(8):
        ends, total, heaviest = [0] * resident, 0, 0
        pair, rank = ctypes.c_int(), ctypes.c_int()
        for slot in range(-(-pairs // 8) * nblk):
            if not rules.place(slot * 8 + xcd, pairs, groups, nblk, ctypes.byref(pair), ctypes.byref(rank)):
                continue
            tiles = -(-min(rows, (nblk - rank.value) * block) // 64)
            total, heaviest = total + tiles, max(heaviest, tiles)
            i = ends.index(min(ends))
            ends[i] += tiles
        worst = max(worst, max(ends) / max(total / resident, heaviest))
    assert worst <= 1.1, worst
