"""Host rules of the launchers of the prefill and the backward (csrc/tpa_prefill.hip, tpa_bwd_mfma.hip), compiled here from their own
text, without a GPU: how the workgroups over dense tiles are ordered on an XCD, and which calls take workgroups of four waves."""

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
        + "enum { TPA_CAUSAL_BOTTOM_RIGHT = 2 };\nconstexpr int kTK = 64;\n"
        + "struct PrefillParams { int B, H, lq, lk, causal, coff; const int32_t* kvseg; };\n"
        + "".join(function(n, "tpa_prefill.hip") for n in ("dense_pair_groups", "wants_four_waves"))
        + "struct BwdParams { int B, H, lq, lk, causal; const int32_t* qseg; };\n"
        + function("bwd_wants_four_waves", "tpa_bwd_mfma.hip")
        + """
extern "C" int bwd_four_waves(int B, int lq, int lk, int H, int causal) { return bwd_wants_four_waves({B, H, lq, lk, causal, nullptr}); }
extern "C" int four_waves(int B, int lq, int lk, int H, int causal, int coff, int ids, int dense) {
  return wants_four_waves({B, H, lq, lk, causal, coff, ids ? &ids : nullptr}, dense);
}
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


# (sequences, tokens, heads) over as many keys: us with eight waves, with four (head size 64, with the reconstruction)
CAUSAL_DENSE = {
    (1, 2048, 32): (48.0, 41.5), (4, 2048, 16): (56.4, 57.6), (1, 2048, 64): (60.4, 61.3), (8, 1500, 16): (70.5, 68.4),
    (8, 1024, 16): (42.8, 40.6), (8, 1024, 64): (148.4, 140.8), (4, 1600, 64): (162.9, 145.7), (8, 2000, 8): (55.3, 56.4),
    (2, 1800, 32): (57.3, 54.9), (3, 2048, 16): (49.2, 51.4), (6, 2048, 16): (82.1, 81.3), (2, 2600, 16): (56.1, 51.7),
    (3, 2560, 16): (63.5, 65.3), (2, 2560, 16): (55.8, 50.3), (1, 2304, 32): (52.8, 47.2), (1, 3200, 64): (117.2, 111.0),
    (2, 4000, 16): (87.3, 91.9), (8, 2200, 64): (517.3, 514.4), (4, 4096, 16): (166.2, 169.2), (1, 8192, 16): (153.3, 162.9),
    (1, 16384, 16): (544.0, 564.2), (3, 2300, 8): (48.5, 40.4), (2, 3500, 8): (63.9, 52.4), (1, 3000, 16): (56.6, 45.9),
    (7, 1300, 24): (85.9, 76.6), (5, 1100, 40): (80.5, 69.0), (1, 2816, 32): (61.3, 57.5), (2, 3000, 32): (105.0, 103.3),
}
CAUSAL_FUSED = {
    (1, 1024, 64): (30.0, 33.6), (1, 900, 64): (25.9, 30.1), (1, 600, 64): (21.4, 20.1), (1, 512, 64): (19.2, 17.2), (1, 1000, 32): (27.2, 23.6),
    (4, 1024, 16): (28.7, 26.7), (2, 1024, 32): (29.5, 25.7), (8, 512, 16): (20.6, 19.6), (2, 512, 64): (20.4, 22.8), (4, 512, 64): (39.0, 34.5),
    (16, 256, 16): (16.1, 15.9), (1, 1600, 40): (41.0, 37.2), (1, 1800, 32): (43.3, 37.9), (1, 1024, 48): (29.0, 32.2), (12, 768, 32): (91.9, 85.6),
    (16, 512, 16): (36.7, 34.7), (1, 700, 16): (21.6, 18.5),
}
PLAIN_DENSE = {(3, 1300, 64): (138.3, 131.2), (2, 2000, 16): (50.7, 59.7), (3, 2048, 16): (79.9, 71.3), (4, 2048, 16): (85.1, 88.0)}
PLAIN_FUSED = {
    (1, 1000, 64): (30.1, 33.8), (4, 1024, 16): (29.6, 34.2), (8, 512, 16): (20.1, 22.5), (1, 600, 64): (22.1, 24.2), (1, 300, 64): (15.9, 13.6),
    (8, 700, 64): (130.0, 134.9), (16, 512, 16): (39.7, 41.9), (8, 300, 64): (59.3, 46.8),
}
# the worse of short documents and one document in a row, against the other kernel
IDS_PLAIN_DENSE = {(2, 2000, 16): (31.1, 34.1), (4, 4096, 16): (148.1, 138.3), (4, 2048, 16): (88.8, 90.5)}


@pytest.mark.parametrize(
    "table,causal,ids,dense",
    [(CAUSAL_DENSE, 1, 0, 1), (CAUSAL_FUSED, 1, 0, 0), (PLAIN_DENSE, 0, 0, 1), (PLAIN_FUSED, 0, 0, 0), (IDS_PLAIN_DENSE, 0, 1, 1)],
)
def test_four_waves_where_they_were_measured_faster(rules, table, causal, ids, dense):
    """Within 3 %, a little more than two runs of one side differ by."""
    for (b, t, h), sides in table.items():
        four = rules.four_waves(b, t, t, h, causal, 0, ids, dense)
        assert sides[four] <= 1.03 * min(sides), ((b, t, h), "four" if four else "eight", sides)


def test_the_rule_ends_where_blocks_are_many(rules):
    """the sum over the blocks is a loop on the host: bounded, and no sum of sizes and offsets overflows"""
    big = 2**31 - 1
    for causal, coff in ((1, 0), (1, -big // 2), (1, big // 2), (2, 0)):
        rules.four_waves(1, big // 2, big // 2, 1, causal, coff, 0, 1)
        rules.four_waves(1, big // 2, 4096, 1, causal, 0, 0, 1)


# the same of training steps
BACKWARD_PLAIN = {
    (3, 4809, 16): (1349, 1382), (4, 5350, 16): (2166, 2238), (1, 5000, 16): (513.6, 534.5), (2, 4000, 16): (610, 639), (4, 3000, 16): (722, 756),
    (2, 3000, 64): (1468, 1509), (1, 10000, 16): (1793, 1827), (4, 2500, 16): (539, 557), (5, 1800, 16): (412, 410), (3, 900, 64): (322, 328),
    (2, 2300, 16): (268.7, 261.7), (3, 2300, 16): (365, 361.7), (3, 1400, 16): (186.7, 182.6), (3, 1300, 64): (554.6, 542.4), (8, 600, 64): (467.5, 438.8),
    (16, 300, 16): (112.7, 104.9), (2, 1700, 32): (291.8, 288.7), (7, 1100, 16): (260.3, 246.6), (1, 2100, 64): (421.4, 413.8), (5, 1200, 32): (395.9, 393.0),
    (1, 1000, 64): (123.1, 124.8), (2, 2000, 16): (192.9, 197.4), (4, 1024, 16): (124.0, 128.8), (4, 2048, 16): (369.4, 377.9), (1, 1500, 16): (95.0, 89.9),
}
BACKWARD_CAUSAL = {
    (1, 2048, 32): (132.3, 129.8), (4, 2048, 16): (244.4, 243.7), (8, 1500, 16): (306.6, 303.6), (8, 1024, 16): (192.7, 174.9), (16, 512, 16): (162.1, 144.9),
    (4, 1600, 64): (687, 660.6), (2, 2816, 16): (209.5, 208.9), (1, 4096, 8): (171.5, 160.3), (1, 4096, 16): (216.4, 214.0), (2, 3500, 16): (286.3, 292.7),
    (1, 5000, 16): (295.4, 295.6), (6, 2500, 16): (500.1, 501.0), (5, 1800, 16): (269.6, 261.8), (7, 1100, 16): (188.6, 177.3), (1, 3300, 32): (260.8, 262.9),
}


@pytest.mark.parametrize("table,causal", [(BACKWARD_PLAIN, 0), (BACKWARD_CAUSAL, 1)])
def test_four_waves_in_the_backward_where_they_were_measured_faster(rules, table, causal):
    """Within 2 %: the forward and the reconstruction are in both sides."""
    for (b, t, h), sides in table.items():
        four = rules.bwd_four_waves(b, t, t, h, causal)
        assert sides[four] <= 1.02 * min(sides), ((b, t, h), "four" if four else "eight", sides)
