"""The generated tile loops of the prefill kernel (csrc/gen_prefill_loop.py) against the C++ side that hands
them their registers (csrc/tpa_prefill.hip), without a GPU: every register an instruction of a loop writes
is an in/out operand of its asm statement or a listed clobber, every register it reads is an operand or was
written earlier in the loop, input-only operands are never written, each copy of the iteration passes
exactly one workgroup barrier, and nothing beyond the 256 registers of a wave is named.  The rare paths, which the asm statement
includes behind the loop, are held to the same rules, each from the place that branches to it."""

import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tensor-product-attention-jax_amd", "csrc")
LOOPS = [(128, "dense"), (64, "dense"), (64, "dense4w"), (128, "r2"), (64, "r2"), (64, "r24w")]  # the ones that are built
REG = re.compile(r"\b([vs])(?:(\d+)|\[(\d+):(\d+)\])")


def regs(text):
    out = set()
    for m in REG.finditer(text):
        lo, hi = (int(m.group(2)),) * 2 if m.group(2) is not None else (int(m.group(3)), int(m.group(4)))
        out.update(f"{m.group(1)}{i}" for i in range(lo, hi + 1))
    return out


def read_lines(path):
    return [ln.strip()[1:].split("\\n")[0] for ln in path.read_text().splitlines() if ln.startswith('"')]


def generate(tmp_path, d, loader, generator=os.path.join(CSRC, "gen_prefill_loop.py")):
    out = tmp_path / f"loop_{d}_{loader}.inc"
    subprocess.run([sys.executable, generator, str(d), loader, str(out)], check=True, capture_output=True)
    lines = read_lines(out)
    clob = re.findall(r'"([^"]+)"', (tmp_path / f"loop_{d}_{loader}_clobbers.inc").read_text())
    return lines, set(clob)


def asm_operands(d, loader):
    """(in/out registers, input-only registers) of the asm statement in tpa_prefill.hip that includes the loop"""
    src = open(os.path.join(CSRC, "tpa_prefill.hip")).read()
    start = src.index(f'#include "gen/prefill_loop_{d}_{loader}.inc"')
    stmt = src[start : src.index(");", start)]
    outs, ins, _ = stmt.split("\n            :")[1:4] if stmt.count("\n            :") >= 3 else (None, None, None)
    assert outs is not None, "operand list of the asm statement not found"
    inout = set().union(*(regs(c) for c in re.findall(r'"\+\{([^}]+)\}"', outs)))
    assert not re.findall(r'"=\{', outs), "write-only operands are not expected"
    inputs = set().union(*(regs(c) for c in re.findall(r'"\{([^}]+)\}"', ins)))
    return inout, inputs


def dst_and_src(line):
    """(registers written, registers read) of one instruction line, None for labels and control flow"""
    if line.endswith(":") or line.startswith(("s_nop", "s_waitcnt", "s_barrier", "s_branch", "s_cbranch")):
        return None
    op, _, rest = line.partition(" ")
    opnds = [o.strip() for o in rest.split(",")]
    opnds = [o.split(" offset:")[0].replace(" offen", "") for o in opnds]
    if op.startswith(("ds_write", "s_cmp")):
        return set(), set().union(*(regs(o) for o in opnds))
    if op.startswith("v_cmp"):
        return {"vcc"}, set().union(*(regs(o) for o in opnds[1:]))
    if op.startswith("v_permlane32_swap"):
        both = regs(opnds[0]) | regs(opnds[1])
        return both, both
    return regs(opnds[0]), set().union(*(regs(o) for o in opnds[1:])) if len(opnds) > 1 else set()


@pytest.mark.parametrize("d,loader", LOOPS)
def test_generated_loop_matches_its_asm_statement(tmp_path, d, loader):
    lines, clob = generate(tmp_path, d, loader)
    inout, inputs = asm_operands(d, loader)
    assert {"vcc", "scc", "memory"} <= clob
    clob_regs = {c for c in clob if REG.fullmatch(c)}
    assert not (inout & inputs) and not (clob_regs & (inout | inputs)), "an operand is listed twice"
    defined = set(inout) | set(inputs)
    n_mfma = 0
    for ln in lines:
        ds = dst_and_src(ln)
        if ds is None:
            continue
        dst, src = ds
        n_mfma += ln.startswith("v_mfma")
        for r in dst | src:
            if r != "vcc":
                assert int(r[1:]) < (256 if r[0] == "v" else 102), f"{r} in `{ln}`"
        assert not (dst & inputs), f"`{ln}` writes an input-only operand"
        stray = {r for r in dst if r != "vcc"} - inout - clob_regs
        assert not stray, f"`{ln}` writes {sorted(stray)}: neither an in/out operand nor a clobber"
        undefined = {r for r in src if r != "vcc"} - defined
        assert not undefined, f"`{ln}` reads {sorted(undefined)} before anything wrote them"
        defined |= dst
    # two copies of the iteration (tile parity), one workgroup barrier each, and the matrix instructions of two tiles
    assert sum(ln == "s_barrier" for ln in lines) == 2
    assert n_mfma == 2 * (2 * (d // 16) + 4 * (d // 32))
    # every clobbered register is really used (a stale clobber would hide a register the compiler could have)
    used = set()
    for ln in lines + read_lines(tmp_path / f"loop_{d}_{loader}_rare.inc"):
        ds = dst_and_src(ln)
        if ds:
            used |= ds[0] | ds[1]
    assert clob_regs <= used, sorted(clob_regs - used)


@pytest.mark.parametrize("d,loader", LOOPS)
def test_a_nan_does_not_take_the_rare_path(tmp_path, d, loader):
    """Whatever branches to a rare path does so on an ordered comparison `slack < sum`: false for NaN, true for an overflow."""
    lines, _ = generate(tmp_path, d, loader)
    branches = [i for i, ln in enumerate(lines) if ln.startswith("s_cbranch_vccnz .Lpf_rare_")]
    assert len(branches) == (8 if loader.startswith("r2") else 4)  # two parities, a group per block (rank 2: two)
    for i in branches:
        writer = next(ln for ln in reversed(lines[:i]) if (dst_and_src(ln) or (set(),))[0] & {"vcc"})
        assert re.fullmatch(r"v_cmp_lt_f32 vcc, s64, v\d+", writer), writer


def rare_paths(lines):
    """label -> instructions, of the lines of the second file"""
    assert lines[-1] == ".Lpf_out_%=:"
    paths, label = {}, None
    for ln in lines[:-1]:
        if ln.endswith(":"):
            label = ln[:-1]
            assert label.startswith((".Lpf_rare_", ".Lpf_full_")) and label not in paths
            paths[label] = []
        else:
            paths[label].append(ln)
    return paths


def check_rare_paths(lines, rare, clob, inout, inputs, n_mfma):
    """the rules of the loop for each rare path, with what is defined where the loop branches to it"""
    clob_regs = {c for c in clob if REG.fullmatch(c)}
    paths, defined = rare_paths(rare), set(inout) | set(inputs)
    entered = []
    for i, ln in enumerate(lines):
        if ln.startswith("s_cbranch_vccnz .Lpf_rare_"):
            label = ln.split()[1]
            back = label.replace("_rare_", "_cont_")
            entered.append(label)
            assert lines[i + 1] == back + ":" and lines.count(back + ":") == 1, "a path returns behind its branch"
            full = label.replace("_rare_", "_full_")
            entered.append(full)
            for path, matrix in ((paths[label], 0), (paths[full], n_mfma)):
                # the first goes on to the second where the sum may have overflowed, before it has written anything
                assert path[-1] == "s_branch " + back and sum(x.startswith("v_mfma") for x in path) == matrix
                head = [x for x in path[:2] if path is paths[label]]
                if head:
                    assert re.fullmatch(r"v_cmp_lt_f32 vcc, 0x7e800000, v\d+", head[0]) and head[1] == "s_cbranch_vccnz " + full
                assert not any(x.startswith(("s_cbranch", "s_branch", "s_barrier", "buffer_", "ds_write")) for x in path[len(head):-1])
            for path, known in ((paths[label], set(defined)), (paths[full], set(defined))):
                for x in path:
                    dst, src = dst_and_src(x) or (set(), set())
                    dst, src = ({r for r in rs if not r.startswith("vcc")} for rs in (dst, src))
                    assert all(int(r[1:]) < (256 if r[0] == "v" else 102) for r in dst | src), x
                    assert not dst & inputs, f"`{x}` writes an input-only operand"
                    assert not dst - inout - clob_regs, f"`{x}` writes {sorted(dst - inout - clob_regs)}: neither an in/out operand nor a clobber"
                    assert not src - known, f"`{x}` reads {sorted(src - known)} before anything wrote them"
                    known |= dst
        defined |= (dst_and_src(ln) or (set(),))[0]
    assert sorted(entered) == sorted(paths), "each path is entered from one place"


@pytest.mark.parametrize("d,loader", LOOPS)
def test_rare_paths_match_the_asm_statement(tmp_path, d, loader):
    lines, clob = generate(tmp_path, d, loader)
    rare = read_lines(tmp_path / f"loop_{d}_{loader}_rare.inc")
    operands = asm_operands(d, loader)
    check_rare_paths(lines, rare, clob, *operands, n_mfma=d // 16)
    inout, inputs = operands
    unlisted = next(f"v{i}" for i in range(255, 0, -1) if f"v{i}" not in inout | inputs | clob)
    at = next(i for i, ln in enumerate(rare) if ln.startswith("v_max_f32"))
    op, dst, src = re.fullmatch(r"(v_max_f32) (v\d+), (.*)", rare[at]).groups()
    for planted, what in ((f"{op} {unlisted}, {src}", "neither"), (f"{op} {dst}, {unlisted}, {unlisted}", "before anything"),
                          (f"{op} {sorted(inputs & regs('v[0:255]'))[0]}, {src}", "input-only"), ("s_barrier", None)):
        with pytest.raises(AssertionError, match=what):
            check_rare_paths(lines, rare[:at] + [planted] + rare[at:], clob, *operands, n_mfma=d // 16)


def test_a_register_of_the_rare_paths_alone_is_a_clobber(tmp_path):
    """Head size 64 with eight waves has one loader pass and leaves a temporary unused in the loop; a rare path that wrote it would
    have to say so."""
    text = open(os.path.join(CSRC, "gen_prefill_loop.py")).read()
    assert text.count("    addr = set_address(e, t1)\n") == 1
    planted = text.replace("    addr = set_address(e, t1)\n", '    addr = set_address(e, t1)\n    e.ins("v_mov_b32", f"v{AAK1}", "0")\n')
    (tmp_path / "gen.py").write_text(planted)
    lines, clob = generate(tmp_path, 64, "r2", str(tmp_path / "gen.py"))
    written = {ln.split()[1].rstrip(",") for ln in read_lines(tmp_path / "loop_64_r2_rare.inc") if ln.startswith("v_mov_b32") and ln.endswith(", 0")}
    assert len(written) == 1 and written <= clob and not any(written & regs(ln) for ln in lines)


@pytest.mark.parametrize("d,loader", LOOPS)
def test_a_growing_row_is_not_computed_again(tmp_path, d, loader):
    """A sum that left the slack without an overflow moves the reference by what is in the registers: no matrix instruction, no
    operand from LDS, no exponential but the factor's, and with the maximum of the logits of the tile that are complete and still to
    come (of the second block, of a lane's other eight), or a row that grows would be back for them at the next group."""
    generate(tmp_path, d, loader)
    maxima = []
    for label, path in rare_paths(read_lines(tmp_path / f"loop_{d}_{loader}_rare.inc")).items():
        if "_rare_" in label:
            assert not any(ln.startswith(("v_mfma", "ds_")) for ln in path), label
            assert sum(ln.startswith("v_exp") for ln in path) == 1, label
            maxima.append(sum(ln.startswith(("v_max_f32", "v_max3_f32")) and ln.count(" v") >= 3 for ln in path))
    # 2 and more two-operand ones combine lanes and maxima; 8 for 16 logits, 4 for 8
    want = [2 + 8, 1] * 2 if not loader.startswith("r2") else [2 + 4, 2 + 8] * 4
    assert [m >= w for m, w in zip(maxima, want)] == [True] * len(want) and len(maxima) == len(want), maxima


def test_generator_takes_no_environment_input():
    """The product generator is a function of its arguments only (experiment switches live elsewhere)."""
    text = open(os.path.join(CSRC, "gen_prefill_loop.py")).read()
    assert "environ" not in text and "getenv" not in text
