"""Orders that the device code has to keep by itself, read from the assembly that hipcc makes of it for gfx950 (no GPU).

The weight rings in LDS (experts_mfma.hip, experts_stream.hip): LDS DMA issued from inline assembly refills the slot that
the wave has just read, and neither the compiler nor the hardware orders the two.  On every path to such a DMA, each LDS
read before it has to be followed by a wait that the source states (inline assembly, or a work-group barrier); a wait
that the compiler happened to place for the read's use does not count."""
import pathlib
import re
import subprocess
import sys

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "xestrata-win_amd" / "csrc"


def functions(text):
    """(name, [(instruction, whether it is inline assembly)]) of each function, labels among the instructions."""
    name, body, inline = None, [], False
    for line in text.splitlines():
        m = re.match(r"^(_Z\w+):", line)
        if m:
            name, body, inline = m.group(1), [], False
        elif line.startswith(".Lfunc_end") and name:
            yield name, body
            name = None
        elif name:
            if "#ASMSTART" in line or "#ASMEND" in line:
                inline = "#ASMSTART" in line
                continue
            s = line.split(";")[0].strip()
            if s and (not s.startswith(".") or s.endswith(":")):
                body.append((s, inline))


def unordered_dmas(body):
    """The LDS DMA instructions that a path with an LDS read not waited for by the source reaches, and all of them."""
    blocks, labels = [[]], {}
    for s, inline in body:
        if s.endswith(":"):
            blocks.append([])
            labels[s[:-1]] = len(blocks) - 1
            continue
        blocks[-1].append((s, inline))
        if re.match(r"s_(c?branch|endpgm)", s):
            blocks.append([])
    nexts = []
    for i, b in enumerate(blocks):
        last = b[-1][0] if b else ""
        m = re.match(r"s_(c?)branch\w*\s+(\S+)", last)
        to = [labels[m.group(2)]] if m else []
        if not last.startswith("s_endpgm") and (not m or m.group(1)):
            to.append(i + 1)
        nexts.append([j for j in to if j < len(blocks)])

    def walk(i, reads, bad=None):
        for s, inline in blocks[i]:
            if s.startswith("ds_read"):
                reads = True
            elif s.startswith("s_barrier") or (inline and "s_waitcnt" in s and "lgkmcnt(0)" in s):
                reads = False
            elif bad is not None and s.startswith("global_load_lds") and reads:
                bad.append(s)
        return reads

    entry = [False] * len(blocks)
    work = list(range(len(blocks)))
    while work:
        i = work.pop()
        out = walk(i, entry[i])
        for j in nexts[i]:
            if out and not entry[j]:
                entry[j] = True
                work.append(j)
    bad = []
    for i in range(len(blocks)):
        walk(i, entry[i], bad)
    return bad, sum(s.startswith("global_load_lds") for b in blocks for s, _ in b)


@pytest.mark.parametrize("source,kernel", [("experts_mfma.hip", "rows_mfma_kernel"), ("experts_stream.hip", "stream_kernel")])
def test_ring_reads_return_before_the_slot_is_refilled(source, kernel, tmp_path):
    sys.path.insert(0, str(CSRC.parent))
    import build
    asm = tmp_path / "k.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S", "-o", str(asm), str(CSRC / source)], check=True,
                   capture_output=True)
    seen = 0
    for name, body in functions(asm.read_text()):
        if kernel not in name:
            continue
        bad, dmas = unordered_dmas(body)
        assert dmas > 0 and not bad, (name, bad)
        seen += 1
    assert seen > 0


def test_the_check_sees_a_missing_wait():
    """The path analysis itself, on a loop whose read of one round meets the DMA of the next."""
    loop = [(".LBB0_1:", False), ("global_load_lds_dwordx4 v[0:1], off", True), ("ds_read_b32 v2, v3", False),
            ("s_waitcnt lgkmcnt(0)", False), ("s_cbranch_scc1 .LBB0_1", False), ("s_endpgm", False)]
    assert len(unordered_dmas(loop)[0]) == 1
    for wait in (("s_waitcnt lgkmcnt(0)", True), ("s_barrier", False)):
        assert unordered_dmas(loop[:1] + [wait] + loop[1:]) == ([], 1)


def test_chain_accumulators_are_apart_from_their_operands(tmp_path):
    """gemv.hip's 16-step chains write their accumulator before they have read all of their operands, so it shares no
    register with one (an early-clobber operand: without it the compiler may share one of equal value)."""
    sys.path.insert(0, str(CSRC.parent))
    import build
    asm = tmp_path / "k.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S", "-o", str(asm), str(CSRC / "gemv.hip")], check=True,
                   capture_output=True)
    runs = 0
    for block in asm.read_text().split("#ASMSTART")[1:]:
        regs = re.findall(r"v_fmac_f32_dpp (v\d+), (v\d+), (v\d+)", block.split("#ASMEND")[0])
        if regs:
            assert len(regs) == 16 and len({d for d, _, _ in regs}) == 1
            assert all(d not in (a, b) for d, a, b in regs), regs
            runs += 1
    assert runs > 0
    assert '"+&v"(acc)' in (CSRC / "gemv.hip").read_text()
