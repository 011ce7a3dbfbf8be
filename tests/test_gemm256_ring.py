"""The LDS ring of the 256 x 256 tiles (madi_amd/csrc/gemm256.hip), on the CPU:
the order of DMAs, waits, barriers and fragment reads of its two groups of
waves, restated here, for streams of one chunk and up.  Every unit has landed
for all waves before any of them reads it, and no slot is written while a wave
may still read it."""
import itertools
import os
import subprocess

import pytest

from isa_vmcnt import hazards, kernels
from test_isa_vmcnt import HIPCC, ROOT

SRC = os.path.join(ROOT, "madi_amd", "csrc", "gemm256.hip")
UNITS = 5


class Wave:
    """One wave of group wm over `tiles` tiles of nk chunks: its events in
    program order, split at the barriers."""

    def __init__(self, wm, nk, tiles, ahead_wait=4, prologue_wait=12):
        self.phases = [[]]
        total = nk * tiles
        at = {"A": 0, "W": 0}  # the load cursors
        sa, first, ahead = 0, True, False

        def event(*e):
            self.phases[-1].append(e)

        def live(op):
            return at[op] < total

        def dma(op, slot):
            event("dma", (op, at[op]), slot % UNITS, 4)

        def meet():
            self.phases.append([])

        for u in range(UNITS):
            op = "W" if u & 1 else "A"
            if live(op):
                dma(op, u)
                ahead = ahead or u == 4
            at[op] += 1
        event("wait", prologue_wait if ahead else 0)
        meet()
        if wm == 1:
            meet()
        chunk = 0
        for _ in range(tiles):
            for _ in range(nk):
                if live("W") and not first:
                    dma("W", sa + 3)
                event("read", ("A", chunk), sa)
                event("read", ("W", chunk), (sa + 1) % UNITS)
                at["W"] += not first
                meet()
                meet()
                if live("A") and not first:
                    dma("A", sa + 4)
                event("read", ("A", chunk), sa)
                event("read", ("W", chunk), (sa + 1) % UNITS)
                if not first:
                    ahead = live("A")
                    at["A"] += 1
                first = False
                if wm == 1:
                    event("wait", ahead_wait if ahead else 0)
                meet()
                if wm == 0:
                    event("wait", ahead_wait if ahead else 0)
                meet()
                sa = (sa + 2) % UNITS
                chunk += 1
            event("stage", (sa + 4) % UNITS)
            event("store", 16)
        if wm == 0:
            meet()


def faults(nk, tiles, **waits):
    waves = [Wave(wm, nk, tiles, **waits) for wm in (0, 1)]
    if len(waves[0].phases) != len(waves[1].phases):
        return ["the groups meet a different number of times"]
    bad = []
    queue = [[], []]     # outstanding vector-memory operations, in issue order
    landed = [{}, {}]    # unit -> the phase in which this wave waited for it
    held = [None] * UNITS  # the unit a slot was last written with
    reads = {}           # slot -> (last phase it was read or staged in)
    writes = {}          # slot -> the phase its DMAs were issued in, by wave
    for phase, events in enumerate(zip(*(w.phases for w in waves))):
        # within a phase the groups run in any order
        other = [{e[2] for e in events[1 - wm] if e[0] == "read"} for wm in (0, 1)]
        for wm, e in itertools.chain(*([(wm, e) for e in ev] for wm, ev in enumerate(events))):
            kind = e[0]
            if kind == "dma":
                _, unit, slot, ops = e
                if (reads.get(slot, -1) >= phase or slot in other[wm]) and held[slot] != unit:
                    bad.append(f"phase {phase}: {unit} over a slot that is being read")
                held[slot] = unit
                writes[slot] = phase
                queue[wm] += [unit] * ops
            elif kind == "store":
                queue[wm] += [None] * e[1]
            elif kind == "wait":
                done = queue[wm][:max(0, len(queue[wm]) - e[1])]
                queue[wm] = queue[wm][len(done):]
                for unit in done:
                    landed[wm][unit] = phase
            elif kind == "read":
                _, unit, slot = e
                if held[slot] != unit:
                    bad.append(f"phase {phase}: slot {slot} holds {held[slot]}, not {unit}")
                for o in (0, 1):
                    if unit in queue[o] or not landed[o].get(unit, phase) < phase:
                        bad.append(f"phase {phase}: {unit} read before it has landed")
                reads[slot] = max(reads.get(slot, -1), phase)
            elif kind == "stage":  # the wave's own part of the last W slot
                slot = e[1]
                if reads.get(slot, -1) >= phase or slot in other[wm]:
                    bad.append(f"phase {phase}: staged in a slot that is being read")
                if held[slot][0] != "W" or writes[slot] >= phase:
                    bad.append(f"phase {phase}: staged in a slot that is being filled")
    if any(queue[wm] and any(u for u in queue[wm]) for wm in (0, 1)):
        bad.append("a DMA is in flight at the end")
    return bad


@pytest.mark.parametrize("nk,tiles", [(nk, t) for nk in (1, 2, 3, 4, 5, 20) for t in (1, 2, 3, 8)])
def test_ring_is_race_free(nk, tiles):
    assert not faults(nk, tiles), (nk, tiles, faults(nk, tiles)[:4])


def test_planted_mistakes_are_found():
    for nk, tiles in ((3, 2), (20, 1)):
        assert faults(nk, tiles, ahead_wait=8)
        assert faults(nk, tiles, prologue_wait=16)


def test_counts_are_the_kernels():
    src = open(SRC).read()
    assert f"kUnits = {UNITS};" in src
    for text in ('s_waitcnt vmcnt(4)', "wait_then_barrier<12>()", "dma_w(wrap(sa + 3))", "dma_a(wrap(sa + 4))"):
        assert src.count(text) == 1, text


def test_every_instance_is_race_free(tmp_path):
    """No register is touched while a load into it is in flight."""
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    from madi_amd.build import HIP_FLAGS
    out = tmp_path / "gemm256.s"
    subprocess.run([HIPCC, *(f for f in HIP_FLAGS if f != "-fPIC"), "--cuda-device-only", "-S", SRC,
                    "-o", str(out)], check=True, capture_output=True)
    asm = kernels(out.read_text())
    assert sum("q8_gemm256_kernel" in n for n in asm) == 3, list(asm)
    assert not {n: b for n, body in asm.items() if (b := hazards(body)[:3])}
