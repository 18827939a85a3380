"""CPU check of the compiled LDS-DMA kernels: no wave passes a barrier with LDS
accesses of its own in flight.

These kernels pass an LDS stage on with a bare s_barrier behind which other
waves' DMA overwrites it. The compiler waits for an LDS read before its first
use, wherever that is; where it moved the uses past the barrier, the read could
still be in flight when the stage was overwritten (the float32 contraction once
reached its barrier so, five reads outstanding). The check walks the compiled
code: an upper bound of the LDS and scalar-memory operations in flight (they
share a counter), taken over every path, at each s_barrier."""

from __future__ import annotations

import re

import pytest

from tests import isa

SOURCES = ["fjx_contract.hip", "fjx_gemm_dma.hip", "fjx_flash_pipe.hip"]
CAP = 64


def _step(out: int, ins: str) -> int:
    if re.match(r"(ds_|s_load_|s_buffer_load_)", ins):
        return min(out + 1, CAP)
    m = re.match(r"s_waitcnt\b.*lgkmcnt\((\d+)\)", ins) if ins.startswith("s_waitcnt") else None
    return min(out, int(m.group(1))) if m else out


def worst_at_barriers(code: list[str]) -> list[int]:
    """For each s_barrier, the largest number of LDS and scalar-memory
    operations that can be in flight when a wave gets there."""
    labels = {c[:-1]: i for i, c in enumerate(code) if c.endswith(":")}
    state = {0: 0}  # in flight on entry, by line
    todo = [0]
    at: dict[int, int] = {}
    while todo:
        i = todo.pop()
        out = state[i]
        while i < len(code):
            ins = code[i]
            if ins == "s_barrier":
                at[i] = max(at.get(i, 0), out)
            out = _step(out, ins)
            nxt = [i + 1]
            m = re.match(r"s_(c?)branch\S*\s+(\S+)", ins)
            if m:
                nxt = [labels[m.group(2)]] + ([i + 1] if m.group(1) else [])
            elif ins.startswith("s_endpgm"):
                nxt = []
            for j in nxt[1:] if m else []:
                if state.get(j, -1) < out:
                    state[j] = out
                    todo.append(j)
            if not nxt:
                break
            j = nxt[0]
            if m or (j < len(code) and code[j].endswith(":")):
                if state.get(j, -1) >= out:
                    break
                state[j] = out
            i = j
    return [at[i] for i in sorted(at)]


def test_walk_counts_what_is_in_flight():
    code = ["ds_read_b128 v[0:3], v4", "ds_read_b128 v[0:3], v4", "s_waitcnt lgkmcnt(1)", "s_barrier",
            "s_cbranch_scc1 .L1", "s_waitcnt vmcnt(0) lgkmcnt(0)", "s_branch .L2", ".L1:", "ds_read_b32 v0, v1",
            ".L2:", "s_barrier", "s_endpgm"]
    assert worst_at_barriers(code) == [1, 2]


@pytest.mark.parametrize("src", SOURCES)
def test_no_lds_access_in_flight_at_a_barrier(src):
    checked = 0
    for name, code in isa.kernels(src).items():
        # operands that arrive by LDS DMA
        if not any(re.match(r"(buffer|global)_load\S*.*\blds\b", c) for c in code):
            continue
        worst = worst_at_barriers(code)
        assert worst, f"{name}: no barrier found"
        assert max(worst) == 0, f"{name}: {worst} LDS or scalar operations in flight at its barriers"
        checked += 1
    assert checked, f"no LDS-DMA kernel found in {src}"


def test_a_tiles_stores_follow_the_next_tiles_dma():
    """A tile's first wait leaves the previous tile's stores in flight, vmcnt(their
    number): it covers the DMA only if every store was issued after it, none is
    missing and nothing else was issued since."""
    checked = set()
    for src in ("fjx_contract.hip", "fjx_gemm_dma.hip"):
        for name, code in isa.kernels(src).items():
            dma = [i for i, c in enumerate(code) if re.match(r"(buffer|global)_load\S*.*\blds\b", c)]
            waits = [m for m in (re.match(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)", c) for c in code) if m]
            left = {int(m.group(1)) for m in waits} - {0}
            if not dma or not left:
                continue
            vmem = [i for i, c in enumerate(code) if re.match(r"(buffer|global|scratch|flat)_(load|store|atomic)", c)]
            after = [i for i in vmem if i > dma[-1]]
            stores = [i for i in vmem if "_store" in code[i]]
            assert left == {len(stores)} and after == stores, (name, left, len(stores), len(after))
            checked.add(re.search(r"contract_dma|contract_split|gemm_dma_pair|gemm_dma_planes", name).group())
    assert len(checked) == 4, checked
