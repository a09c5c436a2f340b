"""Matrix instructions written out by hand (c6_split.h: mma_vector): the compiler does not know what they are, so it
leaves no wait between one and an instruction of its own that reads or writes the sum.  Such a sum has to stay where it is from
the first of a layer's to the wait behind the last: read off the built library's own AMD assembly."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from connect6_amd import _lib

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
SPLIT = ["_ZN2c620split_forward_kernelINS_8PrecF32SEEEvNS_9FwdParamsE", "_ZN2c619half_forward_kernelINS_8PrecF32SEEEvNS_9FwdParamsE"]


def _listing(tmp_path, symbol):
    """The kernel's instructions: (address, text, address it may jump to or None)."""
    shutil.copy(_lib._SO, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    for part in sorted(tmp_path.glob("lib.so.*gfx950")):
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f"--disassemble-symbols={symbol}", part], check=True,
                             capture_output=True, text=True).stdout
        start = re.search(rf"^([0-9a-f]+) <{symbol}>:$", out, re.M)
        if start is None:
            continue
        lines = []
        for text, address, rest in re.findall(r"^\t(.+?)\s*// ([0-9A-F]+):(.*)$", out[start.end():], re.M):
            to = re.search(rf"<{symbol}(?:\+0x([0-9a-f]+))?>", rest)
            lines.append((int(address, 16), text, to and int(start[1], 16) + int(to[1] or "0", 16)))
        return lines
    raise AssertionError(f"{symbol} is in no part of the library")


def _vector(text):
    """Numbers of the vector registers that an instruction names."""
    named = set()
    for one, low, high in re.findall(r"\bv(?:(\d+)\b|\[(\d+):(\d+)\])", text):
        named |= {int(one)} if one else set(range(int(low), int(high) + 1))
    return named


def _layers(lines):
    """(first, wait, sums) per layer: from where the hand-written instructions' loop begins to the wait behind them, and the
    registers of their sums."""
    hand = [i for i, (_, text, _) in enumerate(lines) if re.match(r"v_mfma\S* v\[", text)]
    waits = [i for i in range(len(lines) - 1) if lines[i][1] == "s_nop 15" and lines[i + 1][1] == "s_nop 7"]
    found, done = [], 0
    for wait in waits:
        mine = [i for i in hand if done <= i < wait]
        at = {address: i for i, (address, _, _) in enumerate(lines)}
        # (a jump back in front of the first one: the loop over the taps, whose head runs behind its last one too)
        back = [at[to] for _, _, to in lines[mine[0]:wait] if to is not None and done <= at[to] < mine[0]]
        found.append((min(back + mine[:1]), wait, set().union(*[_vector(lines[i][1].split(",")[0]) for i in mine])))
        done = wait
    assert sum(done <= i for i in hand) == 0, "a sum without its wait"
    return found


def _moved(lines):
    """Instructions that touch a hand-written one's sum while it may still be written."""
    wrong = []
    for first, wait, sums in _layers(lines):
        for i in range(first, wait):
            text = lines[i][1]
            hand = re.match(r"v_mfma\S* (v\[\d+:\d+\]), (\S+), (\S+), (v\[\d+:\d+\])$", text)
            if hand is None:
                wrong += [text] if _vector(text) & sums or text.startswith(("s_swappc", "s_setpc")) else []
            elif hand[1] != hand[4] or (_vector(hand[2]) | _vector(hand[3])) & sums or lines[i - 1][1] != "s_nop 1":
                wrong.append(text)
    return wrong


@pytest.fixture(scope="module", params=SPLIT)
def split(tmp_path_factory, request):
    return _listing(tmp_path_factory.mktemp("split"), request.param)


def test_sums_of_hand_written_instructions_stay_in_their_registers(split):
    layers = _layers(split)
    # three layers of 96 outputs; the two sums of one tile, sixteen registers each
    assert len(layers) == 3 and all(len(sums) == 32 for _, _, sums in layers)
    for first, wait, _ in layers:
        hand = sum(text.startswith("v_mfma") and "v[" in text.split(",")[0] for _, text, _ in split[first:wait])
        assert hand in (24, 36)   # six per k-step of 16 channels: 64 and 96 inputs
    assert _moved(split) == []


@pytest.mark.parametrize("planted", ["v_mov_b32_e32 v{0}, v0", "scratch_store_dword off, v{0}, off", "ds_read_b128 v[{0}:{1}], v0",
                                     "v_accvgpr_write_b32 a0, v{1}", "v_mfma_f32_32x32x16_bf16 a[0:15], v[{0}:{1}], v[0:3], a[0:15]"])
@pytest.mark.parametrize("where", ["head", "middle", "end"])
def test_a_sum_that_moves_is_seen(split, planted, where):
    first, wait, sums = _layers(split)[1]
    low = min(sums)
    text = planted.format(low, low + 3)
    assert _vector(text) & sums
    at = {"head": first + 1, "middle": (first + wait) // 2, "end": wait - 1}[where]
    while split[at - 1][1] == "s_nop 1":   # (the pair of a wait state and its instruction stays one)
        at += 1
    assert text in _moved(split[:at] + [(split[at][0] - 1, text, None)] + split[at:])


# Where two ways meet, a copy of a constant or of a register in front of the instruction that brings the other lanes back is one
# that they do not get.  (The compiler has put such copies there in fp32 kernels whose registers were all in use.)
def _copies_for_some_lanes(lines):
    at = {address: i for i, (address, _, _) in enumerate(lines)}
    found = []
    for i in sorted({at[to] for _, text, to in lines if text.startswith("s_cbranch_execz") and to in at}):
        copies = []
        for _, text, _ in lines[i:]:
            if text.startswith("s_or_b64 exec, exec"):
                found += copies
            if "exec" in text or text.startswith(("s_branch", "s_cbranch", "s_endpgm", "s_setpc")):
                break
            if re.match(r"v_mov_b32|v_mov_b64|v_accvgpr|scratch_load|buffer_load_dword\S* .* off, s\[0:3\]", text):
                copies.append(text)
    return found


@pytest.mark.parametrize("kernel", ["19team_forward_kernelINS_8PrecF32SEEEvNS_10TeamParamsE",
                                    "19half_forward_kernelINS_8PrecF32SEEEvNS_9FwdParamsE",
                                    "20split_forward_kernelINS_8PrecF32SEEEvNS_9FwdParamsE"])
def test_no_copy_is_made_for_some_lanes_only(kernel, tmp_path):
    lines = _listing(tmp_path, "_ZN2c6" + kernel)
    assert _copies_for_some_lanes(lines) == []
    joins = [i for i, (address, text, _) in enumerate(lines) if text.startswith("s_or_b64 exec, exec") and
             any(to == address and other.startswith("s_cbranch_execz") for _, other, to in lines)]
    address, text, to = lines[joins[0]]
    planted = [(address, "v_mov_b32_e32 v1, 0x100", None), (address + 1, text, to)]
    assert _copies_for_some_lanes(lines[:joins[0]] + planted + lines[joins[0] + 1:]) == [planted[0][1]]
