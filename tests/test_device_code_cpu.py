"""Properties of the compiled device code that no run shows reliably: the wait
states between dependent vector instructions, which the compiler keeps for its
own instructions but not for those written as inline assembly (it schedules
without looking inside), and the registers that the traversals are written to
fit in."""
import functools
import os
import re
import subprocess
from pathlib import Path

import pytest

from torchbvh_amd import _build

_SOURCES = [s for s in _build.SOURCES if s != "capi.hip"]  # capi.hip has no kernels


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    """The gfx950 assembly of every source, compiled as the library is."""
    try:
        command = _build.compile_command()
    except RuntimeError:
        pytest.skip("hipcc not found")
    flags = command[:command.index("-o")]
    flags.remove("-shared")
    folder = tmp_path_factory.mktemp("assembly")
    paths = {s: folder / (Path(s).stem + ".asm") for s in _SOURCES}
    running, todo = [], sorted(_SOURCES, key=lambda s: -(_build.CSRC / s).stat().st_size)
    while todo or running:
        while todo and len(running) < min(8, os.cpu_count() or 1):
            s = todo.pop(0)
            running.append((s, subprocess.Popen(
                [*flags, "--cuda-device-only", "-S", "-o", str(paths[s]), str(_build.CSRC / s)],
                stdout=subprocess.DEVNULL, stderr=subprocess.PIPE, text=True)))
        s, process = running.pop(0)
        _, errors = process.communicate()
        assert process.returncode == 0, f"{s}:\n{errors}"
    return {s: p.read_text() for s, p in paths.items()}


_REGISTER = re.compile(r"(?<![\w.])([vs])(?:(\d+)|\[(\d+):(\d+)\])(?!\w)|(?<![\w.])(vcc)(_lo|_hi)?(?!\w)")


@functools.lru_cache(maxsize=None)
def _registers(operand: str) -> frozenset:
    found = set()
    for m in _REGISTER.finditer(operand):
        if m.group(5):
            found |= {"vcc" + h for h in ((m.group(6),) if m.group(6) else ("_lo", "_hi"))}
        elif m.group(2):
            found.add(m.group(1) + m.group(2))
        else:
            found |= {m.group(1) + str(i) for i in range(int(m.group(3)), int(m.group(4)) + 1)}
    return frozenset(found)


class _Instruction:
    __slots__ = ("text", "op", "defs", "uses", "select", "labels", "states")

    def __init__(self, text: str, labels: list):
        self.text, self.labels = text, labels
        self.op, _, rest = text.partition(" ")
        operands = [o.strip() for o in re.split(r",(?![^\[]*\])", rest)] if rest else []
        self.states = int(operands[0], 0) + 1 if self.op == "s_nop" else 1
        vector = self.op.startswith("v_")
        results = 0
        if vector or self.op.startswith("s_"):
            # Carry and divide-scale forms also write a mask; swaps write both.
            results = 2 if re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co|v_div_scale|v_mad_[ui]64|"
                                    r"v_permlane(16|32)_swap|v_swap", self.op) else 1
        self.defs = frozenset().union(*map(_registers, operands[:results]))
        self.uses = frozenset().union(*map(_registers, operands[results:]))
        if vector and (results == 2 and "swap" in self.op or "fmac" in self.op or "dpp" in self.op):
            self.uses |= self.defs
        # The lane select of v_readlane and v_writelane.
        self.select = _registers(operands[-1]) if re.match(r"v_(read|write)lane", self.op) else frozenset()


def _kernels(assembly: str):
    """The instructions of each function, in order, with the labels before them."""
    body, labels = [], []
    for line in assembly.splitlines():
        line = line.split(";")[0].split("//")[0].strip()
        label = re.match(r"([\w.$]+):", line)
        if label:
            if not label.group(1).startswith(".L"):
                if body:
                    yield body
                body = []
            labels.append(label.group(1))
        elif re.match(r"(v|s|ds|global|buffer|flat|scratch)_", line):
            body.append(_Instruction(line, labels))
            labels = []
    if body:
        yield body


def _wait_states(use: _Instruction, register: str) -> int:
    """Wait states that `use` needs after a vector instruction that wrote `register`."""
    if not use.op.startswith("v_"):
        return 0
    if re.match(r"v\d", register):
        if re.match(r"v_read(first)?lane", use.op):
            return 1
        if use.op.startswith("v_permlane") or re.search(r"quad_perm|row_|wave_", use.text):
            return 2
        return 0
    return 4 if register in use.select or use.op.startswith("v_div_fmas") else 2


def _missing_waits(body: list) -> list:
    at = {label: i for i, instruction in enumerate(body) for label in instruction.labels}
    jumps = {}
    for i, instruction in enumerate(body):
        target = re.match(r"s_c?branch\w*\s+(\S+)", instruction.text)
        if target and target.group(1) in at:
            jumps.setdefault(at[target.group(1)], []).append(i)
    missing = []
    for i, use in enumerate(body):
        for register in use.uses:
            needed = _wait_states(use, register)
            todo, seen = ([(i, 0)] if needed else []), set()
            while todo:
                j, passed = todo.pop()
                before = list(jumps.get(j, ()))
                if j > 0 and not re.match(r"s_(branch|endpgm|setpc)", body[j - 1].op):
                    before.append(j - 1)
                for p in before:
                    if register in body[p].defs:
                        if body[p].op.startswith("v_"):
                            missing.append(f"{body[p].text} -> {use.text}: {passed} of {needed}")
                        continue
                    state = (p, passed + body[p].states)
                    if state[1] < needed and state not in seen:
                        seen.add(state)
                        todo.append(state)
    return missing


def test_checker_finds_a_missing_wait():
    body = next(_kernels("k:\n v_readlane_b32 s4, v1, 3\n v_readlane_b32 s5, v2, 3\n v_max_f64 v[0:1], v[0:1], s[4:5]\n"))
    assert len(_missing_waits(body)) == 2
    body = next(_kernels("k:\n v_readlane_b32 s4, v1, 3\n s_nop 1\n v_add_u32 v0, s4, v0\n s_nop 0\n v_readlane_b32 s6, v0, 1\n"))
    assert _missing_waits(body) == []


@pytest.mark.parametrize("source", _SOURCES)
def test_wait_states_between_dependent_vector_instructions(assembly, source):
    missing = [m for body in _kernels(assembly[source]) for m in _missing_waits(body)]
    assert not missing, f"{len(missing)} sites, e.g. {missing[:3]}"


def _vector_registers(assembly: str, kernel: str) -> dict:
    """{template arguments: allocated VGPRs} of the kernels of that name."""
    found = {}
    for name, body in re.findall(r"\.amdhsa_kernel (\S+)\n(.*?)\.end_amdhsa_kernel", assembly, re.S):
        arguments = re.search(rf"\d{kernel}I((?:L[ib]\d+E)+)E", name)
        if arguments:
            key = tuple(int(x) for x in re.findall(r"L[ib](\d+)E", arguments.group(1)))
            found[key] = int(re.search(r"\.amdhsa_next_free_vgpr (\d+)", body).group(1))
    return found


# Waves per SIMD (512 registers in all, allocated in eights).
@pytest.mark.parametrize("dim,k,waves", [(2, 4, 7), (2, 8, 8), (2, 16, 4), (2, 32, 4),
                                         (3, 4, 7), (3, 8, 7), (3, 16, 4), (3, 32, 3)])
def test_implicit_tree_traversal_keeps_its_occupancy(assembly, dim, k, waves):
    registers = _vector_registers(assembly["knn.hip"], "knn_kernel")
    for ordered in (0, 1):  # (D, K, ordered, ragged, routed)
        used = registers[(dim, k, ordered, 0, 0)]
        assert 512 // (-(-used // 8) * 8) >= waves, used


@pytest.mark.parametrize("dim,k,compact,waves", [(2, 8, 0, 8), (3, 8, 0, 7), (3, 16, 0, 6), (3, 16, 1, 6), (3, 32, 0, 4)])
def test_accel_traversal_keeps_its_occupancy(assembly, dim, k, compact, waves):
    registers = _vector_registers(assembly["knn.hip"], "knn_accel_kernel")
    for ordered in (0, 1):  # (D, K, ordered, ragged, routed, compact)
        used = registers[(dim, k, ordered, 0, 0, compact)]
        assert 512 // (-(-used // 8) * 8) >= waves, used


def test_schedule_refinement_fits_two_work_groups_per_cu(assembly):
    """Work-groups of 16 waves: eight waves per SIMD, 64 registers."""
    body = re.search(r"\.amdhsa_kernel \S*refine_kernel\S*\n(.*?)\.end_amdhsa_kernel", assembly["small.hip"], re.S).group(1)
    assert int(re.search(r"\.amdhsa_next_free_vgpr (\d+)", body).group(1)) <= 64
    assert int(re.search(r"\.amdhsa_private_segment_fixed_size (\d+)", body).group(1)) == 0
