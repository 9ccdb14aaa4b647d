"""Hazards in the kernels' gfx950 assembly that the compiler leaves to inline assembly.

The compiler inserts the wait states that an instruction needs after an earlier one, but it
does not look inside inline assembly, where the kernels issue their LDS-DMA. The device code
is compiled here with the library's flags (no GPU needed) and read instruction by instruction.
"""

from __future__ import annotations

import importlib.util
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import pytest

REPO_ROOT = Path(__file__).resolve().parents[1]


def _load_build():
    path = REPO_ROOT / "flash_attention_2_lab_amd" / "_build.py"
    spec = importlib.util.spec_from_file_location("fa2_build", path)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


build = _load_build()

pytestmark = pytest.mark.skipif(not Path(build.HIPCC).exists(), reason="needs ROCm hipcc")


def _instructions(text: str) -> dict[str, list[str]]:
    """The instructions of every kernel, in order; labels, directives and comments left out."""
    kernels: dict[str, list[str]] = {}
    current: list[str] = []
    for line in text.splitlines():
        line = line.split(";")[0].rstrip()
        name = re.match(r"(_Z\w+):", line)
        if name:
            current = kernels.setdefault(name.group(1), [])
        elif line.startswith("\t") and line.strip() and not line.strip().startswith("."):
            current.append(line.strip())
    return {name: body for name, body in kernels.items() if any(i.startswith("s_endpgm") for i in body)}


@pytest.fixture(scope="module")
def kernels(tmp_path_factory) -> dict[str, list[str]]:
    out = tmp_path_factory.mktemp("assembly")

    def compile_one(source: str) -> dict[str, list[str]]:
        target = out / (source + ".s")
        subprocess.run([build.HIPCC, *build.HIP_FLAGS, "--cuda-device-only", "-S", f"-I{build.INCLUDE}",
                        str(build.CSRC / source), "-o", str(target)], check=True, capture_output=True, timeout=300)
        return _instructions(target.read_text())

    with ThreadPoolExecutor(max_workers=2) as pool:
        return {name: body for part in pool.map(compile_one, build.KERNEL_SOURCES) for name, body in part.items()}


def _scalars(operands: str) -> set[str]:
    """The scalar registers named in an operand text."""
    found = set(re.findall(r"\b(?:m0|vcc|s\d+)\b", operands))
    for low, high in re.findall(r"\bs\[(\d+):(\d+)\]", operands):
        found.update(f"s{i}" for i in range(int(low), int(high) + 1))
    return found


def _written(instruction: str) -> set[str]:
    parts = instruction.split(None, 1)
    return _scalars(parts[1].split(",")[0]) if len(parts) == 2 else set()


def _states_since(body: list[str], at: int, writes, limit: int) -> int:
    """Wait states between the instruction at `at` and the last one before it that `writes`."""
    states = 0
    for past in reversed(body[max(0, at - limit - 1):at]):
        if writes(past):
            return states
        states += int(past.split()[1], 0) + 1 if past.startswith("s_nop") else 1
    return limit


def test_lds_dma_waits_for_m0_and_its_scalar_operands(kernels):
    """One wait state from a scalar write of M0 to an LDS-DMA, which takes its LDS address from
    it; five from a VALU write of a scalar register to a buffer access that reads it."""
    fetches = 0
    for name, body in kernels.items():
        for at, instruction in enumerate(body):
            if not instruction.startswith("buffer_"):
                continue
            if instruction.endswith(" lds"):
                fetches += 1
                gap = _states_since(body, at, lambda past: past.startswith("s_") and "m0" in _written(past), 1)
                assert gap >= 1, f"{name}: no wait state before {instruction}"
            read = _scalars(instruction.split(None, 1)[1])
            gap = _states_since(body, at, lambda past: past.startswith("v_") and bool(_written(past) & read), 5)
            assert gap >= 5, f"{name}: {gap} wait states before {instruction}"
    assert fetches > 1000  # every LDS-DMA kernel was read


def test_scores_barriers_wait_for_lds_reads(kernels):
    """Behind each barrier of the scores kernel another wave's LDS-DMA refills the ring slot that
    this wave read before it, so the wave waits for its reads at the barrier itself."""
    scores = {name: body for name, body in kernels.items() if "scores_f32_kernel" in name}
    assert scores
    for name, body in scores.items():
        barriers = [at for at, instruction in enumerate(body) if instruction == "s_barrier"]
        assert barriers
        for at in barriers:
            wait = body[at - 1]
            assert wait.startswith("s_waitcnt") and "lgkmcnt(0)" in wait, f"{name}: {wait}"
