"""Rules on the kernels' sources that no run can show (no GPU)."""

from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "claudemaxing_amd" / "csrc"


def test_workgroup_barriers_are_fenced():
    """The barrier instruction is no memory access to the compiler: without a fence on either side it
    may move an LDS read of the next tile above the barrier, or of the last one below it."""
    found = 0
    for path in sorted([*CSRC.glob("*.h"), *CSRC.glob("*.hip")]):
        lines = [ln.strip() for ln in path.read_text().splitlines()]
        for i, line in enumerate(lines):
            if not line.startswith("__builtin_amdgcn_s_barrier("):
                continue
            found += 1
            where = f"{path.name}:{i + 1}"
            assert lines[i - 1].startswith("__builtin_amdgcn_fence(__ATOMIC_RELEASE"), where
            assert lines[i + 1].startswith("__builtin_amdgcn_fence(__ATOMIC_ACQUIRE"), where
    assert found
