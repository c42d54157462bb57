"""No rounding of the slice loop's kernels is the compiler's choice: which products enter a fused
multiply-add is written out, so the device code is the same with the compiler's own fusing off.  (Left
to it, moving a kernel's loads once changed the choice, and results with it.)  Compiles, no GPU."""
import os
import re
import shlex
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cltem_amd", "csrc")

# kernels outside the slice loop, whose double arithmetic, or scale before the first butterfly, is left
# to the compiler: row modes ROW_IFFT_INTENSITY and ROW_ADJ_SEED; column modes COL_PROBE, COL_FFT_DIFF,
# COL_CTEM_IMAGE and COL_FILTER
LEFT = {"k_row": {5, 6}, "k_col": {3, 5, 9, 10}}


def kernels(path):
    """Instructions of each kernel in an assembly file."""
    out, cur = {}, None
    with open(path) as f:
        for line in f:
            m = re.match(r"^(_Z\w+):", line)
            if m:
                cur = out.setdefault(m.group(1), [])
            elif line.startswith(".Lfunc_end"):
                cur = None
            elif cur is not None and re.match(r"^\t[a-z]", line):
                cur.append(line.split(";")[0].strip())
    return out


def mode(name):
    """("k_row" or "k_col", mode) of those kernels' instantiations, else None."""
    m = re.match(r"_ZN3mse5(k_row|k_col)INS_5Plan\dI(?:Li\d+E)+EELi(\d+)ELi(\d+)E", name)
    return (m.group(1), int(m.group(2 if m.group(1) == "k_row" else 3))) if m else None


@pytest.mark.parametrize("res", [256, 384])
def test_no_fusing_left_to_the_compiler(tmp_path, res):
    plan = subprocess.run(["make", "-B", "-n", "-C", CSRC, os.path.join(CSRC, "_build", f"sweeps_{res}.o")],
                          capture_output=True, text=True, check=True).stdout
    cmd = shlex.split(next(line for line in plan.splitlines() if f"sweeps_{res}.hip" in line))
    if shutil.which(cmd[0]) is None:
        pytest.skip("no hipcc")
    at = cmd.index("-o")
    cmd = [c for i, c in enumerate(cmd) if i not in (at, at + 1) and c != "-c"] + ["--cuda-device-only", "-S"]
    runs = {k: subprocess.Popen(cmd + extra + ["-o", str(tmp_path / k)], cwd=CSRC, stderr=subprocess.DEVNULL)
            for k, extra in (("on", []), ("off", ["-ffp-contract=off"]))}
    assert all(r.wait(timeout=300) == 0 for r in runs.values())
    on, off = kernels(tmp_path / "on"), kernels(tmp_path / "off")
    assert set(on) == set(off)
    seen = set()
    for name, code in on.items():
        m = mode(name)
        seen.add(m)
        if m and m[1] in LEFT[m[0]]:
            continue
        assert code == off[name], name
    # the slice step's kernels are among those compared
    assert {("k_row", 0), ("k_row", 7), ("k_col", 0), ("k_col", 1), ("k_col", 8)} <= seen
    for pipe in ("k_row_step_pipe", "k_col_prop_pipe", "k_col_prop_lean"):
        assert any(pipe in name for name in on)
