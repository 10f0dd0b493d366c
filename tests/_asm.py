"""The gfx950 assembly of a source and the compiler's resource report, from one
compilation per source and session."""
import atexit
import functools
import re
import shutil
import subprocess
import tempfile
from pathlib import Path

from logan_amd import build

CSRC = Path(build.CSRC)


@functools.lru_cache(maxsize=None)
def _dir() -> Path:
    d = Path(tempfile.mkdtemp(prefix="logan_asm_"))
    atexit.register(shutil.rmtree, d, ignore_errors=True)
    return d


@functools.lru_cache(maxsize=None)
def compiled(name: str):
    """(path of the assembly, {mangled kernel: its resources: "ScratchSize
    [bytes/lane]", "LDS Size [bytes/block]", "VGPRs", ...})."""
    out = _dir() / (name + ".s")
    cmd = [build.hipcc(), *build.HIPFLAGS, "-I", str(build.INCLUDE), "--cuda-device-only", "-S", str(CSRC / name),
           "-o", str(out), "-Rpass-analysis=kernel-resource-usage"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    usage, kernel = {}, None
    for line in r.stderr.splitlines():
        m = re.search(r"remark: [^:]+:\d+:\d+:\s+([^:]+): (\S+)", line) or re.search(r"remark:\s+([^:]+): (\S+)", line)
        if not m:
            continue
        if m[1] == "Function Name":
            kernel = usage.setdefault(m[2], {})
        elif kernel is not None:
            kernel[m[1]] = m[2]
    return out, {k: {n: int(v) for n, v in u.items() if v.isdigit()} for k, u in usage.items()}
