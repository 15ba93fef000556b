"""Build libmoespresso_amd.so from the HIP sources in ``csrc/`` with hipcc for gfx950, and the Python extension
``_dispatch.so`` (``binding/dispatch.cpp``) that calls it with torch tensors.

``python -m moespresso_amd.build`` compiles every source to an object file (in
parallel) and links both in-tree next to this file. hipcc
cross-compiles without a GPU.
"""

from __future__ import annotations

import concurrent.futures
import functools
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(HERE, "_obj")
LIB_PATH = os.path.join(HERE, "libmoespresso_amd.so")
DISPATCH_SRC = os.path.join(HERE, "binding", "dispatch.cpp")
DISPATCH_PATH = os.path.join(HERE, "_dispatch.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
COMMON_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # packed FP32 VALU forms are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # The first plain arguments of a kernel, up to 14 words, arrive in registers with its waves instead of through a load at
    # their start (400 to 900 cycles where the argument block is in no cache yet, as at every launch): the score, QAT,
    # selection, rope and 8-bit quantisation kernels. DS4 decode of one sequence 24.1 -> 23.6 us, of five 30.5 -> 30.1, four
    # captured layers of sixteen 211.6 -> 209.7, a 517-token chunk 160.5 -> 156.7. The attention, flash and 8-bit split kernels
    # take what their first loads need this way and what they read later in a struct, which is loaded meanwhile; the 8-bit
    # merge and append and the rows of a quantised prefill take structs only.
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wno-unused-command-line-argument",
    # the asynchronous LDS loads set M0 by hand inside inline asm
    "-Wno-inline-asm",
]


def sources() -> list[str]:
    return sorted(
        os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip") or f.endswith(".cpp")
    )


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
    cmd = [HIPCC, *COMMON_FLAGS, "-c", src, "-o", obj]
    if src.endswith(".cpp"):
        cmd = [HIPCC, "-O2", "-std=c++17", "-fPIC", "-c", src, "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _compile_dispatch() -> str:
    """Object file of the Python extension: host code only, against the headers of the installed torch."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    obj = os.path.join(OBJ_DIR, "dispatch.o")
    cmd = [HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-fPIC", "-DUSE_ROCM",
           f'-DMSPR_TORCH_VERSION="{torch.__version__}"', f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-I{p}" for p in cpp_extension.include_paths("cuda")), f"-I{sysconfig.get_paths()['include']}",
           "-w", "-c", DISPATCH_SRC, "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {DISPATCH_SRC}:\n{proc.stderr}")
    return obj


def _link(out: str, args: list[str]) -> None:
    proc = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out, *args], capture_output=True,
                          text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stderr}")


def build(verbose: bool = True) -> str:
    from torch.utils import cpp_extension

    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sources()
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as pool:
        dispatch = pool.submit(_compile_dispatch)
        objs = list(pool.map(_compile, srcs))
        dispatch = dispatch.result()
    _link(LIB_PATH, [*objs, "-Wl,-soname," + os.path.basename(LIB_PATH)])
    # the library is found next to the extension; torch's own libraries are loaded before the extension is imported
    _link(DISPATCH_PATH, [dispatch, LIB_PATH, "-Wl,-rpath,$ORIGIN",
                          *(f"-L{p}" for p in cpp_extension.library_paths("cuda")[:1]), "-lc10", "-lc10_hip",
                          "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python"])
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources, and {DISPATCH_PATH}")
    return LIB_PATH


@functools.lru_cache(maxsize=None)
def device_assembly(src: str) -> str:
    """gfx950 assembly of one HIP source (device-only compile, nothing runs), made once a process."""
    import tempfile

    with tempfile.TemporaryDirectory() as tmp:
        out = os.path.join(tmp, "kernels.s")
        cmd = [HIPCC, *COMMON_FLAGS, "-S", "--cuda-device-only", "-o", out, src]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{proc.stderr}")
        return open(out).read()


def kernel_resources(src: str, text: str | None = None) -> dict[str, dict[str, int]]:
    """Registers and scratch of every kernel in one HIP source, from the code object metadata of a device-only
    compile to assembly: ``{kernel symbol: {"vgprs", "sgprs", "scratch_bytes", "vgpr_spills", "sgpr_spills"}}``.

    The kernels that count their own vector-memory operations (asynchronous tile copies awaited with
    ``s_waitcnt vmcnt(n)``) rely on the compiler adding none: a register spilled to scratch is one more
    vector-memory operation in the middle of the count, and its reload drains every copy in flight.
    """
    import re

    text = device_assembly(src) if text is None else text
    fields = {"vgprs": "vgpr_count", "sgprs": "sgpr_count", "scratch_bytes": "private_segment_fixed_size",
              "vgpr_spills": "vgpr_spill_count", "sgpr_spills": "sgpr_spill_count"}
    kernels: dict[str, dict[str, int]] = {}
    # one metadata record per kernel: "- .agpr_count: ..." up to the next record; ".name:" carries the symbol
    for record in re.split(r"\n  - \.", text[text.index("amdhsa.kernels:"):])[1:]:
        name = re.search(r"\.name:\s+(\S+)", record)
        if not name:
            continue
        kernels[name.group(1)] = {
            key: int(m.group(1)) if (m := re.search(rf"\.{field}:\s+(\d+)", record)) else 0
            for key, field in fields.items()
        }
    return kernels


def kernel_bodies(text: str) -> dict[str, list[str]]:
    """Instruction lines of every kernel of an assembly text: ``{kernel symbol: [line, ...]}``."""
    import re

    bodies: dict[str, list[str]] = {}
    for m in re.finditer(r"^(\w+):[^\n]*\n(.*?)^\s*\.end_amdhsa_kernel", text, flags=re.S | re.M):
        if ".amdhsa_kernel " + m.group(1) in m.group(2):
            bodies[m.group(1)] = m.group(2).split(".section")[0].splitlines()
    return bodies


def inline_asm_register_loads(lines: list[str]) -> list[str]:
    """Memory loads with a register destination that come from inline asm statements (the compiler brackets those
    with ``;;#ASMSTART`` / ``;;#ASMEND``). The compiler takes the outputs of an asm statement for valid the moment
    the statement ends, so a load issued that way may see its destination register moved, reused or spilled while
    the data is still in flight; loads whose destination is LDS write no register and are exempt."""
    import re

    found, inside = [], False
    for line in lines:
        if "#ASMSTART" in line:
            inside = True
        elif "#ASMEND" in line:
            inside = False
        elif inside and re.search(r"\b(global|buffer|flat|scratch)_load|\bs_(buffer_)?load", line) and "_lds_" not in line:
            found.append(line.strip())
    return found


def m0_hazards(lines: list[str]) -> list[str]:
    """Asynchronous copies into LDS that directly follow the scalar instruction that writes M0, from which they take
    their LDS address. gfx950 wants an instruction between the two; the compiler puts one there for its own copies
    but does not look inside an inline asm statement."""
    import re

    found, previous = [], ""
    for line in lines:
        text = line.split(";")[0].strip()
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        if "_load_lds_" in text and re.match(r"s_\w+ m0\b", previous):
            found.append(f"{previous} / {text}")
        previous = text
    return found


def scalar_register_hazards(lines: list[str]) -> list[str]:
    """Instructions of inline asm statements that read a scalar register too soon after a vector instruction wrote it: two wait
    states have to lie between for another vector instruction, five for a memory instruction. The compiler keeps to that in its
    own code but does not look inside an asm statement."""
    import re

    def scalars(operand: str) -> set[str]:
        if operand == "vcc":
            return {"vcc"}
        m = re.fullmatch(r"s(?:(\d+)|\[(\d+):(\d+)\])", operand)
        return {f"s{i}" for i in range(int(m[1] or m[2]), int(m[1] or m[3]) + 1)} if m else set()

    found, inside, written = [], False, []  # `written`: per wait state, the scalar registers that a vector instruction wrote
    for line in lines:
        if "#ASMSTART" in line or "#ASMEND" in line:
            inside = "#ASMSTART" in line
        text = line.split(";")[0].strip()
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        name, _, rest = text.partition(" ")
        operands = [o.split()[0] if o.split() else "" for o in rest.split(",")]
        vector = name.startswith("v_")
        n_out = 2 if vector and "_co_" in name else 1 if vector else 0
        states = 0 if not inside else 2 if vector else 5 if name.startswith(("global_", "buffer_", "flat_", "scratch_")) else 0
        read = set().union(*map(scalars, operands[n_out:])) if operands[n_out:] else set()
        if states and any(read & w for w in written[-states:]):
            found.append(text)
        written.append(set().union(*map(scalars, operands[:n_out])) if n_out else set())
        if name == "s_nop":
            written += [set()] * int(operands[0], 0)
    return found


if __name__ == "__main__":
    build()
