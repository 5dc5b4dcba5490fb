"""Build libexodus_hip.so for gfx950 with hipcc (cross-compiles without a GPU).

Usage:  python build_hip.py
The library lands next to the Python loader (sinabs/exodus/libexodus_hip.so), and beside it the host side of its calls
(sinabs/exodus/_exodus_torch.so, plain C++ compiled against the installed torch).  A third, small
library with the streaming probes that only bench.py uses (libexodus_bench_probes.so, next to this
script) is built in the same go; it is not part of the product.
"""
import os
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
SRCS = [os.path.join(HERE, "csrc", f) for f in ("exodus_hip.hip", "exodus_layer.hip", "exodus_layer_backward.hip",
                                                  "exodus_layer_forward_roles.hip", "exodus_layer_backward_split.hip",
                                                  "exodus_layer_leaky_split.hip", "exodus_hbm.hip")]
SRC = SRCS[0]
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
OUT = os.path.join(HERE, "sinabs", "exodus", "libexodus_hip.so")
# the host side of the calls (C++ against the installed torch), next to the Python loader
TORCH_SRC = os.path.join(HERE, "csrc", "exodus_torch.cpp")
TORCH_OUT = os.path.join(HERE, "sinabs", "exodus", "_exodus_torch.so")
PROBE_SRC = os.path.join(HERE, "csrc", "bench_probes.hip")
PROBE_OUT = os.path.join(HERE, "libexodus_bench_probes.so")

# -ffp-contract=off : the forward recurrences must round every multiply and add separately
# -packed-fp32-ops disabled : keep the compiler from forming packed fp32 instructions
FLAGS = [
    "-O3", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-Wno-unused-command-line-argument",
]


def built_for() -> str:
    """What the host side of the calls is compiled against and works with: torch's C++ interfaces change with its version."""
    import torch

    return f"torch {torch.__version__}, Python {sys.version_info[0]}.{sys.version_info[1]};"


def _torch_command(out: str) -> list:
    import sysconfig

    from torch.utils import cpp_extension

    rocm = os.path.dirname(os.path.dirname(os.path.realpath(shutil.which("hipcc") or "/opt/rocm/bin/hipcc")))
    command = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
               "-DUSE_ROCM"]
    for path in cpp_extension.include_paths() + [sysconfig.get_paths()["include"], os.path.join(rocm, "include")]:
        command += ["-isystem", path]
    command += [f'-DEXODUS_BUILT_FOR="{built_for()}"', "-I", INCLUDE, TORCH_SRC, "-o", out]
    command += ["-L" + path for path in cpp_extension.library_paths()]
    return command + ["-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip"]


def up_to_date() -> bool:
    """Whether everything is built, from the sources as they are and for the torch and Python that are running."""
    deps = SRCS + [PROBE_SRC, TORCH_SRC, os.path.join(HERE, "csrc", "exodus_common.hpp"), os.path.join(HERE, "csrc", "exodus_layer.hpp"), os.path.join(INCLUDE, "exodus_hip.h")]
    outs = (OUT, PROBE_OUT, TORCH_OUT)
    if not all(os.path.exists(o) for o in outs) or min(map(os.path.getmtime, outs)) < max(map(os.path.getmtime, deps)):
        return False
    with open(TORCH_OUT, "rb") as module:
        return built_for().encode() in module.read()


def build(force: bool = True) -> str:
    if not force and up_to_date():
        return OUT
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    # hipcc's host pass does not know the gfx-only target feature and says so; that line is harmless
    noise = "packed-fp32-ops"
    quiet = lambda text: "\n".join(l for l in text.splitlines() if noise not in l)
    compile_flags = [f for f in FLAGS if f != "-shared"]
    with tempfile.TemporaryDirectory() as tmp:
        # one hipcc process per translation unit, side by side, then one link
        objs = [os.path.join(tmp, os.path.basename(src) + ".o") for src in SRCS]
        procs = [subprocess.Popen([hipcc] + compile_flags + ["-I", INCLUDE, "-c", src, "-o", obj],
                                  stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
                 for src, obj in zip(SRCS, objs)]
        # the bench-only probes: one small translation unit, compiled and linked in one step
        procs.append(subprocess.Popen([hipcc] + FLAGS + ["-I", INCLUDE, PROBE_SRC, "-o", PROBE_OUT + ".tmp"],
                                      stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True))
        procs.append(subprocess.Popen(_torch_command(TORCH_OUT + ".tmp"), stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                                      text=True))
        outputs = [proc.communicate()[0] for proc in procs]
        log = "\n".join(filter(None, (quiet(o).strip() for o in outputs)))
        failed = [f"{os.path.basename(proc.args[0])} failed compiling {os.path.basename(src)}"
                  for proc, src in zip(procs, SRCS + [PROBE_SRC, TORCH_SRC]) if proc.returncode != 0]
        if failed:
            sys.stderr.write(log + "\n")
            raise RuntimeError("; ".join(failed))
        link = subprocess.run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", OUT + ".tmp"] + objs,
                              stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        log = "\n".join(filter(None, (log, quiet(link.stdout).strip())))
        if link.returncode != 0:
            sys.stderr.write(log + "\n")
            raise RuntimeError("hipcc failed linking libexodus_hip.so")
    if log.strip():
        sys.stderr.write(log + "\n")
    os.replace(OUT + ".tmp", OUT)
    os.replace(PROBE_OUT + ".tmp", PROBE_OUT)
    os.replace(TORCH_OUT + ".tmp", TORCH_OUT)
    return OUT


if __name__ == "__main__":
    print(build(force=True))
