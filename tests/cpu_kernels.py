"""Kernels of flipengine3d_amd/csrc compiled for the host, to test on the CPU what a GPU shows only now and then.

`build` rewrites the launches of the .hip sources and compiles them, with a check program that includes them, against
the stand-in header of tests/cpp/cpu_kernels.
"""

import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "flipengine3d_amd", "csrc")
HERE = os.path.join(ROOT, "tests", "cpp", "cpu_kernels")


def _closing(text, at, opening, closing):
    depth = 0
    for q in range(at, len(text)):
        depth += (text[q] in opening) - (text[q] in closing)
        if depth == 0:
            return q
    raise ValueError("unbalanced")


def _split(text):
    parts, depth, cur = [], 0, ""
    for ch in text:
        depth += (ch in "([{") - (ch in ")]}")
        if ch == "," and depth == 0:
            parts.append(cur)
            cur = ""
        else:
            cur += ch
    return parts + [cur]


def for_host(source):
    """kernel<<<grid, block, lds, stream>>>(args) as a call of the stand-in's launch."""
    out, at = "", 0
    for m in re.finditer(r"([A-Za-z_]\w*(?:<[^<>;{}]*>)?)<<<", source):
        if m.start() < at:
            continue
        end = source.index(">>>", m.end())
        cfg = _split(source[m.end():end])
        close = _closing(source, end + 3, "(", ")")
        args = source[end + 4:close]
        lds = cfg[2] if len(cfg) > 2 else "0"
        out += source[at:m.start()]
        out += (f"cpu::launch((unsigned)({cfg[0]}), (unsigned)({cfg[1]}), (size_t)({lds}), "
                f"[=]() mutable {{ {m.group(1)}({args}); }})")
        at = close + 1
    out += source[at:]
    out = out.replace("extern __shared__ float lds[];", "float *const lds = reinterpret_cast<float *>(cpu::dynamic_lds);")
    return re.sub(r"hipExtLaunchKernelGGL\(.*?\);", "std::abort();", out, flags=re.S)


def build(check, kernels, out_dir):
    """Compiles tests/cpp/cpu_kernels/<check>.cpp; it includes "<kernel>.host.inc" for each of `kernels`."""
    for name in kernels:
        with open(os.path.join(CSRC, name + ".hip")) as f:
            text = for_host(f.read())
        with open(os.path.join(out_dir, name + ".host.inc"), "w") as f:
            f.write(text)
    exe = os.path.join(out_dir, check)
    # The sources' own directory comes last: the stand-in's hip/ is found first.  Fibers jump between stacks, which the
    # fortified longjmp takes for an error.
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-U_FORTIFY_SOURCE", "-w", "-I", HERE, "-I",
                    str(out_dir), "-I", CSRC, os.path.join(HERE, check + ".cpp"), os.path.join(HERE, "fibers.cpp"),
                    "-o", exe], check=True)
    return exe
