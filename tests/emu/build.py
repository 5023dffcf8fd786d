"""Builds the library's HIP sources for the CPU (hip/hip_runtime.h, emu.cpp) with the address
sanitizer."""
import os
import re
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
CSRC = os.path.join(ROOT, "tonto_amd", "csrc")
FLAGS = ["g++", "-std=c++17", "-fPIC", "-O1", "-g1", "-w", "-fsanitize=address", "-I" + HERE, "-x", "c++"]


def _matching(s, i, pair="()"):
    """Index after the bracket that closes the one before i."""
    depth = 1
    while depth:
        depth += (s[i] == pair[0]) - (s[i] == pair[1])
        i += 1
    return i


def _split(s):
    out, depth, part = [], 0, ""
    for ch in s:
        if ch == "," and depth == 0:
            out.append(part)
            part = ""
            continue
        depth += (ch in "([{") - (ch in ")]}")
        part += ch
    return out + [part]


def convert(src):
    """Kernel launches, the dynamic LDS and the one register read as C++."""
    src = re.sub(r'asm\("s_getreg[^;]*;', "r = 0;", src)
    src = re.sub(r"extern __shared__ double (\w+)\[\];", r"double *\1 = (double *)emu::dyn_lds;", src)
    out, i = "", 0
    for m in re.finditer(r"((?:\w+::)?\w+(?:<[\w, :]*>)?)<<<(.*?)>>>\(", src, re.S):
        end = _matching(src, m.end())
        cfg = _split(m.group(2))
        lds, stream = (cfg + ["0", "nullptr"])[2:4] if len(cfg) == 2 else (cfg + ["nullptr"])[2:4]
        out += src[i:m.start()]
        out += 'emu::launch("%s", dim3(%s), dim3(%s), %s, %s, [&]{ %s(%s); })' % (
            m.group(1), cfg[0], cfg[1], lds, stream, m.group(1), src[m.end():end - 1])
        i = end
    return out + src[i:]


def build(out):
    """libemu.so in the folder `out`; returns its path."""
    sys.path.insert(0, ROOT)
    from tonto_amd.build import class_list
    src = os.path.join(out, "tonto_amd", "csrc")
    shutil.copytree(CSRC, src)
    shutil.copytree(os.path.join(ROOT, "include"), os.path.join(out, "include"))
    for f in ("tgpu_device.h", "tgpu_host.hip", "jk_class.hip"):
        text = convert(open(os.path.join(src, f)).read())
        open(os.path.join(src, f), "w").write(text)
    jobs = [(os.path.join(src, "tgpu_host.hip"), "host", []), (os.path.join(HERE, "emu.cpp"), "emu", []),
            (shutil.copy(os.path.join(HERE, "shapes.cpp"), src), "shapes", [])]
    for lp, lq, lr, ls, heavy in class_list():
        jobs.append((os.path.join(src, "jk_class.hip"), f"jk_{lp}{lq}{lr}{ls}",
                     [f"-DTGPU_LP={lp}", f"-DTGPU_LQ={lq}", f"-DTGPU_LR={lr}", f"-DTGPU_LS={ls}",
                      f"-DTGPU_HEAVY={heavy}"]))

    def compile_one(job):
        obj = os.path.join(out, job[1] + ".o")
        r = subprocess.run(FLAGS + job[2] + ["-c", job[0], "-o", obj], capture_output=True, text=True)
        if r.returncode:
            raise RuntimeError(f"{job[1]}: {r.stderr[-3000:]}")
        return obj
    with ThreadPoolExecutor(min(8, os.cpu_count() or 8)) as ex:
        objs = list(ex.map(compile_one, jobs))
    lib = os.path.join(out, "libemu.so")
    subprocess.check_call(["g++", "-shared", "-fsanitize=address", "-o", lib] + objs)
    return lib


if __name__ == "__main__":
    print(build(sys.argv[1]))
