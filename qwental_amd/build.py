"""Build recipe of the HIP backend: kernels -> gfx950 code object -> embedded into libqwgpu_hip.so.

    python -m qwental_amd.build

Three steps, all cross-compile without a GPU:
  1. hipcc --genco: csrc/kernels/qw_kernels.hip -> csrc/qw_kernels_gfx950.hsaco (one code object: the same kernels spread over
     several measured 3 % slower on the 48-layer step), and a look at the waits in it that count loads (check_counted_waits);
     beside it the kernels for several launches in one -> csrc/qw_joined_gfx950.hsaco (kernels/qw_joined.hip.h says why they lie apart)
  2. hipcc -c: csrc/qw_noalloc.hip (host + device: the per-device scratch array of the entry point that allocates nothing) -> csrc/qw_noalloc.o
  3. clang -std=c23: csrc/gpu_hip.c and csrc/qw_joined.c (embed the code objects) + csrc/qw_path.c + csrc/qw_gguf.c + csrc/qw_par.c + qw_noalloc.o -> qwental_amd/libqwgpu_hip.so
"""
import concurrent.futures
import heapq
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")
CLANG = os.path.join(ROCM, "llvm", "bin", "clang")
LIB = os.path.join(HERE, "libqwgpu_hip.so")
# Experiments: QW_BUILD_TAG=<tag> makes a second build beside the product's, libqwgpu_hip_<tag>.so with its objects in
# csrc/_<tag>/ (QW_HIP_LIB selects it at run time); QW_BUILD_DEFS adds compiler flags, e.g. -DQW_PARTS=0x37 for a code
# object that holds only some groups of kernels (a short compile; the joined forms are compiled all the same).
TAG = os.environ.get("QW_BUILD_TAG", "")
OBJDIR = os.path.join(CSRC, "_" + TAG) if TAG else CSRC
if TAG:
    os.makedirs(OBJDIR, exist_ok=True)
    LIB = os.path.join(HERE, "libqwgpu_hip_%s.so" % TAG)
HSACO = os.path.join(OBJDIR, "qw_kernels_gfx950.hsaco")
JOINED = os.path.join(OBJDIR, "qw_joined_gfx950.hsaco")
PARTS, JOINED_PARTS = 0x3f, 0x40  # of qw_kernels.hip, groups of kernels in either code object
# -packed-fp32-ops: packed FP32 instructions are kept out of every kernel of this library
HIPFLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"] + os.environ.get("QW_BUILD_DEFS", "").split()


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode:
        sys.stderr.write(out + "\n")
        raise RuntimeError("build step failed: " + " ".join(cmd))
    return out


# Kernels that wait for their direct loads into LDS by the number of loads issued behind them (qw_grouped.hip.h)
COUNTING = ("qwk_pfg_f121", "qwk_pfg_f120")


def listing(kernel, hsaco=None):
    """The instructions of one kernel of the code object, as llvm-objdump prints them (empty: no such kernel)."""
    with open(hsaco or HSACO, "rb") as f:
        elf = f.read()
    elf = elf[elf.index(b"\x7fELF"):]  # behind the header of hipcc's bundle
    tmp = os.path.join(OBJDIR, "qw_listing_%d.o" % os.getpid())
    try:
        with open(tmp, "wb") as f:
            f.write(elf)
        return subprocess.run([os.path.join(ROCM, "llvm", "bin", "llvm-objdump"), "-d", "--disassemble-symbols=" + kernel, tmp],
                              stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True, check=True).stdout
    finally:
        os.unlink(tmp)


def check_counted_waits(text):
    """Raise unless every "s_waitcnt vmcnt(N)" with N > 0 in front of a barrier has, on every path from a direct load into LDS
    that is not waited for otherwise, at least N register loads behind that load. Returns (wait, N, fewest loads) of the waits found."""
    code, start = [], None
    for line in text.splitlines():
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]{12}):[^<]*(?:<\S+?\+0x([0-9a-f]+)>|<\S+>)?", line)
        if m:
            at = int(m[3], 16)
            start = at if start is None else start
            code.append((at, m[1], m[2], start + int(m[4] or "0", 16) if m[1].startswith(("s_cbranch", "s_branch")) else None))
    index = {c[0]: i for i, c in enumerate(code)}

    def vmcnt(i):
        m = re.search(r"vmcnt\((\d+)\)", code[i][2]) if code[i][1] == "s_waitcnt" else None
        return int(m[1]) if m else None

    fewest = {i: None for i in range(len(code) - 1) if vmcnt(i) and code[i + 1][1] == "s_barrier"}
    if not fewest:
        raise RuntimeError("no counted wait found")
    for i, c in enumerate(code):
        if not c[1].startswith("global_load_lds"):
            continue
        done, heap = set(), [(0, i + 1)]
        while heap:  # the fewest loads from here to every place that can be reached
            n, j = heapq.heappop(heap)
            if j in done or j >= len(code):
                continue
            done.add(j)
            _, op, _, to = code[j]
            if j in fewest:
                fewest[j] = n if fewest[j] is None else min(n, fewest[j])
                continue
            if op == "s_endpgm" or vmcnt(j) == 0:
                continue
            n += op.startswith("global_load_") and "_lds_" not in op
            if op != "s_branch":
                heapq.heappush(heap, (n, j + 1))
            if to is not None:
                heapq.heappush(heap, (n, index[to]))
    for i, n in fewest.items():
        if n is not None and n < vmcnt(i):
            raise RuntimeError("a wait for all but %d operations has only %d loads behind what it waits for" % (vmcnt(i), n))
    return [(hex(code[i][0]), vmcnt(i), n) for i, n in fewest.items()]


def build(verbose=False, kernels=True):
    """kernels=False keeps the code object of the last build (host-side iterations: `python -m qwental_amd.build --host-only`)."""
    if kernels or not (os.path.exists(HSACO) and os.path.exists(JOINED)):
        genco = lambda out, parts: _run([HIPCC] + HIPFLAGS + parts + ["--genco", "-I", os.path.join(CSRC, "kernels"), "-o", out, os.path.join(CSRC, "kernels", "qw_kernels.hip")])
        some = any(f.startswith("-DQW_PARTS=") for f in HIPFLAGS)
        with concurrent.futures.ThreadPoolExecutor(2) as two:
            for out in two.map(genco, (HSACO, JOINED), ([] if some else ["-DQW_PARTS=%d" % PARTS], ["-UQW_PARTS", "-DQW_PARTS=%d" % JOINED_PARTS])):
                if verbose and out.strip():
                    print(out)
        for k in COUNTING:
            text = listing(k)
            if text.strip() or not TAG:  # (a working build may hold some groups of kernels only)
                check_counted_waits(text)
    noalloc_o = os.path.join(OBJDIR, "qw_noalloc.o")
    _run([HIPCC] + HIPFLAGS + ["-fPIC", "-I", CSRC, "-I", os.path.join(ROOT, "include"), "-c", os.path.join(CSRC, "qw_noalloc.hip"), "-o", noalloc_o])
    out = _run([CLANG, "-std=c23", "-O2", "-Wall", "-Wextra", "-fPIC", "-shared", "--embed-dir=" + OBJDIR] + [f for f in os.environ.get("QW_BUILD_DEFS", "").split() if f.startswith("-D")] + ["-I", os.path.join(ROOT, "include"), "-I", CSRC,
                "-I", os.path.join(ROCM, "include"), os.path.join(CSRC, "gpu_hip.c"), os.path.join(CSRC, "qw_joined.c"), os.path.join(CSRC, "qw_path.c"), os.path.join(CSRC, "qw_gguf.c"), os.path.join(CSRC, "qw_par.c"), noalloc_o, "-pthread", "-o", LIB,
                "-L", os.path.join(ROCM, "lib"), "-lamdhip64", "-Wl,-rpath," + os.path.join(ROCM, "lib")])
    if verbose and out.strip():
        print(out)
    if TAG:
        return LIB
    # command-line tool with the reference's dqtest contract
    _run([CLANG, "-std=c23", "-O2", "-Wall", "-I", os.path.join(ROOT, "include"), os.path.join(CSRC, "tools", "dqhip.c"), "-o",
          os.path.join(HERE, "dqhip"), "-L", HERE, "-lqwgpu_hip", "-Wl,-rpath,$ORIGIN", "-Wl,-rpath," + os.path.join(ROCM, "lib")])
    return LIB


if __name__ == "__main__":
    print(build(verbose=True, kernels="--host-only" not in sys.argv))
