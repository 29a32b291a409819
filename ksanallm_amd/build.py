"""Builds libksq.so (the HIP kernels + C ABI) for gfx950 with hipcc, in-tree."""
import os
import shutil
import subprocess
import sys
import tempfile
import time

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libksq.so")

# slowest to compile first: they start first (run_compilers)
SOURCES = ["ksq_w4a16_prefill_f16.hip", "ksq_w4a16_prefill_bf16.hip", "ksq_w4a16_stream.hip", "ksq_w4a16_kstat.hip",
           "ksq_fp8_kstat.hip", "ksq_w4a16_astream.hip", "ksq_fp8.hip", "ksq_fp8_prefill.hip", "ksq_fp8_mid.hip",
           "ksq_repack.hip", "ksq_w4a16_prefill.hip", "ksq_api.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
    "-Rpass-analysis=kernel-resource-usage",  # read back by check_scratch below; not printed
    "-I" + os.path.join(ROOT, "include"),
    "-I" + CSRC,
]


# Private (scratch) memory per lane that a kernel may use.  The kernels keep their accumulators in lambdas' captures; if
# the compiler ever stops inlining one of those lambdas the captures move to memory (seen once: 1136 bytes per lane and
# a tenth of the speed, with every test still passing).  Real register spills of the fallback kernels stay below this.
MAX_SCRATCH_BYTES = 512
# The tile kernel's steps have no memory instruction to spare: its forms spill at most 20 registers (two k groups, 128 x 64 a
# wave; counted in the planner's estimates).  31 in one form that the estimates did not know of cost 40 %.
MAX_SCRATCH_BYTES_OF = {"w4a16_prefill_kernel": 88}


def check_scratch(src, remarks):
    """remarks: the compiler's kernel-resource-usage lines for one source file; raises on a kernel over the limit."""
    name = None
    for line in remarks:
        text = line.split("remark:", 1)[1].strip()
        if text.startswith("Function Name:"):
            name = text.split(":", 1)[1].split("[")[0].strip()
        elif text.startswith("ScratchSize"):
            size = int(text.split(":", 1)[1].split("[")[0].strip())
            limit = next((v for k, v in MAX_SCRATCH_BYTES_OF.items() if k in (name or "")), MAX_SCRATCH_BYTES)
            if size > limit:
                raise RuntimeError(f"{src}: kernel {name} uses {size} bytes of scratch memory per lane (limit {limit}): "
                                   "spilled registers, or a lambda of the kernel that is no longer inlined")


def hipcc():
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; libksq.so cannot be built")
    return exe


def run_compilers(commands, done, jobs=None):
    """commands: (source name, command line).  At most `jobs` at a time, each started as soon as another ends;
    done(name, exit status, output) is called as they end, and every one that ended is named on stderr."""
    jobs = jobs or max(1, min(16, int(os.environ.get("MAX_JOBS", "0")) or os.cpu_count() or 1))
    waiting, running = list(commands), []
    try:
        while waiting or running:
            while waiting and len(running) < jobs:
                name, cmd = waiting.pop(0)
                log = tempfile.TemporaryFile(mode="w+")
                running.append((name, subprocess.Popen(cmd, stdout=log, stderr=subprocess.STDOUT), log, time.time()))
            time.sleep(0.05)
            for item in [r for r in running if r[1].poll() is not None]:
                running.remove(item)
                name, p, log, t0 = item
                log.seek(0)
                print(f"[build] {name} {time.time() - t0:.0f} s", file=sys.stderr, flush=True)
                done(name, p.returncode, log.read())
                log.close()
    finally:
        for _, p, log, _ in running:  # another one failed
            p.kill()
            p.wait()
            log.close()


def build_library(verbose=False, jobs=None):
    """Compile every HIP source to an object (in parallel) and link libksq.so next to this file."""
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    cc = hipcc()
    objs, commands = [], []
    for src in SOURCES:
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        objs.append(obj)
        cmd = [cc, *HIPCC_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        commands.append((src, cmd))
    run_compilers(commands, _compiled, jobs)
    link = [cc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    subprocess.check_call(link)
    return LIB


def build_layer_driver():
    """Compile the C++ layer shims (host code over the C ABI) and their test driver next to libksq.so."""
    cc = hipcc()
    layers = os.path.join(CSRC, "layers")
    out = os.path.join(HERE, "layer_driver")
    cmd = [cc, "-std=c++17", "-O2", "-Wall", "-Wno-unused-parameter", "-I" + os.path.join(ROOT, "include"),
           "-I" + layers, os.path.join(ROOT, "tests", "cpp", "layer_driver.cpp"), os.path.join(layers, "layers.cpp"),
           "-L" + HERE, "-lksq", "-Wl,-rpath,$ORIGIN", "-o", out]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if p.returncode != 0:
        raise RuntimeError("layer driver build failed:\n" + p.stdout)
    # host-only check of the workgroup -> tile map shared by the tile kernels (run by tests/test_capi_host.py)
    tm = os.path.join(HERE, "tile_map_test")
    cmd = [cc, "--offload-arch=gfx950", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
           os.path.join(ROOT, "tests", "cpp", "tile_map_test.hip"), "-o", tm]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if p.returncode != 0:
        raise RuntimeError("tile map test build failed:\n" + p.stdout)
    return out


def _compiled(src, status, out):
    """One source file's compiler output: its messages without the resource remarks, which check_scratch reads."""
    remarks, lines, skip = [], [], 0
    for ln in out.splitlines():
        if "-Rpass-analysis=kernel-resource-usage" in ln:
            remarks.append(ln)
            skip = 2  # the source line and the caret that follow a remark
        elif skip and ln.lstrip()[:1] in "0123456789|":
            skip -= 1
        elif "packed-fp32-ops" not in ln and "remarks generated" not in ln and "In file included from" not in ln:
            skip = 0
            lines.append(ln)
    if status != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n" + "\n".join(lines))
    check_scratch(src, remarks)
    if lines:
        print("\n".join(lines), file=sys.stderr)


if __name__ == "__main__":
    print(build_library(verbose=True))
    print(build_layer_driver())
