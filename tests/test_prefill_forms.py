"""The forms of the W4A16 prefill kernel that are compiled are the ones that the planner takes somewhere: the compile time of
the library is mostly theirs.  (Sixteen more were compiled once that only a tuning override reached.)"""
import os
import re
import subprocess

from tests import emu
from tests.emu import bounds_sweep as bs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# (waves, k groups, column tiles, row tiles): a small shape (M, N, K) whose estimate is the smallest
FORMS = {
    (4, 2, 1, 4): (80, 128, 256), (4, 2, 1, 5): (208, 4160, 256), (4, 2, 1, 6): (176, 5456, 256),
    (4, 2, 1, 7): (112, 8336, 256), (4, 2, 1, 8): (128, 8240, 256), (4, 2, 2, 4): (144, 8416, 256),
    (4, 2, 2, 5): (208, 8256, 256), (4, 2, 2, 6): (96, 16480, 256), (4, 2, 2, 7): (112, 16880, 256),
    (4, 2, 2, 8): (128, 16416, 256), (4, 2, 3, 4): (240, 10944, 896), (4, 2, 3, 5): (144, 16480, 256),
    (4, 2, 3, 6): (176, 16592, 256), (4, 2, 3, 7): (208, 16720, 256), (4, 2, 3, 8): (240, 17152, 256),
    (4, 2, 4, 4): (304, 12672, 640), (4, 2, 4, 5): (144, 25568, 256), (4, 2, 4, 6): (272, 16928, 256),
    (4, 2, 4, 7): (400, 13584, 256), (4, 2, 4, 8): (352, 16496, 256), (4, 1, 3, 5): (784, 9744, 1280),
    (4, 1, 3, 6): (576, 16224, 640), (4, 1, 3, 7): (416, 32928, 256), (4, 1, 3, 8): (3680, 3088, 512),
    (4, 1, 4, 5): (704, 28928, 640), (4, 1, 4, 6): (3264, 3824, 1408), (4, 1, 4, 7): (656, 21536, 256),
    (4, 1, 4, 8): (4656, 3168, 256), (8, 1, 3, 5): (144, 32976, 256), (8, 1, 3, 6): (176, 33520, 256),
    (8, 1, 3, 7): (592, 14128, 256), (8, 1, 3, 8): (240, 32784, 256), (8, 1, 4, 5): (144, 49264, 256),
    (8, 1, 4, 6): (272, 34784, 256), (8, 1, 4, 7): (2464, 4624, 256), (8, 1, 4, 8): (464, 26304, 256),
}


def test_every_form_is_planned_somewhere():
    from ksanallm_amd import capi

    for (nw, kg, ct, rt), (M, N, K) in FORMS.items():
        with emu.session():
            capi.set_launch_log(True)
        assert bs.run_w4((M, N, K, 128, "f16", True), 1) is None
        with emu.session():
            log = capi.last_launch()
            capi.set_launch_log(False)
        assert f"rt={rt},nw={nw},kg={kg},ct={ct}>" in log, (M, N, K, log)


def test_no_other_form_is_compiled():
    """The kernels in the library, by the names of their host-side launch functions, for both element types and one and two
    groups per k tile."""
    lib = os.path.join(ROOT, "ksanallm_amd", "libksq.so")
    names = subprocess.run(["nm", lib], stdout=subprocess.PIPE, text=True, check=True).stdout
    found = set(re.findall(r"__device_stub__w4a16_prefill_kernelI(DF16_|DF16b)Li(\d)ELi(\d)ELi(\d)ELi(\d)ELi(\d)E", names))
    got = {(t, int(gpt), *(int(v) for v in form)) for t, gpt, *form in found}
    want = {(t, gpt, *form) for t in ("DF16_", "DF16b") for gpt in (1, 2) for form in FORMS}
    assert got == want, (sorted(got - want), sorted(want - got))


def test_the_build_refuses_spilling_forms():
    """What the compiler says of a form that spills 31 registers (124 bytes a lane) stops the build; 20 (84) do not."""
    import pytest

    from ksanallm_amd import build

    def remarks(size):
        return [f"f.h:1:1: remark: Function Name: _ZN3ksq20w4a16_prefill_kernelIDF16bLi2EEEv [-Rpass-analysis=x]",
                f"f.h:1:1: remark:     ScratchSize [bytes/lane]: {size} [-Rpass-analysis=x]"]

    build.check_scratch("f.hip", remarks(84))
    with pytest.raises(RuntimeError, match="124 bytes"):
        build.check_scratch("f.hip", remarks(124))
