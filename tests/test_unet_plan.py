"""The launch rules of the U-Net's convolutions (csrc/unet_plan.h), on the CPU:
every choice has a compiled form, boxes that would be mostly padding are left
to the direct kernel, and the GPU tests run every form that the default network
reaches."""
import os
import subprocess

import pytest

from hemelb_amd import warmstart as WS
from tests import test_gpu_unet, test_gpu_unet_forms, test_gpu_unet_shapes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "check")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "hemelb_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "unet_plan_check.cpp"), "-o", exe],
                   check=True)

    def run(calls=None):
        text = "".join("%d %d %d %d\n" % c for c in calls) if calls is not None else ""
        out = subprocess.run([exe] + ([] if calls is not None else ["forms"]), input=text,
                             capture_output=True, text=True, check=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]
    return run


LEVELS = [0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0]


def convolutions(side, batch, chans=WS.CHANNELS, backward=True):
    """(N, side, ci, co) of the forward convolutions, and with `backward` of the
    data gradients of all layers but the first."""
    calls = []
    for (name, ci, co), level in zip(WS.layer_shapes(chans), LEVELS):
        calls.append((batch, side >> level, ci, co))
        if backward and name != "e1a":
            calls.append((batch, side >> level, co, ci))
    return calls


def test_every_choice_is_compiled_and_concatenations_read_in_place_have_a_form(plan):
    forms = set(plan())
    calls = [(n, s, 16 * a, 16 * b) for n in (1, 2, 5, 70, 900) for s in range(1, 129, 1)
             if n * s ** 3 < 1 << 26 for a in range(1, 15) for b in (1, 2, 3, 4, 6, 12)]
    for call, (*form, _, width) in zip(calls, plan(calls)):
        assert tuple(form) in forms or not form[0], (call, form)
        # the choice of reading a concatenation in place looks at ci alone
        if width and call[2] // 16 in (1, 2, 3, 4, 6, 8, 12):
            assert form[0], call


@pytest.mark.parametrize("call,box", [
    # levels of side 1 to 4 with many samples: boxes would be mostly padding
    ((1000, 1, 128, 128), False), ((1000, 2, 32, 64), False), ((256, 2, 64, 192), False),
    ((300, 2, 128, 128), False), ((1000, 4, 32, 96), False),
    # few samples leave the chip empty anyhow; half empty boxes are the faster ones
    ((6, 1, 128, 128), True), ((64, 2, 32, 64), True), ((6, 3, 192, 64), True),
    ((300, 4, 192, 64), True), ((4, 64, 16, 16), True), ((4, 8, 128, 128), True),
])
def test_boxes_are_not_mostly_padding(plan, call, box):
    assert bool(plan([call])[0][0]) == box


def convolutions_tested():
    """Those of the GPU tests that compare with the oracle."""
    trained = list(test_gpu_unet_forms.CASES)
    for module in (test_gpu_unet, test_gpu_unet_shapes):
        for mark in module.test_forward_and_gradients_match_oracle.pytestmark:
            if mark.name == "parametrize":
                trained += [getattr(c, "values", c) for c in mark.args[1]]
    return [c for case in trained for c in convolutions(*case)] + [
        c for case in test_gpu_unet_forms.OUTPUT_CASES for c in convolutions(*case, backward=False)]


def test_gpu_tests_run_every_form(plan):
    run = {(*form, sliced) for *form, sliced, _ in plan(convolutions_tested()) if form[0]}
    assert {form[:7] for form in run} == set(plan())
    # crops up to 128^3, half of what a 128^3 crop holds per batch, 6 at most
    reached = {(*form, sliced): (side, batch) for side in range(8, 129, 8)
               for batch in range(1, max(1, min(6, 128 ** 3 // (2 * side ** 3))) + 1)
               for *form, sliced, _ in plan(convolutions(side, batch)) if form[0]}
    missing = {k: v for k, v in reached.items() if k not in run}
    assert not missing, missing
