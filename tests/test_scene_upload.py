"""The host layer's scene upload with a step that fails once (memory that ran
out, say): the next try has to leave the scene on the device that an upload
without the fault leaves. The host sources are compiled against a device that
remembers what it is given, so this runs without a GPU."""

import glob
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_a_failed_upload_is_made_whole_by_the_next(tmp_path):
    csrc = os.path.join(ROOT, "vkrt_amd", "csrc")
    exe = str(tmp_path / "scene_upload")
    # the device calls that an upload does not make stay unresolved and unused
    subprocess.run(["gcc", "-O1", "-std=gnu11", "-I", os.path.join(ROOT, "include"), "-I", csrc, "-I",
                    os.path.join(csrc, "host"), os.path.join(ROOT, "tests", "native", "scene_upload.c"),
                    *sorted(glob.glob(os.path.join(csrc, "host", "*.c"))), "-o", exe, "-Wl,--wrap=malloc",
                    "-Wl,--unresolved-symbols=ignore-all", "-ldl", "-lm", "-lz"], check=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout + run.stderr
