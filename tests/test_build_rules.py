"""What a changed file has rebuilt, without building."""
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuv_amd", "csrc")


def _compiled(changed):
    """The objects and device binaries that make would compile if this file were new."""
    out = subprocess.run(["make", "-n", "-W", changed, "-C", CSRC], capture_output=True, text=True, check=True).stdout
    return {os.path.basename(o) for o in re.findall(r" -c -o (\S+)", out)}


def test_other_switches_make_every_object_anew():
    objects = re.findall(r"\$\(OBJDIR\)/([\w.]+)\.o\b", re.search(r"OBJS.*?\n\n", open(os.path.join(CSRC, "Makefile")).read(), re.S)[0])
    device = [o for o in objects if o not in ("api", "plan")]
    made = _compiled("Makefile")
    assert len(objects) > 10 and made >= {o + ".o" for o in objects} | {o + ".hipfb" for o in device} | {"binding.o"}
