"""What the library's Makefile builds again, by its own account (nothing is compiled here)."""
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "peregrine_amd", "csrc")


def rebuilt(tmp_path, changed):
    """The sources compiled again after `changed` where everything else is built."""
    objects, out = tmp_path / "obj", tmp_path / "lib"
    objects.mkdir()
    out.mkdir()
    for source in os.listdir(CSRC):
        if source.endswith(".hip"):
            (objects / source.replace(".hip", ".o")).touch()
    (out / "libperegrine_hip.so").touch()
    said = subprocess.run(["make", "-C", CSRC, "-n", "OBJ=%s" % objects, "OUT=%s" % out, "-W", changed, "all"], capture_output=True, text=True, check=True).stdout
    return set(re.findall(r"-c (\S+\.hip)", said))


def test_a_change_of_flags_builds_every_source_again(tmp_path):
    """Objects compiled with other flags are not linked with new ones."""
    assert rebuilt(tmp_path, "Makefile") == {f for f in os.listdir(CSRC) if f.endswith(".hip")}


def test_a_change_of_one_source_builds_that_one_again(tmp_path):
    assert rebuilt(tmp_path, "pg_moe.hip") == {"pg_moe.hip"}
