"""The C library's build: it needs no Python, and the build script a Rust host is given watches every source of it."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rustorch_amd", "csrc")


def test_the_default_target_is_the_c_library_alone(tmp_path):
    tools = tmp_path / "bin"  # a PATH without python3
    tools.mkdir()
    for name in ("make", "bash", "sh", "grep", "mkdir"):
        os.symlink(subprocess.check_output(["which", name], text=True).strip(), tools / name)
    r = subprocess.run(["make", "-n", "-B", "-C", CSRC, f"OUTDIR={tmp_path}"], capture_output=True, text=True,
                       env={"PATH": str(tools)})
    assert r.returncode == 0 and not r.stderr, r.stderr
    assert "librt_attn_hip.so" in r.stdout and "pynative" not in r.stdout and "python" not in r.stdout


def test_the_build_script_watches_every_source():
    with open(os.path.join(CSRC, "Makefile")) as f:
        makefile = f.read()
    sources = set(re.search(r"^SRCS\s*:=(.*)$", makefile, re.M).group(1).split())
    headers = {h for h in re.search(r"^HDRS\s*:=(.*)$", makefile, re.M).group(1).split() if "/" not in h}
    with open(os.path.join(ROOT, "INTEGRATION.md")) as f:
        text = f.read()
    listed = re.search(r"for f in \[(.*?)\] \{.*?rerun-if-changed", text, re.S).group(1)
    assert set(re.findall(r'"([^"]+)"', listed)) == sources | headers | {"Makefile"}
    assert sources == {n for n in os.listdir(CSRC) if n.endswith(".hip")}
