"""The meeting of the workgroups that share a token strip (csrc/strip_meeting.h), in every order its touches of the word can
fall: a part held up anywhere, for however long, leaves neither a word that is not zero nor a share that nobody projects."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_every_order_of_the_touches_ends_at_zero(tmp_path):
    exe = tmp_path / "strip_meeting_orders"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", str(ROOT / "scpaper-2021_amd" / "csrc"),
                    str(ROOT / "tests" / "cpp" / "strip_meeting_orders.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout
    assert res.stdout.count(" 0 wrong") == 14, res.stdout
