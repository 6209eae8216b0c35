"""The F stage's assignment of blocks to workgroups: complete, neighbouring
blocks on one XCD, and every XCD used however few the blocks."""
import os
import subprocess

BUILD = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "difx-svn2git-try3_amd", "_build")


def test_places():
    exe = os.path.join(BUILD, "test_place")
    assert os.path.exists(exe), "build first (__graft_entry__.build())"
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
