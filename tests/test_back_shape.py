"""The windows of the backprojector that a geometry and a tuning (or none) lead
to hold every plane that a tile's samples touch. On the CPU:
tests/back_shape_check.cpp asks the launcher's own choice."""
import subprocess

from host_program import build


def test_windows_hold_every_plane(tmp_path):
    out = subprocess.run([build("back_shape_check.cpp", tmp_path)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    win, views, gather, bad = map(int, out.stdout.split())
    assert win > 10_000 and views > 1000 and gather > 10_000 and bad == 0
