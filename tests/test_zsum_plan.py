"""The partials of the log-likelihood that a forward pass writes fit the buffer
made for them, whatever the geometry, the subset's length, the tile shape and the
chunks of the rotation; the kernel is one for all subsets of a subset count. On
the CPU: tests/zsum_plan_check.cpp asks the library's own launch plan."""
import subprocess

from host_program import build


def test_partials_fit_their_buffer(tmp_path):
    out = subprocess.run([build("zsum_plan_check.cpp", tmp_path), "1000"], capture_output=True,
                         text=True)
    assert out.returncode == 0, out.stdout
    passes, narrow_short, cut, bad = map(int, out.stdout.split())
    # uneven subsets of narrow waves and cut chunks occur
    assert passes > 50_000 and narrow_short > 1000 and cut > 50 and bad == 0


def test_rows_lie_in_the_volume(tmp_path):
    """The rows of a sample that a wave of 4, 6 or 8 planes loads are planes of
    the volume, also in groups of fewer planes at its ends
    (tests/zsum_rows_check.cpp)."""
    out = subprocess.run([build("zsum_rows_check.cpp", tmp_path)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    samples, ends, irregular, bad = map(int, out.stdout.split())
    assert samples > 100_000 and ends > 1000 and irregular > 1000 and bad == 0
