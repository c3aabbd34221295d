"""VCMTracer's merge queue names an eye vertex in one word: every (lane, vertex) that wr_render_vcm takes
(lanes * records below 2^31, records 3 to 35 a path) comes back, on the CPU at the ends of the range and
on the GPU in an image of more than 2^24 pixels."""
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "walkray_amd", "csrc")

PROGRAM = """
#include "merge_entry.h"
int main() {
    for (uint32_t maxv = 3; maxv <= 35; maxv++) {
        const uint32_t lanes = 0x7FFFFFFFu / maxv, at[] = {0, 1, (1u << 22) - 1, (1u << 24) - 1, 1u << 24, (1u << 24) + 5,
                                                         lanes - 1};
        for (uint32_t lane : at)
            for (uint32_t i = 1; i < maxv; i++) {
                const uint32_t w = wr::merge_entry(lane, i, maxv);
                if (wr::merge_lane(w, maxv) != lane || wr::merge_vertex(w, maxv) != i) return 1;
            }
    }
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ is not installed")
def test_entries_come_back(tmp_path):
    src = tmp_path / "m.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(tmp_path / "m")], check=True)
    assert subprocess.run([str(tmp_path / "m")]).returncode == 0


@pytest.mark.gpu
def test_image_of_more_than_2_24_pixels(ctx):
    """A pass whose last rows are past lane 2^24, with 25M merges, which the queue holds.  Rows whose merges
    went elsewhere would stand out: merging makes a quarter of them, and the twenty rows before the line and
    the twenty after it, 82,000 pixels each, differ by 2%."""
    from walkray_amd import _lib as W
    from walkray_amd import scenes as S

    width, height = 4100, 4200
    objs, cam = S.cornell(k=2, width=width, height=height)
    film = W.Film(ctx, width, height)
    W.render_vcm(W.Scene(ctx, objs), cam, film, 1, 1, 3, 0.0003)
    rows = film.read()["mean"].reshape(height, width, 3).mean(axis=(1, 2))
    line = (1 << 24) // width
    before, after = rows[line - 20:line].mean(), rows[line + 1:line + 21].mean()
    assert before > 0
    assert abs(after / before - 1) < 0.1, (before, after)


@pytest.mark.gpu
def test_more_than_2_32_merges(ctx):
    """Two passes side by side with 6.0e9 merges between them, and one after the other with 3.0e9 each: the
    same film (a pixel sums up to 250,000 nonnegative contributions, in runs of different lengths)."""
    from walkray_amd import _lib as W
    from walkray_amd import scenes as S

    objs, cam = S.cornell(k=1, width=160, height=160)
    sc, films = W.Scene(ctx, objs), []
    for calls in ((2,), (1, 1)):
        film = W.Film(ctx, 160, 160)
        for spp in calls:
            W.render_vcm(sc, cam, film, spp, 3, 3, 2.0)
        films.append(film.read()["sum"])
    assert (films[0] > 0).mean() > 0.5
    assert np.allclose(films[0], films[1], rtol=250000 * 2.0 ** -24)
