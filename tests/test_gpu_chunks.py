"""Windows cut into few and many chunks: the record reduction at the chunk counts where it changes (sums of eight loads at
a time, one entry per thread below 64 chunks and four wavefronts per entry from there), and the default chunk size."""
import numpy as np
import pytest

import cuvslam_amd as ca

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [1, 2, 7, 8, 9, 16, 23, 24, 25, 31, 33, 40, 63, 64, 65, 97])
def test_reduced_system_does_not_depend_on_the_chunk_count(chunks):
    # a Schur tile holds 16 points, so 16 points per tile and one tile per chunk give the wanted count
    p, _, _ = ca.scene.generate(seed=3, num_points=16 * chunks, num_keyframes=8, num_fixed_keyframes=2, z_min=8.0,
                                xy_extent=2.0)
    fine = ca.SchurComplementBundlerGpu(loss=ca.LOSS_HUBER, chunk_pairs=1)
    whole = ca.SchurComplementBundlerGpu(loss=ca.LOSS_HUBER, chunk_pairs=1 << 20)
    a, b = fine.batch([p]), whole.batch([p])
    assert a.info()["chunks"] == chunks and b.info()["chunks"] == 1
    S, e, *_ = a.debug_step(1e-3)
    S1, e1, *_ = b.debug_step(1e-3)
    # FP32 sums of `chunks` records instead of one running sum, relative to the reduced system's own rounding bound
    assert np.linalg.norm(S - S1) <= 2e-5 * np.linalg.norm(S1)
    assert np.linalg.norm(e - e1) <= 2e-5 * np.linalg.norm(e1)


@pytest.mark.parametrize("points, key_frames", [(16, 5), (300, 6), (2000, 7), (3000, 40)])
def test_default_chunks_match_one_chunk(points, key_frames):
    p, _, _ = ca.scene.generate(seed=4, num_points=points, num_keyframes=key_frames, num_fixed_keyframes=3, max_iterations=6)
    out = []
    for chunk_pairs in (0, 1 << 20):
        q = p.copy()
        assert ca.SchurComplementBundlerGpu(loss=ca.LOSS_STUDENT_T, fixed_iterations=True, chunk_pairs=chunk_pairs).solve(q)
        out.append(q)
    assert abs(out[0].last_cost_f64 - out[1].last_cost_f64) <= 1e-6 * out[1].last_cost_f64


@pytest.mark.parametrize("points, key_frames", [(40, 4), (200, 5), (2000, 7)])
def test_autotuner_times_the_default(points, key_frames, tmp_path):
    # below a tile per workgroup of the chip the default is one tile per chunk; two tiles per chunk take 1.3 times as long
    # or more, so the tuner must come back with the default's plan (40 points: the default is the smallest size, one pair)
    p, _, _ = ca.scene.generate(seed=4, num_points=points, num_keyframes=key_frames, num_fixed_keyframes=2, max_iterations=7)
    make = lambda **kw: ca.SchurComplementBundlerGpu(loss=ca.LOSS_STUDENT_T, fixed_iterations=True, **kw)  # noqa: E731
    best, _ = make().autotune([p], repeats=10)
    default = make().batch([p]).info()["chunks"]
    assert default > 1 and best > 0 and make(chunk_pairs=best).batch([p]).info()["chunks"] == default
    table = str(tmp_path / "table.txt")
    tuned = make().autotune_table([p], table, repeats=10)
    assert make(chunk_pairs=tuned[0]).batch([p]).info()["chunks"] == default and not tuned[2]
    assert make().autotune_table([p], table) == (tuned[0], tuned[1], True)  # read back from the file
