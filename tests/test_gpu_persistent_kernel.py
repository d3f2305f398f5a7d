"""The persistent batch kernel itself against launches per step: checks less
than 16 steps apart, with which no sample runs on chip.  Fixed steps with many
checks, stops at different steps, and runs that end between two checks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def masks(plb):
    return [plb.mask_spheres((24, 20, 28), 3.0, 5.0, 0.4, 1), plb.mask_noise((32, 16, 24), 2.0, 0.45, 2),
            np.zeros((6, 5, 7), np.uint8), plb.mask_spheres((17, 23, 19), 2.0, 4.0, 0.35, 3),
            plb.mask_noise((40, 36, 44), 2.0, 0.3, 4)]


TAUS, GXS = [0.8, 1.0, 0.7, 0.6, 0.9], [1e-5, 2e-5, 1e-5, 5e-6, 1e-5]
SHAPES = [dict(precision=1, bb_mode=1, index_kind=1, layout=1, ordering=2, brick=(64, 4, 1)),
          dict(precision=0, bb_mode=0, index_kind=0, layout=0),
          dict(precision=2, bb_mode=1, index_kind=1, layout=1, fp16_scale_log2=20, fp16_rounding=1),
          dict(precision=1, bb_mode=1, index_kind=1, layout=1, block_size=128, waves_per_simd=5)]


@pytest.mark.parametrize("kw", SHAPES)
@pytest.mark.parametrize("max_steps,check,tol", [(137, 10, 0.0), (15, 15, 0.0), (7, 15, 0.0), (20_000, 15, 1e-5)])
def test_persistent_kernel_equals_launches_per_step(plb, kw, max_steps, check, tol):
    fl = masks(plb)
    out = []
    for persistent in (False, True):
        b = plb.Batch(fl, TAUS, GXS, **kw)
        try:
            for _ in range(2):   # the second run starts from what the first left
                steps, upd, _ = b.run(max_steps, check, tol, persistent=persistent)
                out.append((list(steps), upd, b.reduce(), [b.read_macros(s) for s in range(len(fl))]))
        finally:
            b.close()
    first, rest = out[0], out[1:]
    assert first[0][2] == 0 and (tol > 0.0 or all(n == max_steps for n in first[0][:2] + first[0][3:]))
    if tol > 0.0:
        stops = [n for k, n in enumerate(first[0]) if k != 2]
        # (some oscillate from one odd-numbered check to the next, and go on to the end)
        assert min(stops) < max_steps and len(set(stops)) >= 2
    for other in rest:
        assert first[:3] == other[:3]
        assert all(np.array_equal(x, y) for x, y in zip(first[3], other[3]))
