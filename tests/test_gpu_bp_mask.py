"""Tiles outside the circle mask, which the back-projection does not sum:
same values as masking the unmasked image, also where samples are not finite
(0 * inf and 0 * NaN are NaN outside the mask too)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bp(x, ang, center, acc, radius, scale):
    from algotom_amd.rec import reconstruction as rec
    return rec._backproject_stack(x, ang, center, acc, mask_radius=radius,
                                  apply_scale=scale)


@pytest.mark.parametrize("acc,nslice", [(0, 1), (1, 5), (2, 3), (3, 2)])
@pytest.mark.parametrize("special", [None, np.inf, np.nan, 3e38])
def test_masked_tiles_equal_masked_image(acc, nslice, special):
    import torch
    ncol, nrow, center, radius = 300, 70, 146.3, 100.0
    gen = torch.Generator(device="cuda").manual_seed(acc)
    x = torch.randn((nrow, nslice, ncol), generator=gen, device="cuda")
    if special is not None:
        x[31, nslice - 1, 7] = special      # reaches corners, not the circle
    ang = np.linspace(0.0, np.pi, nrow, endpoint=False)
    got = _bp(x, ang, center, acc, radius, True)
    full = _bp(x, ang, center, acc, -1.0, False)
    yy, xx = np.mgrid[:ncol, :ncol] - ncol // 2
    inside = torch.from_numpy(xx ** 2 + yy ** 2 <= radius ** 2).cuda()
    # the mask comes before the scale (a masked 3e38 does not overflow)
    want = full.cpu().numpy() * inside.cpu().numpy()[:, None, :].astype(
        np.float32)
    want = want * np.float32(np.pi) / np.float32(nrow - 1)
    assert np.array_equal(got.cpu().numpy(), want, equal_nan=True)
    assert not got.permute(1, 0, 2)[0][~inside].nan_to_num(0).any()


def test_masked_tiles_with_derivative():
    import torch
    from algotom_amd.rec import autograd
    geom = autograd.FBPGeometry(90, 200, ratio=0.5)
    gen = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn((90, 3, 200), generator=gen, device="cuda")
    out, der = geom.backproject_with_derivative(x, 98.6)
    ref = geom.backproject(x, 98.6)
    dref = geom.backproject(x, 98.6, 3)
    assert torch.equal(out, ref) and torch.equal(der, dref)
    yy, xx = np.mgrid[:200, :200] - 100
    outside = torch.from_numpy(xx ** 2 + yy ** 2 > 50 ** 2).cuda()
    assert not out.permute(1, 0, 2)[:, outside].any()
    assert not der.permute(1, 0, 2)[:, outside].any()


def test_masked_tiles_of_a_single_angle():
    """One angle in a batch: the scale divides by nrow - 1 = 0, so a pixel
    outside the mask is 0 / 0 in a skipped tile as in a summed one."""
    from algotom_amd.rec import batch
    rng = np.random.default_rng(3)
    sino = rng.uniform(0.5, 1.0, (1, 300)).astype(np.float32)
    plan = batch.BatchFBP([sino.shape], [149.5], ratio=0.5)
    plan.load([sino])
    plan.run()
    got = plan.results()[0]
    yy, xx = np.mgrid[:300, :300] - 150
    assert np.isnan(got[xx ** 2 + yy ** 2 > 75 ** 2]).all()
