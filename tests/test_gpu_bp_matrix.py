"""Matrix-core back-projection of stacks (ath_back_projection_matrix).

Bar, against the float64-sum kernel on the same (16-bit: widened) samples:
relative 2-norm error at most max(error of ATH_ACC_F32SEQ, 3e-7).  3e-7 is
the sum of what the design allows at few angles, where a float32 sum after
every angle rounds less often: samples and weights of 22 bits (2^-23 each),
a truncated float32 sum over four angles (3 products at 2^-24 of it, at most
doubled by the difference between a partial sum and the total).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# ncol, nrow, nslice, centre, angle span, edge_pad.  Tiles are 32 x 32 (pairs
# of 16 slices) and 64 x 32 (a last group), steps 4 angles, staged strips end
# at the row's last column pair.
CASES = [
    (65, 37, 5, 32.0, np.pi, False),         # one padded group, odd width
    (64, 4, 16, 31.5, np.pi, True),          # one step
    (97, 5, 17, 96.0, np.pi, True),          # one angle past a step; a pair
    (257, 61, 33, 128.0 - 7.25, 2 * np.pi, True),  # pair + one group
    (130, 181, 48, 3.0, np.pi, False),       # centre at the edge
    (512, 181, 16, 255.1, np.pi, False),     # whole tiles
    (1025, 130, 9, 512.37, np.pi, False),    # one column past 16 tiles
    (7192, 9, 6, 3595.5, 2 * np.pi, False),  # 64-bit offsets, widest windows
]


def _case(ncol, nrow, nslice, span, seed):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((nrow, nslice, ncol), generator=gen, device="cuda")
    ang = np.linspace(0.0, span, nrow, endpoint=False) + 1e-3 * seed
    return x, ang


def _rel(got, ref):
    return ((got.double() - ref.double()).norm() / ref.double().norm()).item()


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_error_against_float64_sums(case, dtype):
    import torch
    from algotom_amd.rec import reconstruction as rec
    ncol, nrow, nslice, center, span, edge = CASES[case]
    print("case", CASES[case], dtype, flush=True)
    x, ang = _case(ncol, nrow, nslice, span, case)
    x = x.to(getattr(torch, dtype))
    ref = rec._backproject_stack(x.float(), ang, center, 0, edge)
    seq = rec._backproject_stack(x.float(), ang, center, 1, edge)
    got = rec._backproject_matrix(x, ang, center,
                                  1 if dtype == "float32" else 2, edge)
    err, bound = _rel(got, ref), max(_rel(seq, ref), 3e-7)
    print("error %.3g, bound %.3g" % (err, bound))
    assert err <= bound


@pytest.mark.parametrize("data", ["noise", "positive", "filtered"])
@pytest.mark.parametrize("ncol,nrow,nslice,center", [
    (64, 128, 6, 31.2),                 # the rule's smallest
    (131, 181, 17, 70.0),               # a pair
    (1025, 128, 33, 512.37),            # a pair and a lone group
    (700, 400, 9, 3.0),                 # half of the pixels' angles in range
    (300, 400, 6, -20.5), (300, 400, 6, 313.0),     # outside the detector
    (513, 901, 6, 250.4)])
def test_error_below_float32_sums(ncol, nrow, nslice, center, data):
    """What sends float32 stacks of 128 and more angles to the matrix cores:
    their error against float64 sums is no larger than that of a float32 sum
    after every angle (no allowance).  Noise, projections of a disc with edge
    padding, and the same filtered."""
    import torch
    from algotom_amd.rec import reconstruction as rec
    x, ang = _case(ncol, nrow, nslice, np.pi, 4)
    edge = data == "positive"
    if data != "noise":
        u = torch.linspace(-1, 1, ncol, device="cuda")
        x = ((2.0 * (1 - u * u).sqrt() + 0.02 * x).abs() + 1e-3).contiguous()
    if data == "filtered":
        pad = min(int(0.15 * ncol), 150)
        taps = rec._window_taps(None, nrow, ncol + 2 * pad, "hann")
        x = rec._filter_stack(x, pad, "edge", False, taps, torch.float32)
    ref = rec._backproject_stack(x, ang, center, 0, edge)
    err = [_rel(rec._backproject_stack(x, ang, center, 1, edge), ref),
           _rel(rec._backproject_matrix(x, ang, center, 1, edge), ref)]
    print("float32 sums %.3g, matrix %.3g" % tuple(err))
    assert err[1] <= err[0]


def test_slice_bits_do_not_depend_on_the_stack():
    """A slice in either group of a pair, in a padded group or beside other
    slices keeps its bits, and so do mask and scale (zero outside the circle).
    (At 200 columns every launch takes pairs of groups.)"""
    import torch
    from algotom_amd.rec import reconstruction as rec
    x, ang = _case(200, 133, 37, np.pi, 3)
    kw = dict(mask_radius=90.0, apply_scale=True)
    full = rec._backproject_matrix(x, ang, 97.6, 1, **kw)
    for j0, j1 in ((0, 5), (20, 36), (36, 37), (3, 33)):
        part = rec._backproject_matrix(x[:, j0:j1].contiguous(), ang, 97.6,
                                       1, **kw)
        assert torch.equal(part, full[:, j0:j1])
    again = rec._backproject_matrix(x, ang, 97.6, 1, **kw)
    assert torch.equal(full, again)
    yy, xx = np.mgrid[:200, :200] - 100
    outside = torch.from_numpy(xx ** 2 + yy ** 2 > 90 ** 2).cuda()
    assert not full.permute(1, 0, 2)[:, outside].any()


def _last_group_alone(ncol, nslice):
    """run_matrix's choice for an odd number of groups: the last one by itself
    (64 x 32 tiles) rather than in a pair (32 x 32) with an idle one."""
    def rounds(tx, ty, units):
        return -(-(-(-ncol // tx) * -(-ncol // ty) * units) // 256)
    pairs, odd = divmod(-(-nslice // 16), 2)
    return bool(odd) and not (
        rounds(32, 32, pairs + 1) * 0.69
        < rounds(32, 32, pairs) * 0.69 + rounds(64, 32, 1) * 0.88)


@pytest.mark.parametrize("ncol,nrow,center,edge", [
    (1025, 721, 512.37, False), (1025, 200, 1021.5, True),
    # at angle 0 every block's lowest position is an even column and 3/4 of
    # the slack 2^-20, and the columns out of range end in the left half of
    # a 64-column tile
    (1065, 160, 2.0 + 3 * 2.0 ** -22, False),
    (1065, 160, 2.0 + 3 * 2.0 ** -22, True)])
def test_slice_bits_do_not_depend_on_the_tile_shape(ncol, nrow, center, edge):
    """Slices whose group is launched alone (64 x 32 tiles) have the bits that
    they have in a pair (32 x 32 tiles), also in blocks whose tile of one
    shape lies within the row and whose tile of the other does not."""
    import torch
    from algotom_amd.rec import reconstruction as rec
    nslice = 48
    assert _last_group_alone(ncol, nslice) and not _last_group_alone(ncol, 32)
    x, ang = _case(ncol, nrow, nslice, np.pi, 1)
    ang[::2] = 0.0
    kw = dict(edge_pad=edge, mask_radius=ncol / 2)
    full = rec._backproject_matrix(x, ang, center, 1, **kw)
    pair = rec._backproject_matrix(x[:, 16:].contiguous(), ang, center, 1,
                                   **kw)
    assert torch.equal(full[:, 16:], pair)


def test_large_stacks_in_parts(monkeypatch):
    """A stack of more than 2 GiB of split samples is summed in parts: same
    bits, bounded workspace; without room for it the vector kernel's."""
    import torch
    from algotom_amd import _native as nat
    from algotom_amd.rec import reconstruction as rec
    nrow, nslice, ncol = 4096, 1100, 128     # 64 + 5 groups
    size = nat.load().ath_back_projection_matrix_workspace_bytes
    assert size(nat.ATH_F32, nrow, nslice, ncol) < (2 << 30) + (1 << 24)
    assert size(nat.ATH_F32, nrow, 32, ncol) < (65 << 20)
    x, ang = _case(ncol, nrow, nslice, np.pi, 2)
    x[3, 1030, 5] = float("inf")
    full = rec._backproject_matrix(x, ang, 63.7, 1)
    for j0, j1 in ((0, 7), (1008, 1040), (1088, 1100)):
        part = rec._backproject_matrix(x[:, j0:j1].contiguous(), ang, 63.7, 1)
        assert np.array_equal(part.cpu().numpy(),
                              full[:, j0:j1].cpu().numpy(), equal_nan=True)

    def no_room(*args):
        raise torch.OutOfMemoryError("no room")

    y = x[:, :20].contiguous()
    del x, full
    monkeypatch.setattr(rec, "_matrix_workspace", no_room)
    assert torch.equal(rec._backproject_matrix(y, ang, 63.7, 1),
                       rec._backproject_stack(y, ang, 63.7, 1))


def test_scales_and_special_samples():
    """Slices of any magnitude keep their relative error; an all-zero slice
    gives zeros; slices with inf, NaN or huge samples are exactly the vector
    kernel's and leave their neighbours untouched."""
    import torch
    from algotom_amd.rec import reconstruction as rec
    x, ang = _case(96, 140, 12, np.pi, 5)
    x[:, 1] *= 1e-38
    x[:, 2] *= 1e25
    x[:, 3] = 0
    x[:, 4, 1:] = 0          # one sample among zeros
    clean = rec._backproject_matrix(x, ang, 47.2, 1)
    ref = rec._backproject_stack(x, ang, 47.2, 0)
    for j in (0, 1, 2, 4):
        scale = ref[:, j].double().abs().max()
        assert _rel(clean[:, j].double() / scale,
                    ref[:, j].double() / scale) <= 5e-7, j
    assert not clean[:, 3].any()
    y = x.clone()
    y[7, 6, 40] = float("inf")
    y[9, 8, 11] = float("nan")
    y[3, 9, 50] = 3e38
    got = rec._backproject_matrix(y, ang, 47.2, 1)
    vec = rec._backproject_stack(y, ang, 47.2, 1)
    for j in range(12):
        want = vec[:, j] if j in (6, 8, 9) else clean[:, j]
        assert np.array_equal(got[:, j].cpu().numpy(), want.cpu().numpy(),
                              equal_nan=True), j


def _outliers(x, kind):
    """A stack whose slices 1 .. have huge samples among ordinary ones."""
    nrow, _, ncol = x.shape
    gen = np.random.default_rng(7)
    if kind == "one sample":
        for j, v in enumerate((1e20, -3e6, 2.0 ** 99, 7e30), 1):
            x[37 + j, j, 11 * j] = v
    elif kind == "hot column":      # beside, at and far from the centre
        for j, c in enumerate((0, 70, 47, ncol - 1), 1):
            x[:, j, c] *= 1e9
    else:                           # a sample of every 3rd row
        for j in range(1, 5):
            rows = np.arange(0, nrow, 3)
            x[rows, j, gen.integers(0, ncol, rows.size)] = 1e12
    return x


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("kind", ["one sample", "hot column", "scattered"])
def test_ordinary_samples_beside_huge_ones(kind, dtype):
    """Finite outliers do not flush the other samples of their slice: such
    slices are exactly the vector kernel's, the others' bits stay."""
    import torch
    from algotom_amd.rec import reconstruction as rec
    x, ang = _case(150, 200, 9, np.pi, 6)
    x = x.to(getattr(torch, dtype))
    acc = 1 if dtype == "float32" else 2
    clean = rec._backproject_matrix(x, ang, 77.3, acc, True)
    y = _outliers(x.clone(), kind)
    got = rec._backproject_matrix(y, ang, 77.3, acc, True)
    vec = rec._backproject_stack(y, ang, 77.3, acc, True)
    assert torch.equal(got[:, 1:5], vec[:, 1:5])
    for j in (0, 5, 8):
        assert torch.equal(got[:, j], clean[:, j])
        assert not torch.equal(got[:, j], vec[:, j])   # not redone


@pytest.mark.parametrize("nrow", [128, 400])
@pytest.mark.parametrize("data", ["noise", "2 orders of columns", "tails",
                                  "object in air"])
def test_small_samples_that_are_kept(nrow, data):
    """Slices with a large range that stay on the matrix cores: the error in
    every ring of pixels is at most that of a float32 sum after every angle
    (2-norm over the ring)."""
    import torch
    from algotom_amd.rec import reconstruction as rec
    ncol, cen = 160, 79.6
    x, ang = _case(ncol, nrow, 6, np.pi, 8)
    col = torch.arange(ncol, device="cuda") - cen
    if data == "noise":
        x[5, :, 3] = 2.0 ** 13      # an outlier within the range
    elif data == "2 orders of columns":
        x = x * torch.where(col.abs() < 40, 1.0, 100.0)
    elif data == "tails":           # a narrow object's filtered tails
        x = x * torch.exp2(-(col.abs() / 6))
    else:                           # a blurred one, air down to 2^-32 of it
        x = x.abs() * torch.exp2(-((col.abs() - 12).clamp(min=0) / 2))
    x = x.contiguous()
    ref = rec._backproject_stack(x, ang, cen, 0, True)
    seq = rec._backproject_stack(x, ang, cen, 1, True)
    got = rec._backproject_matrix(x, ang, cen, 1, True)
    assert not torch.equal(got, seq)
    r = torch.from_numpy(np.hypot(*(np.mgrid[:ncol, :ncol] - 79.5))).cuda()
    for lo in range(0, 80, 16):
        ring = ((r >= lo) & (r < lo + 16))[:, None, :].expand_as(ref)
        err, bound = _rel(got[ring], ref[ring]), _rel(seq[ring], ref[ring])
        print("%s %d angles, ring %d: %.3g, %.3g" % (data, nrow, lo, err,
                                                     bound))
        assert err <= bound


def test_fbp_dispatch_and_graph_replay():
    """fbp_reconstruction takes the matrix path by its rule, a batch member
    gets the single call's bits, also from a replayed graph."""
    import torch
    from algotom_amd.rec import batch, reconstruction as rec
    rng = np.random.default_rng(2)
    sinos = [rng.uniform(0.1, 1, (131, 6, 90)).astype(np.float32),
             rng.uniform(0.1, 1, (60, 5, 64)).astype(np.float32),
             rng.uniform(0.1, 1, (131, 90)).astype(np.float32)]
    assert rec._matrix_stack(131, 6, 90, 1, torch.float32)
    assert not rec._matrix_stack(60, 5, 64, 1, torch.float32)
    plan = batch.BatchFBP([s.shape for s in sinos], [44.2, 31.0, 45.0],
                          apply_log=True)
    plan.load(sinos)
    plan.capture()
    for _ in range(3):
        torch.randn(1 << 18, device="cuda").sum().item()
        for o in plan.outputs:
            o.fill_(7.0)
        plan.run()
        torch.cuda.synchronize()
        for s, c, g in zip(sinos, [44.2, 31.0, 45.0], plan.results()):
            ref = rec.fbp_reconstruction(s.copy(), c, apply_log=True)
            assert np.array_equal(g, ref), s.shape
