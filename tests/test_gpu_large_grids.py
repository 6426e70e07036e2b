"""The forms that the solver's operators take on grids past the one-launch limits (16,384 elements for the packed
element-matrix products, 4,096 coarse elements for the restriction, 3,072 of span 4 in FP32) and in their several shares of the work: two
and four coarse layers to a workgroup of the tiled restriction, 16 to 1 slices of the children in the super-element
assembly, several entry tiles to a wavefront in the level-2 product.  The boxes are whole, so every operator has a
closed form: the restriction is the transpose of a product of 1-D hat-function interpolations, and level 2 is
R K P."""
import numpy as np
import pytest

from oracle.solver import build_pch

pytestmark = pytest.mark.gpu


def _solver(shape, super_, precision):
    import torch
    from top_gpu_on_matlab_amd.model import cuboid_model
    from top_gpu_on_matlab_amd.solver import Solver
    s = Solver(cuboid_model(*shape, 1, precision=precision, super_element=super_))
    e = torch.arange(int(np.prod(shape)), dtype=torch.int64)
    ey, ex, ez = e % shape[0], (e // shape[0]) % shape[1], e // (shape[0] * shape[1])
    x = 0.2 + 0.1 * torch.sin(ex / 7.0) * torch.cos(ey / 5.0) * torch.sin(ez / 6.0 + 1)
    E = (1e-6 + x.double() ** 3)
    if super_:  # 64 sub-voxels an element, element-major
        E = (E[:, None] * (1 + 0.3 * torch.sin(torch.arange(64.0, dtype=torch.float64)))[None, :]).reshape(-1)
    s.set_modulus(E.cuda())
    s.assemble()
    return s


def _rel(a, b):
    return float((a - b).abs().max() / b.abs().max())


def _rand(n, seed):
    import torch
    return (2 * torch.rand(n, generator=torch.Generator().manual_seed(seed), dtype=torch.float64) - 1).cuda()


def _hats(coarse, fine):
    """Fine nodes x coarse nodes: the hat functions of a 1-D grid of `coarse` elements at the nodes of `fine`."""
    import torch
    span = fine // coarse
    f = torch.arange(fine + 1, dtype=torch.float64)[:, None] / span
    return (1 - (f - torch.arange(coarse + 1, dtype=torch.float64)[None, :]).abs()).clamp(min=0).cuda()


BOXES = [((104, 104, 104), False),    # level 2: 17,576 elements, two layers, two entry tiles
         ((16, 16, 4128), False),     # level 2: 4 x 4 x 1032 elements, four layers in both precisions
         ((64, 56, 56), False),       # level 2: 3,136 elements, past FP32's limit of the restriction's one launch, not FP64's
         ((8, 8, 8), True), ((24, 24, 24), True), ((32, 32, 32), True), ((40, 40, 40), True),
         ((48, 48, 48), True)]        # 16, 8, 4, 2 slices and one; from 32^3 the finest level takes two launches


@pytest.mark.parametrize('shape, super_', BOXES)
def test_operators_past_the_small_grid_limits(shape, super_):
    """Restriction against the interpolation's transpose (sums of at most 343 FP64 terms with weights that add up to 64:
    1e-13); level 2 as R K P away from the clamped face, level 3's matrices from level 2's with the oracle's
    P_s, in the children's order of the method (a few thousand terms an entry: 1e-12); the element-matrix products,
    alone (1e-13) and in a V-cycle (the coarsest solve passes rounding on: 1e-10), against the full matrices
    split over eight threads; the mixed V-cycle's FP32 forms against the FP64 ones (1e-4)."""
    import torch
    s = _solver(shape, super_, 'fp64')
    dims = [(l['resY'], l['resX'], l['resZ']) for l in s.levels]
    assert dims[0] == shape
    for level in range(2, s.num_levels + 1):
        (fy, fx, fz), (cy, cx, cz) = dims[level - 2], dims[level - 1]
        r = _rand(s.ndof(level - 1), level).reshape(fz + 1, fx + 1, fy + 1, 3)
        got = s.restrict(r.reshape(-1), level).reshape(cz + 1, cx + 1, cy + 1, 3)
        ref = torch.tensordot(_hats(cz, fz), r, ([0], [0]))
        ref = torch.tensordot(_hats(cx, fx), ref, ([0], [1])).transpose(0, 1)
        ref = torch.tensordot(_hats(cy, fy), ref, ([0], [2])).permute(1, 2, 0, 3)
        assert _rel(got, ref) < 1e-13, level
    cy, cx, cz = dims[1]
    u = _rand(s.ndof(2), 12).reshape(cz + 1, cx + 1, cy + 1, 3)
    u[:, :2] = 0  # nothing in the elements at the clamped face
    u = u.reshape(-1)
    assert _rel(s.kbyu(u, 2), s.restrict(s.kbyu(s.interpolate(u, 2)), 2)) < 1e-12
    if s.num_levels > 2:
        cy, cx, cz = dims[2]
        fine = s.ks(2).reshape(cz, 2, cx, 2, cy, 2, 24, 24)
        P = torch.from_numpy(build_pch(2)).cuda()
        ref = 0
        for c in range(8):
            B = P[:, :, c].contiguous()
            K = fine[:, c >> 2, :, (c >> 1) & 1, :, c & 1].reshape(-1, 24, 24)
            ref = ref + B.T @ (K @ B)
        assert _rel(s.ks(3), ref) < 1e-12
    v = _rand(s.ndof(), 3)
    z = s.vcycle(v)
    got = {l: s.kbyu(_rand(s.ndof(l), 20 + l), l) for l in range(1, s.num_levels)}
    s.set_tuning(kelem_parts=8)
    for l in got:
        assert _rel(got[l], s.kbyu(_rand(s.ndof(l), 20 + l), l)) < 1e-13, l
    assert _rel(z, s.vcycle(v)) < 1e-10
    del s
    mixed = _solver(shape, super_, 'mixed')
    assert _rel(mixed.vcycle(v), z) < 1e-4


@pytest.mark.parametrize('shape', [(24, 24, 40), (72, 64, 64), (104, 104, 104)])
def test_restriction_keeps_what_is_not_finite_where_it_has_a_weight(shape):
    """A NaN or infinity of the fine residual on a plane of coarse nodes reaches coarse nodes of that plane alone, and between
    two such planes those two alone: in one launch, and tiled with one and with two layers (levels 2 and 3)."""
    import torch
    s = _solver(shape, False, 'fp64')
    dims = [(l['resY'], l['resX'], l['resZ']) for l in s.levels]
    for level in range(2, s.num_levels + 1):
        (fy, fx, fz), (cy, cx, cz) = dims[level - 2], dims[level - 1]
        span = fz // cz
        for z in (0, span, 2 * span, 2 * span + 1, 3 * span, fz):
            for bad in (float('nan'), float('inf')):
                r = _rand(s.ndof(level - 1), level).reshape(fz + 1, fx + 1, fy + 1, 3)
                r[z, fx // 2, fy // 2] = bad
                got = s.restrict(r.reshape(-1), level).reshape(cz + 1, -1)
                hit = (~torch.isfinite(got)).any(dim=1).cpu().numpy()
                near = np.abs(np.arange(cz + 1) * span - z) < span
                assert np.array_equal(hit, near), (level, z, bad)
