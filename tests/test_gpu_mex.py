"""GPU parity of the six MEX entry points (through the C ABI) against the oracle's restatement
of the reference kernels, on reference-shaped inputs."""
import numpy as np
import pytest

from oracle import mesh as M
from oracle import solver as S
from tests.conftest import random_modulus

pytestmark = pytest.mark.gpu


def _ga(a, dtype=None):
    """Column-major numpy array -> GpuArray on the device."""
    import torch
    from top_gpu_on_matlab_amd.mex import GpuArray
    a = np.asarray(a)
    if dtype is not None:
        a = a.astype(dtype)
    flat = torch.from_numpy(np.ascontiguousarray(a.reshape(-1, order='F'))).cuda()
    return GpuArray(flat, a.shape if a.ndim > 1 else (a.shape[0], 1))


def _np(ga):
    return ga.t.cpu().numpy().reshape(ga.dims, order='F')


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
def test_gather_scatter(dtype):
    from top_gpu_on_matlab_amd import mex
    rng = np.random.default_rng(0)
    Nn, Ne = 1000, 700
    eNod = rng.integers(1, Nn + 1, size=(Ne, 8)).astype(np.int32)
    u = rng.standard_normal((Nn, 3)).astype(dtype)
    gU = _ga(u)
    gM = _ga(np.zeros((Ne, 24), dtype))
    mex.Gathering_inplace(gM, gU, _ga(eNod))
    assert np.array_equal(_np(gM), S.gathering(u, eNod))
    mex.Gathering_inplace(gM, gU, _ga(eNod.astype(np.uint32)))      # uint32 indices accepted
    assert np.array_equal(_np(gM), S.gathering(u, eNod))
    V = rng.standard_normal((Ne, 24)).astype(dtype)
    Y0 = rng.standard_normal((Nn, 3)).astype(dtype)
    eBad = eNod.copy()
    eBad[3, 2] = Nn + 5                                              # skipped (Scattering_inplace.cu:70)
    gY = _ga(Y0)
    mex.Scattering_inplace(gY, _ga(eBad), _ga(V))
    ref = S.scattering(Y0.astype(np.float64), eBad, V.astype(np.float64))
    tol = 1e-13 if dtype == np.float64 else 1e-5
    assert np.abs(_np(gY) - ref).max() < tol * np.abs(ref).max()
    keys = rng.integers(0, 130, size=900).astype(np.int32)
    Tm = rng.standard_normal((900, 3)).astype(dtype)
    X0 = np.zeros((120, 3), dtype)
    gX = _ga(X0)
    mex.scatter_accum3_inplace(_ga(keys), _ga(Tm), gX)
    ref = S.scatter_accum3(keys, Tm.astype(np.float64), np.zeros((120, 3)))
    assert np.abs(_np(gX) - ref).max() < tol * np.abs(ref).max()
    # deterministic: a second run gives identical bits
    gX2 = _ga(X0)
    mex.scatter_accum3_inplace(_ga(keys), _ga(Tm), gX2)
    assert np.array_equal(_np(gX), _np(gX2))


def test_assemble_entries_match_oracle():
    from top_gpu_on_matlab_amd import mex
    m = M.build_cuboid_model(8, 16, 8, opt_case=1)
    lv1, lv2, lv3 = m.levels
    E = random_modulus(lv1.numElements, seed=5)
    Pch = S.build_pch(4)
    ref2 = S.assemble_ks_level2(lv2.elementUpwardMap, E, lv1.Ke.reshape(-1, order='F'), Pch, m.mapUniqueKes,
                                m.uniqueKesFree, m.uniqueKesFixed)
    dKs = _ga(np.zeros((24, 24, lv2.numElements)))
    mex.assembleKs_level2_inplace(dKs, _ga(lv2.elementUpwardMap), _ga(E), _ga(lv1.Ke.reshape(-1, order='F')),
                                  _ga(Pch), _ga(m.mapUniqueKes), _ga(m.uniqueKesFree), _ga(m.uniqueKesFixed))
    got2 = _np(dKs)
    assert np.abs(got2 - ref2).max() < 1e-14 * np.abs(ref2).max()
    # empty boundary matrices: every child uses E*K0
    ref2b = S.assemble_ks_level2(lv2.elementUpwardMap, E, lv1.Ke.reshape(-1, order='F'), Pch)
    dKs2 = _ga(np.zeros((24, 24, lv2.numElements)))
    empty = _ga(np.zeros((576, 0)))
    mex.assembleKs_level2_inplace(dKs2, _ga(lv2.elementUpwardMap), _ga(E), _ga(lv1.Ke.reshape(-1, order='F')),
                                  _ga(Pch), _ga(m.mapUniqueKes), empty, empty)
    assert np.abs(_np(dKs2) - ref2b).max() < 1e-14 * np.abs(ref2b).max()
    Psub = S.build_pch(2)
    ref3 = S.assemble_ks_higher_level(lv3.elementUpwardMap, ref2, Psub)
    dKs3 = _ga(np.zeros((24, 24, lv3.numElements)))
    mex.assembleKs_higherLevel_inplace(dKs3, _ga(lv3.elementUpwardMap), _ga(ref2), _ga(Psub))
    assert np.abs(_np(dKs3) - ref3).max() < 1e-14 * np.abs(ref3).max()


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('Ne, nCh', [(1, 1), (70, 3), (65, 8), (130, 64), (3, 70)])
def test_assembly_entries_children_and_element_counts(Ne, nCh, dtype):
    """Children counts that the wavefronts share unevenly and element counts at the edges of the tiles, with voids and
    children with boundary matrices at random, general P: entry by entry within the rounding of a sum of nCh products of two 24-term sums,
    (nCh + 50) unit roundoffs of the same sums over absolute values."""
    from top_gpu_on_matlab_amd import mex
    rng = np.random.default_rng(Ne + nCh)
    nF, nU = 2 * Ne * nCh, 5
    up = np.where(rng.random((Ne, nCh)) < 0.1, 0, rng.integers(1, nF + 1, size=(Ne, nCh))).astype(np.int32)
    E = rng.random(nF).astype(dtype)
    K0, P = rng.standard_normal((24, 24)).astype(dtype), rng.standard_normal((24, 24, nCh)).astype(dtype)
    uid = np.where(rng.random(nF) < 0.3, rng.integers(1, nU + 1, size=nF), 0).astype(np.int32)
    free, fixed = (rng.standard_normal((576, nU)).astype(dtype) for _ in range(2))
    prev = rng.standard_normal((24, 24, nF)).astype(dtype)

    def ref(child):  # the sums and the same of absolute values, in FP64
        out, mag = np.zeros((24, 24, Ne)), np.zeros((24, 24, Ne))
        for e in range(Ne):
            for s in range(nCh):
                if up[e, s] > 0:
                    B = P[:, :, s].astype(np.float64)
                    K, A = child(up[e, s] - 1)
                    out[:, :, e] += B.T @ K @ B
                    mag[:, :, e] += abs(B).T @ A @ abs(B)
        return out, mag

    def level2(f):
        m = float(E[f])
        if uid[f] == 0:
            return K0.astype(np.float64) * m, abs(K0).astype(np.float64) * m
        u, x = (a[:, uid[f] - 1].astype(np.float64).reshape(24, 24, order='F') for a in (free, fixed))
        return u * m + x, abs(u) * m + abs(x)

    eps = (nCh + 50) * np.finfo(dtype).eps
    out, mag = ref(level2)
    g = _ga(np.full((24, 24, Ne), np.nan), dtype)
    mex.assembleKs_level2_inplace(g, _ga(up), _ga(E), _ga(K0.reshape(-1, order='F')), _ga(P), _ga(uid), _ga(free), _ga(fixed))
    assert (abs(_np(g) - out) <= eps * mag).all()
    out, mag = ref(lambda f: (prev[:, :, f].astype(np.float64), abs(prev[:, :, f]).astype(np.float64)))
    g = _ga(np.full((24, 24, Ne), np.nan), dtype)
    mex.assembleKs_higherLevel_inplace(g, _ga(up), _ga(prev), _ga(P))
    assert (abs(_np(g) - out) <= eps * mag).all()


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('Ne, nCh', [(2048, 3), (2049, 3), (2049, 8), (7200, 8), (7200, 64), (2100, 1)])
def test_assembly_entries_many_elements(Ne, nCh, dtype):
    """All three entries with element counts on both sides of the wavefronts' rule and where a wavefront has several
    tiles of the FP64 level-2 product (past 7,168), with voids and children with boundary matrices, general P: the first and
    last elements and a sample of the others, entry by entry within the rounding of sums of nCh products of two 24-term
    sums, of moduli over 64 sub-voxels for super-elements: (nCh + 115) unit roundoffs of the sums over absolute values."""
    from top_gpu_on_matlab_amd import mex
    rng = np.random.default_rng(Ne + nCh)
    nU = 5
    nF = min(2 * Ne * nCh, 100000)
    up = np.where(rng.random((Ne, nCh)) < 0.1, 0, rng.integers(1, nF + 1, size=(Ne, nCh))).astype(np.int32)
    E = rng.random(nF).astype(dtype)
    K0, P = rng.standard_normal((24, 24)).astype(dtype), rng.standard_normal((24, 24, nCh)).astype(dtype)
    uid = np.where(rng.random(nF) < 0.2, rng.integers(1, nU + 1, size=nF), 0).astype(np.int32)
    free, fixed = (rng.standard_normal((576, nU)).astype(dtype) for _ in range(2))
    prev = rng.standard_normal((24, 24, nF)).astype(dtype)
    sub = rng.random((64, nF)).astype(dtype)
    free64 = rng.standard_normal((576, 64, nU)).astype(dtype)
    some = np.unique(np.concatenate([np.arange(3), np.arange(Ne - 70, Ne), rng.integers(0, Ne, 40)]))
    f64 = lambda a: a.astype(np.float64)
    mat = lambda v: v.reshape(24, 24, order='F')

    def higher(f):
        return f64(prev[:, :, f]), abs(f64(prev[:, :, f]))

    def level2(f):
        m = float(E[f])
        if uid[f] == 0:
            return f64(K0) * m, abs(f64(K0)) * m
        u, x = mat(f64(free[:, uid[f] - 1])), mat(f64(fixed[:, uid[f] - 1]))
        return u * m + x, abs(u) * m + abs(x)

    def super_(f):
        if uid[f] == 0:
            return higher(f)
        u, x, m = f64(free64[:, :, uid[f] - 1]), f64(fixed[:, uid[f] - 1]), f64(sub[:, f])
        return mat(u @ m + x), mat(abs(u) @ m + abs(x))

    dup, dP, duid, dfixed, dprev = _ga(up), _ga(P), _ga(uid), _ga(fixed), _ga(prev)
    entries = [
        (level2, lambda g: mex.assembleKs_level2_inplace(g, dup, _ga(E), _ga(K0.reshape(-1, order='F')), dP, duid, _ga(free), dfixed)),
        (higher, lambda g: mex.assembleKs_higherLevel_inplace(g, dup, dprev, dP)),
        (super_, lambda g: mex.assembleKs_level2_superEle_inplace(g, dup, dprev, dP, duid, _ga(sub), _ga(free64), dfixed)),
    ]
    for child, entry in entries:
        g = _ga(np.full((24, 24, Ne), np.nan), dtype)
        entry(g)
        got = _np(g)
        assert np.isfinite(got).all()
        for e in some:
            out, mag = np.zeros((24, 24)), np.zeros((24, 24))
            for s in range(nCh):
                if up[e, s] > 0:
                    B = f64(P[:, :, s])
                    K, A = child(up[e, s] - 1)
                    out += B.T @ K @ B
                    mag += abs(B).T @ A @ abs(B)
            assert (abs(got[:, :, e] - out) <= (nCh + 115) * np.finfo(dtype).eps * mag).all(), (child.__name__, e)


def test_assemble_super_element_entry():
    from top_gpu_on_matlab_amd import mex
    m = M.build_cuboid_model(10, 20, 10, opt_case=2, super_element=True)
    lv1, lv2 = m.levels[0], m.levels[1]
    Esub = random_modulus(64 * lv1.numElements, seed=6).reshape(64, -1, order='F')
    Kmat = m.I_mat @ Esub
    Pch = S.build_pch(4)
    ref = S.assemble_ks_level2_super(lv2.elementUpwardMap, Kmat, Pch, m.mapUniqueKes, Esub, m.uniqueKesFree,
                                     m.uniqueKesFixed)
    for free in (m.uniqueKesFree, m.uniqueKesFree.reshape(576 * 64, -1, order='F')):   # 3-D and 2-D forms
        dKs = _ga(np.zeros((24, 24, lv2.numElements)))
        mex.assembleKs_level2_superEle_inplace(dKs, _ga(lv2.elementUpwardMap), _ga(Kmat), _ga(Pch),
                                               _ga(m.mapUniqueKes), _ga(Esub), _ga(free), _ga(m.uniqueKesFixed))
        assert np.abs(_np(dKs) - ref).max() < 1e-13 * np.abs(ref).max()


def test_entry_errors_on_device_inputs():
    from top_gpu_on_matlab_amd import mex
    from top_gpu_on_matlab_amd._lib import TopGpuError
    u = _ga(np.zeros((10, 3)))
    with pytest.raises(TopGpuError) as ei:
        mex.Gathering_inplace(_ga(np.zeros((4, 24), np.float32)), u, _ga(np.ones((4, 8), np.int32)))
    assert ei.value.identifier == 'Gathering_inplace:Type'
    with pytest.raises(TopGpuError) as ei:
        mex.scatter_accum3_inplace(_ga(np.ones(5, np.int32)), _ga(np.zeros((4, 3))), _ga(np.zeros((3, 3))))
    assert ei.value.identifier == 'scatter_accum3:shape'


def test_entries_accept_empty_inputs():
    """Zero elements (and zero keys) are valid inputs for all six entries: nothing is launched and the
    accumulated outputs keep their values (the reference's kernels run zero blocks)."""
    from top_gpu_on_matlab_amd import mex
    Y0 = np.arange(30, dtype=np.float64).reshape(10, 3)
    u = _ga(Y0)
    gM = _ga(np.zeros((0, 24)))
    mex.Gathering_inplace(gM, u, _ga(np.zeros((0, 8), np.int32)))
    gY = _ga(Y0)
    mex.Scattering_inplace(gY, _ga(np.zeros((0, 8), np.int32)), _ga(np.zeros((0, 24))))
    assert np.array_equal(_np(gY), Y0)
    gX = _ga(Y0)
    mex.scatter_accum3_inplace(_ga(np.zeros(0, np.int32)), _ga(np.zeros((0, 3))), gX)
    assert np.array_equal(_np(gX), Y0)
    m = M.build_cuboid_model(8, 16, 8, opt_case=1)
    lv1 = m.levels[0]
    E = random_modulus(lv1.numElements, seed=5)
    Pch, Psub = S.build_pch(4), S.build_pch(2)
    empty_ks = _ga(np.zeros((24, 24, 0)))
    mex.assembleKs_level2_inplace(empty_ks, _ga(np.zeros((0, 64), np.int32)), _ga(E),
                                  _ga(lv1.Ke.reshape(-1, order='F')), _ga(Pch), _ga(m.mapUniqueKes),
                                  _ga(m.uniqueKesFree), _ga(m.uniqueKesFixed))
    mex.assembleKs_higherLevel_inplace(empty_ks, _ga(np.zeros((0, 8), np.int32)),
                                       _ga(np.zeros((24, 24, 5))), _ga(Psub))
    ms = M.build_cuboid_model(10, 20, 10, opt_case=2, super_element=True)
    Esub = random_modulus(64 * ms.levels[0].numElements, seed=6).reshape(64, -1, order='F')
    mex.assembleKs_level2_superEle_inplace(empty_ks, _ga(np.zeros((0, 64), np.int32)), _ga(ms.I_mat @ Esub),
                                           _ga(Pch), _ga(ms.mapUniqueKes), _ga(Esub), _ga(ms.uniqueKesFree),
                                           _ga(ms.uniqueKesFixed))


def test_scatter_incidence_cache_follows_the_connectivity():
    """The scatter entry points keep the sorted incidence per connectivity; reuse must follow the
    array's content (a connectivity rewritten in place is sorted again) and stay bitwise repeatable."""
    import torch
    from top_gpu_on_matlab_amd import mex
    rng = np.random.default_rng(3)
    Nn, Ne = 3000, 2000
    eA = rng.integers(1, Nn + 1, size=(Ne, 8)).astype(np.int32)
    eB = rng.integers(1, Nn + 1, size=(Ne, 8)).astype(np.int32)
    V = rng.standard_normal((Ne, 24))
    gV = _ga(V)
    gA, gB = _ga(eA), _ga(eB)

    def run(gE):
        gY = _ga(np.zeros((Nn, 3)))
        mex.Scattering_inplace(gY, gE, gV)
        return _np(gY)

    rA, rB = S.scattering(np.zeros((Nn, 3)), eA, V), S.scattering(np.zeros((Nn, 3)), eB, V)
    yA = run(gA)
    assert np.abs(yA - rA).max() < 1e-13 * np.abs(rA).max()
    assert np.array_equal(run(gA), yA)                              # cached: identical bits
    assert np.abs(run(gB) - rB).max() < 1e-13 * np.abs(rB).max()    # a second connectivity
    assert np.array_equal(run(gA), yA)
    gA.t.copy_(torch.from_numpy(np.ascontiguousarray(eB.reshape(-1, order='F'))).cuda())  # rewritten in place
    assert np.abs(run(gA) - rB).max() < 1e-13 * np.abs(rB).max()
    # scatter_accum3: the same keys array rewritten in place
    keys = rng.integers(1, 400, size=5000).astype(np.int32)
    Tm = rng.standard_normal((5000, 3))
    gk, gT = _ga(keys), _ga(Tm)
    for it in range(2):
        gX = _ga(np.zeros((390, 3)))
        mex.scatter_accum3_inplace(gk, gT, gX)
        ref = S.scatter_accum3(keys, Tm, np.zeros((390, 3)))
        assert np.abs(_np(gX) - ref).max() < 1e-13 * np.abs(ref).max()
        keys = rng.integers(1, 400, size=5000).astype(np.int32)
        gk.t.copy_(torch.from_numpy(keys).cuda())


@pytest.mark.parametrize('shift', [0, 1])
@pytest.mark.parametrize('n', [1, 3, 4, 4097, 8_400_003])
def test_scatter_notices_one_changed_key(n, shift):
    """A kept incidence is used again only for the same keys: one key changed in place, at the array's ends and inside,
    of lengths with and without a rest of the hash's groups and of one and of several groups a thread, on an
    array aligned to 16 bytes and one 4 bytes past that.  Whole numbers, so the sums are exact."""
    import torch
    from top_gpu_on_matlab_amd.mex import GpuArray, scatter_accum3_inplace
    M = 50
    rng = np.random.default_rng(n)
    flat = torch.zeros(n + shift, dtype=torch.int32, device='cuda')
    gk = GpuArray(flat[shift:], (n, 1))
    keys = rng.integers(1, M + 1, size=n).astype(np.int32)
    flat[shift:] = torch.from_numpy(keys).cuda()
    vals = rng.integers(-4, 5, size=(n, 3)).astype(np.float64)
    gT = _ga(vals)
    for at in (None, 0, n - 1, n // 2):
        if at is not None:
            keys[at] = keys[at] % M + 1
            gk.t[at] = int(keys[at])
        ref = np.stack([np.bincount(keys - 1, weights=vals[:, c], minlength=M) for c in range(3)], axis=1)
        for _ in range(2):
            gX = _ga(np.zeros((M, 3)))
            scatter_accum3_inplace(gk, gT, gX)
            assert np.array_equal(_np(gX), ref), at
