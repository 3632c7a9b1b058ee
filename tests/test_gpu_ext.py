"""GPU tests of the extensions: FP32 sweeps + FP64 refinement, the adjoint
(and its autograd wrapper), and ragged batches in one persistent launch.

Tolerances (normwise, max|err| / max|ref|):
  mixed, 1 or 2 refinements, vs the long-double oracle  <= 1e-12
  mixed, 0 refinements (pure FP32 sweeps)          <= 1e-5
  adjoint FP64 vs the oracle's FP64 adjoint        <= 1e-12 (each output)
  adjoint FP32 vs the same                          <= 1e-5
  central differences, h = 1e-6, vs the adjoint     <= 1e-6 absolute + relative
  ragged vs the oracle per system                   <= 1e-12 FP64, 1e-5 FP32
"""
import numpy as np
import pytest

import oracle
from tests import helpers as H

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tridsolver_amd import api  # noqa: E402
from tridsolver_amd.autograd import trid_solve  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


# --------------------------------------------------------------------------
# FP32 sweeps + FP64 refinement
# --------------------------------------------------------------------------
@pytest.mark.parametrize("dims", [[64, 48, 40], [37, 21, 19], [512, 3, 2], [9, 700, 2],
                                  [1000], [8192, 3], [3, 4096]])
def test_mixed_refinement_accuracy(dims):
    rng = np.random.default_rng(sum(dims))
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    for sd in range(len(dims)):
        xl = oracle.batch_ld(a, b, c, d, ndim=len(dims), solvedim=sd, dims=dims)
        errs = []
        for refine in (0, 1, 2):
            td = dev(d)
            api.mixed_strided_batch(dev(a), dev(b), dev(c), td, solvedim=sd, dims=dims,
                                    refinements=refine, sync=True)
            errs.append(H.norm_rel_err(td.cpu().numpy(), xl))
        assert errs[0] <= 1e-5, errs
        assert errs[1] <= 1e-12, errs
        assert errs[2] <= 1e-12, errs
        assert errs[1] < errs[0]
        assert api.last_config()[0] == 2


# The 512^3 row length along each direction, at a fraction of the grid; the
# shapes the autotuner picked for the mixed solve at 512^3 (M = 16 rows per
# lane, P = 32 lanes, W systems per workgroup, G, variant 3 = a and c in LDS).
N512_CASES = [(0, [512, 40, 6], (16, 32, 4, 8, 3)),
              (1, [48, 512, 6], (16, 32, 8, 16, 3)),
              (2, [48, 6, 512], (16, 32, 16, 16, 3))]


@pytest.mark.parametrize("sd,dims,tuned", N512_CASES)
def test_mixed_one_refinement_n512(sd, dims, tuned):
    """One refinement -- the setting the benchmark reports -- against the
    long-double oracle at N = 512 along x, y and z: with the default shape,
    with the shape tuned at 512^3 forced, and with the shape the autotuner
    picks for this geometry. Each within 1e-12."""
    rng = np.random.default_rng(512 + sd)
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    xl = oracle.batch_ld(a, b, c, d, ndim=3, solvedim=sd, dims=dims)
    ta, tb, tc = dev(a), dev(b), dev(c)
    errs = {}

    def run(tag):
        td = dev(d)
        api.mixed_strided_batch(ta, tb, tc, td, solvedim=sd, dims=dims, refinements=1,
                                sync=True)
        errs[tag] = (H.norm_rel_err(td.cpu().numpy(), xl), api.last_config())

    run("default")
    with api.forced_hybrid(*tuned):
        run("tuned at 512^3")
        assert errs["tuned at 512^3"][1][1:4] == tuned[:3]
    api.autotune_mixed(sd, dims)
    run("autotuned here")
    print("mixed, 1 refinement, solvedim %d dims %s vs long-double oracle: %s"
          % (sd, dims, errs))
    for tag, (err, cfg) in errs.items():
        assert err <= 1e-12, (tag, err, cfg)


def test_mixed_padded_layout():
    rng = np.random.default_rng(77)
    dims = [30, 22, 14]
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    arrs = [H.pad_halo(t, dims) for t in (a, b, c, d)]
    off, pads = H.halo_offset(dims), [t + 2 for t in dims]
    for sd in range(3):
        td = dev(arrs[3])
        api.mixed_strided_batch(*(dev(t) for t in arrs[:3]), td, solvedim=sd, dims=dims,
                                pads=pads, offset=off, refinements=2, sync=True)
        od = arrs[3].copy()
        oracle.batch(arrs[0], arrs[1], arrs[2], od, ndim=3, solvedim=sd, dims=dims, pads=pads,
                     offset=off)
        got = td.cpu().numpy()
        H.assert_norm_close(got, od, np.float64)
        mask = H.pad_halo(np.ones(n, dtype=bool), dims)
        assert np.array_equal(got[~mask], arrs[3][~mask])


def _mixed_lds_shape(dims, sd, W):
    """A valid shape of the mixed kernel with a and c in LDS (M = 16):
    contiguous systems W per workgroup; strided W x-neighbours (64- or
    128-byte rows), P rounded to whole waves."""
    N = dims[sd]
    P = -(-N // 16)
    if sd > 0:
        P = -(-P // (64 // W)) * (64 // W)
    return (16, P, W, 8, 3)


@pytest.mark.parametrize("dims", [[64, 48, 40], [37, 21, 19], [9, 700, 2], [1000, 3]])
def test_mixed_lds_variant(dims):
    """The M = 16 kernels with a and c in LDS (contiguous tiles; strided
    tiles filled by global->LDS loads), forced, against the long-double
    oracle: 2 refinements <= 1e-12, 0 refinements FP32-accurate. Covers
    partial workgroups (n0 not a multiple of W), lanes past N and both row
    widths."""
    rng = np.random.default_rng(sum(dims) + 3)
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    for sd in range(len(dims)):
        xl = oracle.batch_ld(a, b, c, d, ndim=len(dims), solvedim=sd, dims=dims)
        for W in ((1, 4) if sd == 0 else (8, 16)):
            shape = _mixed_lds_shape(dims, sd, W)
            if sd > 0 and shape[1] * W > 512:
                continue  # longer than one 512-thread workgroup holds at this width
            with api.forced_hybrid(*shape):
                errs = []
                for refine in (0, 2):
                    td = dev(d)
                    api.mixed_strided_batch(dev(a), dev(b), dev(c), td, solvedim=sd,
                                            dims=dims, refinements=refine, sync=True)
                    assert api.last_config()[1:4] == shape[:3]
                    errs.append(H.norm_rel_err(td.cpu().numpy(), xl))
            assert errs[0] <= 1e-5 and errs[1] <= 1e-12, (sd, W, errs)


@pytest.mark.parametrize("M", [4, 8])
def test_mixed_register_variant(M):
    """The kernels with every operand in registers (M = 4, 8), forced, along
    x, y and z: 2 refinements <= 1e-12 against the long-double oracle."""
    rng = np.random.default_rng(90 + M)
    dims = [40, 33, 50]
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    for sd in range(3):
        xl = oracle.batch_ld(a, b, c, d, ndim=3, solvedim=sd, dims=dims)
        P = -(-dims[sd] // M)
        W = max(1, 256 // P) if sd == 0 else 4
        with api.forced_hybrid(M, P, W, 8, 0):
            td = dev(d)
            api.mixed_strided_batch(dev(a), dev(b), dev(c), td, solvedim=sd, dims=dims,
                                    refinements=2, sync=True)
            assert api.last_config()[1:4] == (M, P, W)
        assert H.norm_rel_err(td.cpu().numpy(), xl) <= 1e-12


def test_mixed_lds_variant_padded():
    """Halo-padded layout through the LDS variant: results match the oracle
    and the halo is untouched."""
    rng = np.random.default_rng(78)
    dims = [30, 22, 14]
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    arrs = [H.pad_halo(t, dims) for t in (a, b, c, d)]
    off, pads = H.halo_offset(dims), [t + 2 for t in dims]
    for sd in range(3):
        shape = _mixed_lds_shape(dims, sd, 4 if sd == 0 else 16)
        td = dev(arrs[3])
        with api.forced_hybrid(*shape):
            api.mixed_strided_batch(*(dev(t) for t in arrs[:3]), td, solvedim=sd, dims=dims,
                                    pads=pads, offset=off, refinements=2, sync=True)
        od = arrs[3].copy()
        oracle.batch(arrs[0], arrs[1], arrs[2], od, ndim=3, solvedim=sd, dims=dims, pads=pads,
                     offset=off)
        got = td.cpu().numpy()
        H.assert_norm_close(got, od, np.float64)
        mask = H.pad_halo(np.ones(n, dtype=bool), dims)
        assert np.array_equal(got[~mask], arrs[3][~mask])


# --------------------------------------------------------------------------
# FP64 solution of systems stored in FP32 (tridDmtsvStridedBatchMixedF32)
# --------------------------------------------------------------------------
def _f32_case(rng, n):
    return H.diag_dominant(rng, n, np.float32)


@pytest.mark.parametrize("dims", [[64, 48, 40], [37, 21, 19], [512, 3, 2], [9, 700, 2],
                                  [1000], [8192, 3], [3, 4096], [2, 8192], [96, 80, 512]])
def test_mixed_f32_vs_long_double_oracle(dims):
    """The system is the FP32 values promoted to FP64: 0 refinements is
    FP32-accurate, 1 and 2 are within 1e-12 of the long-double oracle's
    solution of that system; d is left as it was."""
    rng = np.random.default_rng(sum(dims) + 11)
    n = int(np.prod(dims))
    a, b, c, d = _f32_case(rng, n)
    ta, tb, tc, td = (dev(t) for t in (a, b, c, d))
    for sd in range(len(dims)):
        xl = oracle.batch_ld(a, b, c, d, ndim=len(dims), solvedim=sd, dims=dims)
        errs = []
        for refine in (0, 1, 2):
            x = api.mixed_f32_strided_batch(ta, tb, tc, td, solvedim=sd, dims=dims,
                                            refinements=refine, sync=True)
            assert api.last_config()[0] == 10
            errs.append(H.norm_rel_err(x.cpu().numpy(), xl))
        assert errs[0] <= 1e-5 and errs[1] <= 1e-12 and errs[2] <= 1e-12, (sd, errs)
        assert errs[1] < errs[0]
        assert np.array_equal(td.cpu().numpy(), d)


def _general_ok(shape):
    """Shapes with a kernel for more than one refinement: the register kernel
    at 8 rows per lane, the contiguous LDS kernel, the wide kernel at 16 rows
    per lane with 64-byte rows."""
    M, _, W, _, V = shape
    return (V == 0 and M == 8) or V == 1 or (V == 3 and (M, W) == (16, 16))


@pytest.mark.parametrize("shape", [(32, 16, 32, 8, 3), (32, 16, 16, 8, 3), (16, 32, 16, 8, 3),
                                   (16, 32, 16, 8, 0), (8, 64, 8, 8, 0)])
def test_mixed_f32_forced_strided_shapes(shape):
    """Each strided kernel shape forced along y and z of a 40 x 30 x 500 grid
    (partial system groups): the wide kernel at 32 rows per lane with 128-
    and 64-byte rows and at 16 with 64-byte rows, the register kernel at 16
    and 8; one refinement, and two (the general refinement loop) where the
    shape has a kernel for it -- elsewhere two are refused."""
    M, P, W, G, V = shape
    rng = np.random.default_rng(M * 7 + V)
    dims = [40, 30, 500]
    n = int(np.prod(dims))
    a, b, c, d = _f32_case(rng, n)
    t = [dev(v) for v in (a, b, c, d)]
    for sd in (1, 2):
        N = dims[sd]
        Pn = -(-N // M)
        if V == 3:  # whole waves: W * P a multiple of 64
            Pn = -(-Pn // (64 // W)) * (64 // W)
        if Pn > P:
            continue  # longer than this shape holds
        xl = oracle.batch_ld(a, b, c, d, ndim=3, solvedim=sd, dims=dims)
        with api.forced_hybrid(M, Pn, W, G, V):
            for refine in (1, 2):
                if refine == 2 and not _general_ok(shape):
                    with pytest.raises(Exception):
                        api.mixed_f32_strided_batch(*t, solvedim=sd, dims=dims,
                                                    refinements=refine, sync=True)
                    continue
                x = api.mixed_f32_strided_batch(*t, solvedim=sd, dims=dims, refinements=refine,
                                                sync=True)
                assert api.last_config()[1:4] == (M, Pn, W)
                assert H.norm_rel_err(x.cpu().numpy(), xl) <= 1e-12, (sd, refine)


@pytest.mark.parametrize("dims,sd,want", [
    ([32, 512, 33], 2, (16, 16, 0)), ([32, 513, 33], 2, (32, 32, 3)),
    ([33, 256, 33], 2, (16, 16, 0)), ([33, 257, 256], 2, (32, 32, 3)),
    ([33, 257, 257], 2, (32, 32, 3)), ([33, 257, 321], 2, (32, 16, 3)),
    ([17, 384, 520], 1, (32, 16, 3)), ([20, 450, 513], 1, (32, 32, 3)),
    ([5, 700, 9], 1, (16, 16, 0))])
def test_mixed_f32_default_strided_shapes(dims, sd, want):
    """The untuned strided shapes on both sides of their rules (512 workgroups of
    32 systems; 8 lanes per system and whole waves at 16 systems), 0 and 1
    refinements, against the long-double oracle of the promoted system at the
    bars of test_mixed_f32_vs_long_double_oracle."""
    rng = np.random.default_rng(sum(dims) + sd)
    a, b, c, d = _f32_case(rng, int(np.prod(dims)))
    xl = oracle.batch_ld(a, b, c, d, ndim=3, solvedim=sd, dims=dims)
    t = [dev(v) for v in (a, b, c, d)]
    for refine, tol in ((0, 1e-5), (1, 1e-12)):
        x = api.mixed_f32_strided_batch(*t, solvedim=sd, dims=dims, refinements=refine, sync=True)
        algo, M, _, W, _ = api.last_config()
        assert (algo, M) == (10, want[0]) and W <= want[1], api.last_config()
        assert H.norm_rel_err(x.cpu().numpy(), xl) <= tol, refine


@pytest.mark.parametrize("dims,sd,want", [
    # one round of workgroups of 16 systems, and one workgroup more
    ([32, 512, 128], 1, (16, 0)), ([32, 512, 129], 1, (32, 3)),
    ([17, 257, 128], 1, (16, 0)), ([17, 257, 129], 1, (32, 3)),
    ([15, 256, 512], 1, (16, 0)), ([15, 256, 513], 1, (32, 3)),
    ([15, 160, 768], 1, (16, 0)), ([15, 160, 769], 1, (32, 3)),
    ([16, 128, 1024], 1, (16, 0)), ([16, 128, 1025], 1, (32, 3))])
def test_mixed_f32_strided_rounds(dims, sd, want):
    """The kernel in registers only while all its workgroups run at once (two waves per
    SIMD), with 0 and 1 refinements, at the bars of test_mixed_f32_vs_long_double_oracle."""
    rng = np.random.default_rng(sum(dims) + sd)
    a, b, c, d = _f32_case(rng, int(np.prod(dims)))
    xl = oracle.batch_ld(a, b, c, d, ndim=3, solvedim=sd, dims=dims)
    t = [dev(v) for v in (a, b, c, d)]
    for refine, tol in ((0, 1e-5), (1, 1e-12)):
        x = api.mixed_f32_strided_batch(*t, solvedim=sd, dims=dims, refinements=refine, sync=True)
        algo, M, _, W, _ = api.last_config()
        assert (algo, M) == (10, want[0]), (api.last_config(), refine)
        assert H.norm_rel_err(x.cpu().numpy(), xl) <= tol, refine


@pytest.mark.parametrize("shape", [(16, 2, 1), (16, 4, 8), (8, 1, 8), (8, 8, 1)])
@pytest.mark.parametrize("N", [512, 300, 700, 37])
def test_mixed_f32_forced_contig_lds(shape, N):
    """The contiguous kernel with a and c kept in LDS (variant 1), forced at
    8 and 16 rows per lane, one-wave and wider workgroups, lengths that are
    not multiples of M and systems of more than 64 lanes (the 9-step PCR),
    at 0, 1 and 2 refinements, against the long-double oracle of the
    promoted system."""
    M, W, G = shape
    dims = [N, 7, 3]
    rng = np.random.default_rng(N * 3 + M + W)
    n = int(np.prod(dims))
    a, b, c, d = _f32_case(rng, n)
    t = [dev(v) for v in (a, b, c, d)]
    P = -(-N // M)
    if W * P > 512:
        W = max(1, 512 // P)
    xl = oracle.batch_ld(a, b, c, d, ndim=3, solvedim=0, dims=dims)
    with api.forced_hybrid(M, P, W, G, 1):
        for refine, tol in ((0, 1e-5), (1, 1e-12), (2, 1e-12)):
            x = api.mixed_f32_strided_batch(*t, solvedim=0, dims=dims, refinements=refine,
                                            sync=True)
            assert api.last_config() == (10, M, P, W, G)
            assert H.norm_rel_err(x.cpu().numpy(), xl) <= tol, (refine, M, P, W)
    assert np.array_equal(t[3].cpu().numpy(), d)


def test_mixed_f32_padded_layout():
    """Halo-padded layout: x gets the solution at the interior offsets and
    keeps its halo."""
    rng = np.random.default_rng(91)
    dims = [30, 22, 14]
    n = int(np.prod(dims))
    a, b, c, d = _f32_case(rng, n)
    arrs = [H.pad_halo(v, dims) for v in (a, b, c, d)]
    off, pads = H.halo_offset(dims), [v + 2 for v in dims]
    t = [dev(v) for v in arrs]
    mask = H.pad_halo(np.ones(n, dtype=bool), dims)
    for sd in range(3):
        x0 = torch.full((arrs[0].size,), 7.0, dtype=torch.float64, device="cuda")
        x = api.mixed_f32_strided_batch(*t, x0, solvedim=sd, dims=dims, pads=pads, offset=off,
                                        refinements=1, sync=True).cpu().numpy()
        want = oracle.batch_ld(a, b, c, d, ndim=3, solvedim=sd, dims=dims)
        assert np.all(x[~mask] == 7.0)
        H.assert_norm_close(x[mask], want, np.float64, tol=1e-12)


@pytest.mark.parametrize("dims,sd", [([9000, 3], 0), ([20000, 2], 0), ([3, 5000], 1),
                                     ([4, 3, 4500], 2), ([2, 9000, 2], 1)])
def test_mixed_long_systems(dims, sd):
    """Systems no mixed kernel holds: the FP64-stored call (kernels up to
    8192 contiguous / 4096 strided rows) runs the FP64 batched solve
    (algorithm 15); the FP32-stored call (kernels up to 8192 rows) promotes
    the batch and runs it too (algorithm 16). Within 1e-12 of the
    long-double oracle of their system at every refinement count; the FP32
    operands are left as they were."""
    rng = np.random.default_rng(sum(dims) + 40)
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    xl = oracle.batch_ld(a, b, c, d, ndim=len(dims), solvedim=sd, dims=dims)
    ta, tb, tc = (dev(t) for t in (a, b, c))
    for refine in (0, 1):
        td = dev(d)
        api.mixed_strided_batch(ta, tb, tc, td, solvedim=sd, dims=dims, refinements=refine,
                                sync=True)
        assert api.last_config()[0] == 15
        assert H.norm_rel_err(td.cpu().numpy(), xl) <= 1e-12
    a32, b32, c32, d32 = _f32_case(rng, n)
    xl32 = oracle.batch_ld(a32, b32, c32, d32, ndim=len(dims), solvedim=sd, dims=dims)
    t32 = [dev(t) for t in (a32, b32, c32, d32)]
    promoted = dims[sd] > 8192
    for refine in (1, 2) if not promoted else (0, 2):
        x = api.mixed_f32_strided_batch(*t32, solvedim=sd, dims=dims, refinements=refine,
                                        sync=True)
        assert api.last_config()[0] == (16 if promoted else 10)
        assert H.norm_rel_err(x.cpu().numpy(), xl32) <= 1e-12
    assert np.array_equal(t32[3].cpu().numpy(), d32)
    if promoted:
        assert api.autotune_mixed_f32(sd, dims) == 0.0  # nothing to tune: recorded


def test_mixed_f32_long_padded():
    """The promoted long-system path on the interior of a halo-padded
    allocation: x's halo is untouched."""
    rng = np.random.default_rng(93)
    dims = [3, 9000, 2]
    n = int(np.prod(dims))
    a, b, c, d = _f32_case(rng, n)
    xl = oracle.batch_ld(a, b, c, d, ndim=3, solvedim=1, dims=dims)
    off, pads = H.halo_offset(dims), [v + 2 for v in dims]
    t = [dev(H.pad_halo(v, dims)) for v in (a, b, c, d)]
    x = dev(np.full(int(np.prod(pads)), 7.0))
    api.mixed_f32_strided_batch(*t, x, solvedim=1, dims=dims, pads=pads, offset=off, sync=True)
    assert api.last_config()[0] == 16
    g = x.cpu().numpy()
    mask = H.pad_halo(np.ones(n, dtype=bool), dims)
    assert np.all(g[~mask] == 7.0)
    assert H.norm_rel_err(g[mask], xl) <= 1e-12


def test_mixed_f32_rejects_bad_arguments():
    rng = np.random.default_rng(92)
    dims = [16, 8, 4]
    a, b, c, d = (dev(v) for v in _f32_case(rng, int(np.prod(dims))))
    with pytest.raises(TypeError):
        api.mixed_f32_strided_batch(a.double(), b.double(), c.double(), d.double(), solvedim=0,
                                    dims=dims)
    with pytest.raises(Exception):  # refinements out of range
        api.mixed_f32_strided_batch(a, b, c, d, solvedim=0, dims=dims, refinements=9, sync=True)
    with api.forced_hybrid(16, 1, 32, 8, 3):  # wide kernel shape on contiguous systems
        with pytest.raises(Exception):
            api.mixed_f32_strided_batch(a, b, c, d, solvedim=0, dims=dims, sync=True)


def test_mixed_lds_rejects_unfit_shapes():
    rng = np.random.default_rng(79)
    dims = [64, 600, 2]
    a, b, c, d = (dev(t) for t in H.diag_dominant(rng, int(np.prod(dims))))
    bad = [(16, 40, 16, 8, 3),   # strided: 640 threads
           (16, 38, 8, 8, 3),    # strided: 304 threads, not whole waves
           (16, 40, 4, 8, 3),    # strided: 32-byte rows
           (8, 76, 8, 8, 3)]     # LDS variant is built for M = 16 only
    for shape in bad:
        with api.forced_hybrid(*shape):
            with pytest.raises(Exception):
                api.mixed_strided_batch(a, b, c, d, solvedim=1, dims=dims, sync=True)


# --------------------------------------------------------------------------
# Adjoint
# --------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims", [[40, 36, 28], [37, 21, 19], [700, 3], [5, 300]])
def test_adjoint_vs_oracle(dims, dtype):
    rng = np.random.default_rng(len(dims) * 31 + dims[0])
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    w = rng.standard_normal(n)
    tol = 1e-12 if dtype == np.float64 else 1e-5
    for sd in range(len(dims)):
        x = d.copy()
        oracle.batch(a, b, c, x, ndim=len(dims), solvedim=sd, dims=dims)
        ref = oracle.adjoint(a, b, c, x, w, ndim=len(dims), solvedim=sd, dims=dims)
        t = [dev(v.astype(dtype)) for v in (a, b, c, x, w)]
        out = api.adjoint_strided_batch(*t, solvedim=sd, dims=dims, grad_a=True, grad_b=True,
                                        grad_c=True, sync=True)
        for got, want in zip(out, ref):
            H.assert_norm_close(got.cpu().numpy(), want, tol=tol)
        # only lam requested: gradients untouched
        lam_only = api.adjoint_strided_batch(*t, solvedim=sd, dims=dims, sync=True)
        assert lam_only[1] is None and lam_only[2] is None and lam_only[3] is None
        H.assert_norm_close(lam_only[0].cpu().numpy(), ref[0], tol=tol)
        # lam alone does not read x: NULL x gives the same bits
        no_x = api.adjoint_strided_batch(t[0], t[1], t[2], None, t[4], solvedim=sd, dims=dims,
                                         sync=True)
        assert np.array_equal(no_x[0].cpu().numpy(), lam_only[0].cpu().numpy())
        with pytest.raises(ValueError):
            api.adjoint_strided_batch(t[0], t[1], t[2], None, t[4], solvedim=sd, dims=dims,
                                      grad_b=True)
        # duality <w, A^-1 d> = <A^-T w, d>
        lam = out[0].cpu().numpy().astype(np.float64)
        assert abs(np.dot(w, x) - np.dot(lam, d)) <= 50 * tol * np.abs(w).sum()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims,sd", [([5000, 3], 0), ([20000, 2], 0), ([3, 9000], 1),
                                     ([4, 3, 9000], 2), ([2, 17000, 2], 1)])
def test_adjoint_long_vs_oracle(dims, sd, dtype):
    """Systems longer than the adjoint kernel holds (FP64 contiguous above
    4096 rows, any above 8192): the transpose's off-diagonals written out,
    A^T lam = w by the batched solve at any length (the one-workgroup hybrid
    or the long-system path), then the gradients. Against the oracle's
    adjoint, with lam alone and with NULL x."""
    rng = np.random.default_rng(sum(dims) + sd)
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    w = rng.standard_normal(n)
    tol = 1e-12 if dtype == np.float64 else 1e-5
    x = d.copy()
    oracle.batch(a, b, c, x, ndim=len(dims), solvedim=sd, dims=dims)
    ref = oracle.adjoint(a, b, c, x, w, ndim=len(dims), solvedim=sd, dims=dims)
    t = [dev(v.astype(dtype)) for v in (a, b, c, x, w)]
    out = api.adjoint_strided_batch(*t, solvedim=sd, dims=dims, grad_a=True, grad_b=True,
                                    grad_c=True, sync=True)
    algo = api.last_config()[0]
    assert algo in (4, 14), algo
    if dims[sd] > 8192 or (dtype == np.float64 and sd == 0):
        assert algo == 14, algo
    for got, want in zip(out, ref):
        H.assert_norm_close(got.cpu().numpy(), want, tol=tol)
    lam_only = api.adjoint_strided_batch(t[0], t[1], t[2], None, t[4], solvedim=sd, dims=dims,
                                         sync=True)
    assert np.array_equal(lam_only[0].cpu().numpy(), out[0].cpu().numpy())


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("M,seg", [(16, 128), (16, 256), (32, 128), (32, 256)])
@pytest.mark.parametrize("dims,sd", [
    ([16, 64, 3], 1), ([37, 65, 2], 1), ([64, 2, 128], 2), ([33, 3, 31], 2), ([5, 1, 1], 1),
    ([32, 256, 2], 1), ([70, 2, 255], 2)])
def test_adjoint_wide(dims, sd, M, seg, dtype):
    """The wide adjoint kernel against the oracle at the parity bars: rows that
    fill the workgroup's chunks exactly (no row past the last is read) and not,
    waves with and without rows past N or systems past n0, one-row systems,
    aligned and misaligned rows, each gradient alone."""
    esize = np.dtype(dtype).itemsize
    W = seg // esize
    per_wave = max(1, 64 // W)
    P = -(-dims[sd] // M)
    P = -(-P // per_wave) * per_wave
    rng = np.random.default_rng(sum(dims) + M)
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    w = rng.standard_normal(n)
    x = d.copy()
    oracle.batch(a, b, c, x, ndim=len(dims), solvedim=sd, dims=dims)
    a, b, c, x, w = (v.astype(dtype) for v in (a, b, c, x, w))
    ref = oracle.adjoint(*(v.astype(np.float64) for v in (a, b, c, x, w)), ndim=len(dims),
                         solvedim=sd, dims=dims)
    tol = 1e-12 if dtype == np.float64 else 1e-5
    t = [dev(v) for v in (a, b, c, x, w)]
    with api.forced_hybrid(M, P, W, 8, 3):
        for want in ((True, True, True), (True, None, None), (None, True, None),
                     (None, None, True), (None, None, None)):
            out = api.adjoint_strided_batch(*t, solvedim=sd, dims=dims, grad_a=want[0],
                                            grad_b=want[1], grad_c=want[2], sync=True)
            for got, exact in zip(out, ref):
                if got is not None:
                    H.assert_norm_close(got.cpu().numpy(), exact, tol=tol)


def test_adjoint_long_autotune():
    """Tuning a geometry the adjoint kernel does not hold records the
    transposed path (nothing to time) and succeeds; the solve then runs it."""
    dims = [9000, 3]
    assert api.autotune_adjoint(torch.float64, 0, dims) == 0.0
    rng = np.random.default_rng(92)
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    w = rng.standard_normal(n)
    x = d.copy()
    oracle.batch(a, b, c, x, ndim=2, solvedim=0, dims=dims)
    ref = oracle.adjoint(a, b, c, x, w, ndim=2, solvedim=0, dims=dims)
    out = api.adjoint_strided_batch(*(dev(v) for v in (a, b, c, x, w)), solvedim=0, dims=dims,
                                    grad_b=True, sync=True)
    assert api.last_config()[0] == 14
    H.assert_norm_close(out[0].cpu().numpy(), ref[0], tol=1e-12)
    H.assert_norm_close(out[2].cpu().numpy(), ref[2], tol=1e-12)


def test_adjoint_long_padded():
    """The long-system adjoint on the interior of a halo-padded allocation:
    the halo of lam and of every gradient is untouched."""
    rng = np.random.default_rng(91)
    dims = [3, 9000, 2]
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    w = rng.standard_normal(n)
    x = d.copy()
    oracle.batch(a, b, c, x, ndim=3, solvedim=1, dims=dims)
    ref = oracle.adjoint(a, b, c, x, w, ndim=3, solvedim=1, dims=dims)
    off, pads = H.halo_offset(dims), [v + 2 for v in dims]
    ins = [dev(H.pad_halo(v, dims)) for v in (a, b, c, x, w)]
    outs = [dev(np.full(int(np.prod(pads)), 7.0)) for _ in range(4)]
    api.adjoint_strided_batch(*ins, solvedim=1, dims=dims, pads=pads, offset=off, lam=outs[0],
                              grad_a=outs[1], grad_b=outs[2], grad_c=outs[3], sync=True)
    assert api.last_config()[0] == 14
    mask = H.pad_halo(np.ones(n, dtype=bool), dims)
    for got, want in zip(outs, ref):
        g = got.cpu().numpy()
        H.assert_norm_close(g[mask], want, tol=1e-12)
        assert np.all(g[~mask] == 7.0)


def _fd_check(a, b, c, d, w, dims, sd, grads, rng, count=100, h=1e-6):
    """Central differences of L = sum(w * A^-1 d) on `count` random entries of
    each of a, b, c, d, evaluated on the GPU; L is summed over the perturbed
    entry's own system only (the other systems do not depend on it)."""
    names = "abcd"
    arrs = [a, b, c, d]
    n = len(d)
    sys_of = np.zeros(n, dtype=np.int64)
    slices = list(H.system_slices(len(dims), sd, dims))
    for k, idx in enumerate(slices):
        sys_of[idx] = k
    td = [dev(t) for t in arrs]
    tw = dev(w)
    picks = {k: rng.choice(n, count, replace=False) for k in range(4)}
    worst = 0.0
    for k in range(4):
        for i in picks[k]:
            idx = torch.from_numpy(slices[sys_of[i]]).cuda()
            vals = []
            for sgn in (1, -1):
                t = td[k].clone()
                t[i] += sgn * h
                args = [td[j] if j != k else t for j in range(4)]
                x = args[3].clone()
                api.trid_strided_batch(args[0], args[1], args[2], x, solvedim=sd, dims=dims)
                vals.append(float((tw[idx] * x[idx]).sum()))
            fd = (vals[0] - vals[1]) / (2 * h)
            g = float(grads[k][i])
            err = abs(fd - g) / max(1.0, abs(g))
            worst = max(worst, err)
            assert err <= 1e-6, (names[k], int(i), fd, g)
    return worst


@pytest.mark.parametrize("sd", [0, 1, 2])
def test_adjoint_central_differences(sd):
    rng = np.random.default_rng(100 + sd)
    dims = [24, 20, 18]
    n = int(np.prod(dims))
    a, b, c, d = H.diag_dominant(rng, n)
    w = rng.standard_normal(n)
    x = d.copy()
    oracle.batch(a, b, c, x, ndim=3, solvedim=sd, dims=dims)
    lam, ga, gb, gc = (t.cpu().numpy() for t in api.adjoint_strided_batch(
        dev(a), dev(b), dev(c), dev(x), dev(w), solvedim=sd, dims=dims, grad_a=True,
        grad_b=True, grad_c=True, sync=True))
    _fd_check(a, b, c, d, w, dims, sd, [ga, gb, gc, lam], rng)


@pytest.mark.parametrize("sd", [0, 1, 2])
def test_config_adjoint_256_fp64(sd):
    """Differentiable solve on 256^3 FP64: forward x = A^-1 d, L = sum(w x),
    w ~ N(0,1); adjoint gradients wrt a, b, c, d vs the CPU FP64 adjoint and
    vs central differences (h = 1e-6) on 100 random entries of each."""
    rng = np.random.default_rng(256 + sd)
    dims = [256, 256, 256]
    n = 256 ** 3
    a, b, c, d = H.diag_dominant(rng, n)
    w = rng.standard_normal(n)
    ta, tb, tc, td = (dev(t) for t in (a, b, c, d))
    tx = td.clone()
    api.trid_strided_batch(ta, tb, tc, tx, solvedim=sd, dims=dims, sync=True)
    x = tx.cpu().numpy()
    out = api.adjoint_strided_batch(ta, tb, tc, tx, dev(w), solvedim=sd, dims=dims,
                                    grad_a=True, grad_b=True, grad_c=True, sync=True)
    lam, ga, gb, gc = (t.cpu().numpy() for t in out)
    ref = oracle.adjoint(a, b, c, x, w, ndim=3, solvedim=sd, dims=dims)
    errs = [H.assert_norm_close(g, r, tol=1e-12) for g, r in zip((lam, ga, gb, gc), ref)]
    worst = _fd_check(a, b, c, d, w, dims, sd, [ga, gb, gc, lam], rng)
    print("adjoint 256^3 sd=%d: vs CPU adjoint %s, worst FD rel err %.2e"
          % (sd, ["%.1e" % e for e in errs], worst))


def test_autograd_gradcheck_and_dense_reference():
    rng = np.random.default_rng(3)
    shape = (5, 4, 6)  # torch order [z, y, x]
    n = int(np.prod(shape))
    a, b, c, d = (dev(t).reshape(shape).requires_grad_() for t in H.diag_dominant(rng, n))
    for sd in range(3):
        assert torch.autograd.gradcheck(lambda *t: trid_solve(*t, sd), (a, b, c, d),
                                        eps=1e-6, atol=1e-8, rtol=1e-6)
    # dense reference on the CPU for solvedim 0 (last torch dim)
    x = trid_solve(a, b, c, d, 0)
    wt = torch.randn_like(x)
    (x * wt).sum().backward()
    A = torch.diag_embed(b.detach().cpu()) + torch.diag_embed(a.detach().cpu()[..., 1:], -1) + \
        torch.diag_embed(c.detach().cpu()[..., :-1], 1)
    Ad = A.clone().requires_grad_()
    dd = d.detach().cpu().clone().requires_grad_()
    xd = torch.linalg.solve(Ad, dd.unsqueeze(-1)).squeeze(-1)
    (xd * wt.cpu()).sum().backward()
    np.testing.assert_allclose(d.grad.cpu().numpy(), dd.grad.numpy(), rtol=1e-12, atol=1e-14)
    np.testing.assert_allclose(b.grad.cpu().numpy(),
                               torch.diagonal(Ad.grad, dim1=-2, dim2=-1).numpy(), rtol=1e-12,
                               atol=1e-14)
    ga = a.grad.cpu().numpy()
    assert np.all(ga[..., 0] == 0)
    np.testing.assert_allclose(ga[..., 1:], torch.diagonal(Ad.grad, -1, -2, -1).numpy(),
                               rtol=1e-12, atol=1e-14)


# --------------------------------------------------------------------------
# Ragged batches
# --------------------------------------------------------------------------
def ragged_case(rng, lens, dtype):
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    a, b, c, d = H.diag_dominant(rng, int(off[-1]), dtype)
    return off, a, b, c, d


def check_ragged(off, a, b, c, d, got, dtype, u0=None):
    want = d.copy()
    u = None if u0 is None else u0.copy()
    oracle.ragged(a, b, c, want, off, u, inc=u0 is not None)
    ref = want if u0 is None else u
    tol = 1e-12 if dtype == np.float64 else 1e-5
    if u0 is None:
        err = H.assert_norm_close(got, ref, dtype, tol=tol)
    else:
        err = H.assert_norm_close(got - u0, ref - u0, dtype, tol=tol)
    # per-system check on a sample
    for s in np.random.default_rng(1).choice(len(off) - 1, min(50, len(off) - 1), False):
        sl = slice(off[s], off[s + 1])
        if off[s + 1] > off[s]:
            x, r = got[sl].astype(np.float64), ref[sl].astype(np.float64)
            assert np.abs(x - r).max() <= tol * max(np.abs(r).max(), 1e-30) * 10
    return err


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("M,launches", [(0, 1), (4, 1), (8, 1), (16, 1), (4, 2), (8, 2),
                                        (16, 2)])
def test_ragged_vs_oracle(dtype, M, launches):
    """Default (tuned or untuned) and forced shapes, in one persistent solve
    launch or split in two (long systems, then the rest)."""
    rng = np.random.default_rng(M + 1)
    max_len = 2048 if M == 4 and dtype == np.float64 else 4096
    lens = np.round(np.exp(rng.uniform(np.log(1), np.log(max_len), 3000))).astype(np.int64)
    lens[:5] = [0, 1, 2, 0, max_len]
    off, a, b, c, d = ragged_case(rng, lens, dtype)
    ctx = api.forced_ragged(M, launches=launches) if M else None
    if ctx:
        ctx.__enter__()
    try:
        for inc in (False, True):
            td = dev(d)
            tu = dev(rng.uniform(-1, 1, len(d)).astype(dtype)) if inc else None
            u0 = None if tu is None else tu.cpu().numpy()
            api.ragged_batch(dev(a), dev(b), dev(c), td, dev(off), max_len=max_len, u=tu,
                             sync=True)
            if M:
                assert api.last_config()[:4:3] == (5, launches)  # (algorithm, W = launches)
            got = (tu if inc else td).cpu().numpy()
            if inc:
                assert np.array_equal(td.cpu().numpy(), d)
            check_ragged(off, a, b, c, d, got, dtype, u0)
    finally:
        if ctx:
            ctx.__exit__(None, None, None)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("per_cu", [1, 2])
def test_ragged_split_launch(per_cu, dtype):
    """Batch with systems over 4096 rows through the split launch: the long
    systems at 32 rows per lane with `a` moved into the LDS tile by
    global->LDS loads (FP32: two half-wave loads per 64 rows), then the rest.
    Lengths at the class edges (4096, 4097, 8191, 8192 rows), empty and
    one-row systems, plain and Inc, against the oracle; the split is refused
    at other rows per lane and for the mixed solve."""
    rng = np.random.default_rng(33 + per_cu)
    lens = np.round(np.exp(rng.uniform(np.log(1), np.log(8192), 1200))).astype(np.int64)
    lens[:10] = [0, 1, 4096, 4097, 8191, 8192, 2, 0, 5000, 4160]
    off, a, b, c, d = ragged_case(rng, lens, dtype)
    with api.forced_ragged(16, per_cu=per_cu, launches=3):
        for inc in (False, True):
            td = dev(d)
            tu = dev(rng.uniform(-1, 1, len(d)).astype(dtype)) if inc else None
            u0 = None if tu is None else tu.cpu().numpy()
            api.ragged_batch(dev(a), dev(b), dev(c), td, dev(off), max_len=8192, u=tu,
                             sync=True)
            assert api.last_config()[:4:3] == (5, 3)
            got = (tu if inc else td).cpu().numpy()
            if inc:
                assert np.array_equal(td.cpu().numpy(), d)
            check_ragged(off, a, b, c, d, got, dtype, u0)
        if dtype == np.float64:
            with pytest.raises(Exception):
                api.ragged_batch_mixed(dev(a), dev(b), dev(c), dev(d), dev(off), max_len=8192,
                                       sync=True)
    with api.forced_ragged(8, launches=3):
        with pytest.raises(Exception):
            api.ragged_batch(dev(a), dev(b), dev(c), dev(d), dev(off), max_len=4096,
                             sync=True)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("said,longest,count", [(2048, 2048, 3000), (4096, 4096, 2000),
                                                (2048, 1030, 17000), (2048, 8192, 400),
                                                (4096, 8192, 400)])
def test_ragged_default_shapes(said, longest, count, dtype):
    """The untuned shapes, one workgroup per item: lengths at the edges of the
    classes (8 and 16 rows per lane, up to 256 lanes), empty systems, more items
    than the launch has workgroups (17,000 of 1025-1030 rows), and systems longer
    than max_len says, which are solved up to 8192 rows; the arrays start at
    different places inside a 128-byte line. Plain and Inc, against the oracle,
    with the batch's tolerance."""
    rng = np.random.default_rng(said + longest)
    if count == 17000:
        lens = rng.integers(1025, longest + 1, count)
    else:
        lens = np.round(np.exp(rng.uniform(0, np.log(longest), count))).astype(np.int64)
        edges = [0, 1, 2, 8, 9, 16, 17, 511, 512, 513, 1023, 1024, 1025, longest - 1, longest, 0]
        lens[:len(edges)] = edges
    off, a, b, c, d = ragged_case(rng, lens, dtype)
    u = rng.uniform(-1, 1, len(d)).astype(dtype)

    def placed(v, k):
        t = torch.zeros(len(v) + 32, dtype=dev(v).dtype, device="cuda")[k:k + len(v)]
        return t.copy_(torch.from_numpy(v))

    for inc in (False, True):
        td = placed(d, 3)
        tu = placed(u, 7) if inc else None
        api.ragged_batch(placed(a, 0), placed(b, 1), placed(c, 5), td, dev(off), max_len=said,
                         u=tu, sync=True)
        got = (tu if inc else td).cpu().numpy()
        if inc:
            assert np.array_equal(td.cpu().numpy(), d)
        check_ragged(off, a, b, c, d, got, dtype, u if inc else None)


@pytest.mark.parametrize("launches", [0, 1, 2])
@pytest.mark.parametrize("max_len", [2048, 8192])
def test_ragged_mixed_f32_vs_oracle(max_len, launches):
    """FP64 solution of a ragged batch stored in FP32 (empty and one-row
    systems included): 1 and 2 refinements within 1e-12 of the FP64 oracle's
    solution of the promoted values, 0 refinements FP32-accurate; d is not
    written and x keeps its value past the last system. Default launches
    (two where systems may exceed 4096 rows), or forced one or two."""
    rng = np.random.default_rng(max_len + 9)
    lens = np.round(np.exp(rng.uniform(np.log(1), np.log(max_len), 1500))).astype(np.int64)
    lens[:5] = [0, 1, 2, 0, max_len]
    off, a, b, c, d = ragged_case(rng, lens, np.float32)
    # three elements past the last system, which no system owns
    a, b, c, d = (np.concatenate([v, np.full(3, 2.0, np.float32)]) for v in (a, b, c, d))
    want = d.astype(np.float64)
    oracle.ragged(*(v.astype(np.float64) for v in (a, b, c)), want, off)
    t = [dev(v) for v in (a, b, c, d)]
    toff = dev(off)
    want_launches = launches or (2 if max_len > 4096 else 1)
    ctx = api.forced_ragged(16, launches=launches) if launches else None
    if ctx:
        ctx.__enter__()
    try:
        for refine, tol in ((0, 1e-5), (1, 1e-12), (2, 1e-12)):
            x0 = torch.full((len(d),), 3.0, dtype=torch.float64, device="cuda")
            x = api.ragged_batch_mixed_f32(*t, toff, x0, max_len=max_len, refinements=refine,
                                           sync=True).cpu().numpy()
            assert api.last_config()[:4:3] == (11, want_launches)
            n = int(off[-1])
            err = H.assert_norm_close(x[:n], want[:n], np.float64, tol=tol)
            if refine == 0:
                assert err > 1e-12
            assert np.all(x[n:] == 3.0)
    finally:
        if ctx:
            ctx.__exit__(None, None, None)
    assert np.array_equal(t[3].cpu().numpy(), d)


def test_ragged_too_long_is_reported():
    rng = np.random.default_rng(4)
    off, a, b, c, d = ragged_case(rng, [10, 9000, 5], np.float64)
    td = dev(d)
    with pytest.raises(Exception):
        api.ragged_batch(dev(a), dev(b), dev(c), td, dev(off), max_len=8192, sync=True)
    with pytest.raises(Exception):  # max_len beyond what the kernel supports
        api.ragged_batch(dev(a), dev(b), dev(c), td, dev(off), max_len=100000, sync=True)


def test_mixed_f32_graph_replay():
    """The FP32-stored solves (strided along z, and ragged with its workspace
    reserved first) captured once into one hipGraph and replayed several times
    with eager work in between: every replay equals the eager results."""
    rng = np.random.default_rng(17)
    dims = [64, 40, 96]
    a, b, c, d = (dev(v) for v in _f32_case(rng, int(np.prod(dims))))
    lens = np.round(np.exp(rng.uniform(np.log(8), np.log(4096), 300))).astype(np.int64)
    off, ra, rb, rc, rd = ragged_case(rng, lens, np.float32)
    r = [dev(v) for v in (ra, rb, rc, rd)]
    toff = dev(off)
    eager_s = api.mixed_f32_strided_batch(a, b, c, d, solvedim=2, dims=dims, sync=True)
    eager_r = api.ragged_batch_mixed_f32(*r, toff, max_len=4096, sync=True)
    s = torch.cuda.Stream()
    xs = torch.empty_like(eager_s)
    xr = torch.empty_like(eager_r)
    with torch.cuda.stream(s):
        assert api._lib.lib().tridHipSetStream(api.C.c_void_p(s.cuda_stream)) == 0
        assert api._lib.lib().tridHipReserveWorkspace(
            api._lib.lib().tridHipRaggedWorkspaceBytes(len(lens))) == 0
        api.mixed_f32_strided_batch(a, b, c, d, xs, solvedim=2, dims=dims, stream=s)
        api.ragged_batch_mixed_f32(*r, toff, xr, max_len=4096, stream=s)  # warm-up
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        api.mixed_f32_strided_batch(a, b, c, d, xs, solvedim=2, dims=dims, stream=s)
        api.ragged_batch_mixed_f32(*r, toff, xr, max_len=4096, stream=s)
    for k in range(4):
        xs.zero_()
        xr.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(xs, eager_s) and torch.equal(xr, eager_r), k
        d.mul_(1.0)  # eager work between replays
    api.use_torch_stream(torch.cuda.default_stream())


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_ragged_graph_replay(dtype):
    """Capture the planning kernels and the persistent solve once; replay it
    several times with eager work in between; every replay equals the eager
    result."""
    rng = np.random.default_rng(9)
    lens = np.round(np.exp(rng.uniform(np.log(8), np.log(4096), 500))).astype(np.int64)
    off, a, b, c, d = ragged_case(rng, lens, dtype)
    ta, tb, tc, toff = dev(a), dev(b), dev(c), dev(off)
    t_in = dev(d)
    eager = t_in.clone()
    api.ragged_batch(ta, tb, tc, eager, toff, max_len=4096, sync=True)
    s = torch.cuda.Stream()
    work = torch.empty_like(t_in)
    with torch.cuda.stream(s):
        # workspace must exist before capture
        assert api._lib.lib().tridHipSetStream(api.C.c_void_p(s.cuda_stream)) == 0
        assert api._lib.lib().tridHipReserveWorkspace(
            api._lib.lib().tridHipRaggedWorkspaceBytes(len(lens))) == 0
        work.copy_(t_in)
        api.ragged_batch(ta, tb, tc, work, toff, max_len=4096, stream=s)  # warm-up
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        api.ragged_batch(ta, tb, tc, work, toff, max_len=4096, stream=s)
    for k in range(4):
        work.copy_(t_in)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(work, eager), k
        t_in.mul_(1.0)  # eager work between replays
    api.use_torch_stream(torch.cuda.default_stream())


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_config_ragged_40k_graph(dtype):
    """The 40,000-system config as a hipGraph-captured repeat: planning
    kernels and the persistent solve captured once, replayed with eager work
    in between; every replay equals the eager solve bit for bit, and the
    replayed result matches the oracle."""
    rng = np.random.default_rng(40000)
    lens = np.round(np.exp(rng.uniform(np.log(8), np.log(8192), 40000))).astype(np.int64)
    off, a, b, c, d = ragged_case(rng, lens, dtype)
    ta, tb, tc, toff, t_in = dev(a), dev(b), dev(c), dev(off), dev(d)
    eager = t_in.clone()
    api.ragged_batch(ta, tb, tc, eager, toff, max_len=8192, sync=True)
    s = torch.cuda.Stream()
    work = torch.empty_like(t_in)
    with torch.cuda.stream(s):
        api.reserve_workspace(api.ragged_workspace_bytes(len(lens)), stream=s)
        work.copy_(t_in)
        api.ragged_batch(ta, tb, tc, work, toff, max_len=8192, stream=s)  # warm-up
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        api.ragged_batch(ta, tb, tc, work, toff, max_len=8192, stream=s)
    try:
        for k in range(3):
            work.copy_(t_in)
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(work, eager), k
            t_in.mul_(1.0)  # eager work between replays
    finally:
        api.use_torch_stream(torch.cuda.default_stream())
    err = check_ragged(off, a, b, c, d, work.cpu().numpy(), dtype)
    print("ragged 40k %s graph replay: config %s, normwise rel err vs oracle %.2e"
          % (np.dtype(dtype).name, api.last_config(), err))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_config_ragged_40k(dtype):
    """40,000 systems, lengths round(exp(U(ln 8, ln 8192))) (FP32: up to 8192
    with M = 8), diagonally dominant; one persistent launch vs the oracle."""
    rng = np.random.default_rng(40000)
    lens = np.round(np.exp(rng.uniform(np.log(8), np.log(8192), 40000))).astype(np.int64)
    off, a, b, c, d = ragged_case(rng, lens, dtype)
    td = dev(d)
    api.ragged_batch(dev(a), dev(b), dev(c), td, dev(off), max_len=8192, sync=True)
    err = check_ragged(off, a, b, c, d, td.cpu().numpy(), dtype)
    print("ragged 40k %s: %d unknowns, config %s, normwise rel err vs oracle %.2e"
          % (np.dtype(dtype).name, off[-1], api.last_config(), err))


@pytest.mark.parametrize("refine", [1, 2])
def test_config_ragged_40k_mixed(refine):
    """The 40,000-system ragged config (lengths round(exp(U(ln 8, ln 8192))))
    by FP32 sweeps + FP64 refinement, default launches (two: the systems over
    4096 rows, then the rest): within 1e-12 of the FP64 oracle."""
    rng = np.random.default_rng(40000)
    lens = np.round(np.exp(rng.uniform(np.log(8), np.log(8192), 40000))).astype(np.int64)
    off, a, b, c, d = ragged_case(rng, lens, np.float64)
    td = dev(d)
    api.ragged_batch_mixed(dev(a), dev(b), dev(c), td, dev(off), max_len=8192,
                           refinements=refine, sync=True)
    assert api.last_config()[:2] == (9, 16)
    err = check_ragged(off, a, b, c, d, td.cpu().numpy(), np.float64)
    print("ragged 40k mixed, %d refinements: normwise rel err vs FP64 oracle %.2e"
          % (refine, err))


@pytest.mark.parametrize("M,launches", [(0, 2), (4, 1), (8, 1), (16, 1), (16, 2)])
def test_ragged_mixed_vs_oracle(M, launches):
    """FP64 ragged batch by FP32 sweeps + FP64 refinement: within 1e-12 of the
    FP64 oracle after 2 refinements; 0 refinements is an FP32-accurate solve.
    M = 4 and 8 keep every operand in registers, M = 16 (the default) keeps
    a and c in LDS, in one solve launch or split in two (the default when
    systems may exceed 4096 rows)."""
    rng = np.random.default_rng(40 + M)
    max_len = {4: 2048, 8: 4096}.get(M, 8192)
    lens = np.round(np.exp(rng.uniform(np.log(1), np.log(max_len), 2000))).astype(np.int64)
    lens[:5] = [0, 1, 2, 0, max_len]
    off, a, b, c, d = ragged_case(rng, lens, np.float64)
    ctx = api.forced_ragged(M, launches=launches) if M else None
    if ctx:
        ctx.__enter__()
    try:
        td = dev(d)
        api.ragged_batch_mixed(dev(a), dev(b), dev(c), td, dev(off), max_len=max_len,
                               refinements=2, sync=True)
        assert api.last_config()[:4:3] == (9, launches)
        check_ragged(off, a, b, c, d, td.cpu().numpy(), np.float64)
        t1 = dev(d)  # one refinement: the setting the benchmark reports
        api.ragged_batch_mixed(dev(a), dev(b), dev(c), t1, dev(off), max_len=max_len,
                               refinements=1, sync=True)
        xl = oracle.ragged_ld(a, b, c, d, off)
        assert H.norm_rel_err(t1.cpu().numpy(), xl) <= 1e-12
        t0 = dev(d)
        api.ragged_batch_mixed(dev(a), dev(b), dev(c), t0, dev(off), max_len=max_len,
                               refinements=0, sync=True)
        want = d.copy()
        oracle.ragged(a, b, c, want, off)
        err = H.norm_rel_err(t0.cpu().numpy(), want)
        assert 1e-12 < err <= 1e-5  # FP32 accuracy without refinement
    finally:
        if ctx:
            ctx.__exit__(None, None, None)


def test_ragged_mixed_rejects():
    rng = np.random.default_rng(41)
    off, a, b, c, d = ragged_case(rng, [10, 9000, 5], np.float64)
    with pytest.raises(Exception):  # longer than 8192
        api.ragged_batch_mixed(dev(a), dev(b), dev(c), dev(d), dev(off), max_len=9000,
                               sync=True)
    with pytest.raises(Exception):  # max_len within the limit, one system beyond it
        api.ragged_batch_mixed(dev(a), dev(b), dev(c), dev(d), dev(off), max_len=8192,
                               sync=True)
    off, a, b, c, d = ragged_case(rng, [10, 5000, 5], np.float64)
    with api.forced_ragged(8):  # all operands in registers: 4096 rows at most
        with pytest.raises(Exception):
            api.ragged_batch_mixed(dev(a), dev(b), dev(c), dev(d), dev(off), max_len=5000,
                                   sync=True)
    off, a, b, c, d = ragged_case(rng, [10, 4000, 5], np.float64)
    with api.forced_ragged(4):  # 2048 rows at most; max_len promises less than needed
        with pytest.raises(Exception):
            api.ragged_batch_mixed(dev(a), dev(b), dev(c), dev(d), dev(off), max_len=1000,
                                   sync=True)
    with pytest.raises(TypeError):
        api.ragged_batch_mixed(dev(a.astype(np.float32)), dev(b.astype(np.float32)),
                               dev(c.astype(np.float32)), dev(d.astype(np.float32)), dev(off),
                               max_len=4096)


def _adjoint_config(dims, sd, dtype, grads):
    """The shape an untuned adjoint of the batch takes, on random operands."""
    n = int(np.prod(dims))
    t = torch.float64 if dtype == np.float64 else torch.float32
    a, c, x, w = (torch.rand(n, dtype=t, device="cuda") - 0.5 for _ in range(4))
    g = dict(grad_a=True, grad_b=True, grad_c=True) if grads else {}
    api.adjoint_strided_batch(a, 2 + a.abs() + c.abs(), c, x if grads else None, w, solvedim=sd,
                              dims=dims, sync=True, **g)
    return api.last_config()


@pytest.mark.parametrize("dims,seg", [([32, 128, 400], 128), ([96, 200, 200], 128),
                                      ([64, 128, 400], 256), ([288, 128, 100], 256)])
def test_adjoint_rows_of_lines_that_end_in_half_a_segment(dims, seg):
    """The FP32 adjoint's 256-byte rows: not where they leave half of a group empty."""
    cfg = _adjoint_config(dims, 1, np.float32, True)
    assert cfg[0] == 4 and cfg[3] * 4 == seg, cfg


@pytest.mark.parametrize("N,systems,dtype,grads,M", [
    (16, 70000, np.float32, True, 1), (12, 65536, np.float32, True, 1),
    (12, 16384, np.float32, True, 4), (80, 32768, np.float32, True, 2),
    (80, 8192, np.float32, True, 4), (64, 1024, np.float32, True, 1),
    (64, 8192, np.float32, True, 4), (8, 512, np.float32, False, 1),
    (16, 512, np.float32, False, 4), (16, 65536, np.float64, True, 1),
    (16, 16384, np.float64, True, 2), (16, 65536, np.float64, False, 2)])
def test_adjoint_of_short_contiguous_systems(N, systems, dtype, grads, M):
    """Rows per lane of short contiguous systems, on both sides of the rule's lines."""
    cfg = _adjoint_config([N, systems], 0, dtype, grads)
    assert cfg[:2] == (4, M), cfg


def test_adjoint_of_a_few_longer_contiguous_systems():
    assert _adjoint_config([1000, 256], 0, np.float64, True) == (4, 8, 125, 1, 1)
    assert _adjoint_config([1000, 257], 0, np.float64, True)[3] == 2


@pytest.mark.parametrize("dims,dtype,grads,plain", [
    ([16, 16, 384], np.float64, True, True), ([16, 40, 384], np.float64, False, True),
    ([16, 40, 513], np.float64, False, False), ([22, 31, 110], np.float64, True, True),
    ([16, 600, 96], np.float64, True, True), ([16, 600, 97], np.float64, True, False),
    ([32, 46, 500], np.float32, True, True), ([32, 900, 61], np.float32, True, False),
    ([32, 900, 60], np.float32, True, True)])
def test_adjoint_of_few_systems(dims, dtype, grads, plain):
    """Few strided systems take the kernel without staging, at its fewer rows per lane
    or narrower rows; more take the wide one (16 or 32 rows, 128 bytes or more)."""
    cfg = _adjoint_config(dims, 1, dtype, grads)
    wide = cfg[1] in (16, 32) and cfg[3] * np.dtype(dtype).itemsize >= 128
    assert cfg[0] == 4 and wide != plain, cfg


@pytest.mark.parametrize("dims,dtype,grads,plain", [
    # lines of at most half a 128-byte segment
    ([8, 1000, 512], np.float64, False, True), ([9, 600, 129], np.float64, False, False),
    ([16, 300, 1024], np.float32, True, True), ([8, 621, 309], np.float32, False, True),
    ([8, 621, 321], np.float32, True, False), ([17, 300, 129], np.float32, True, False),
    # whole waves: aligned and misaligned lines
    ([16, 128, 40], np.float64, False, False), ([33, 128, 80], np.float64, False, True),
    ([33, 128, 101], np.float64, True, False), ([16, 128, 512], np.float64, True, True),
    # one long misaligned line
    ([28001, 256], np.float64, True, True), ([28000, 256], np.float64, True, False),
    ([28001, 256], np.float64, False, False)])
def test_adjoint_kernel_by_the_shape_of_the_lines(dims, dtype, grads, plain):
    """The wide kernel runs 16 rows per lane on 128 bytes or more (32 in FP32)."""
    cfg = _adjoint_config(dims, 1, dtype, grads)
    wide = cfg[1] in (16, 32) and cfg[3] * np.dtype(dtype).itemsize >= 128
    assert cfg[0] == 4 and wide != plain, cfg


@pytest.mark.parametrize("dims,W,G", [
    ([64, 256, 80], 32, 8), ([64, 256, 79], 16, 8), ([48, 256, 200], 16, 8),
    ([64, 192, 300], 32, 1), ([66, 192, 300], 32, 8), ([64, 513, 80], 16, 8)])
def test_adjoint_rows_and_order(dims, W, G):
    """FP64 adjoint on strided systems: 256-byte rows from 160 workgroups, plain order for
    short systems on aligned lines, and the results at the bar above."""
    assert _adjoint_config(dims, 1, np.float64, True)[3:] == (W, G)
    rng = np.random.default_rng(sum(dims))
    n = int(np.prod(dims))
    a, b, c, x = H.diag_dominant(rng, n, np.float64)
    w = rng.standard_normal(n)
    ref = oracle.adjoint(a, b, c, x, w, ndim=3, solvedim=1, dims=dims)
    out = api.adjoint_strided_batch(*(dev(v) for v in (a, b, c, x, w)), solvedim=1, dims=dims,
                                    grad_a=True, grad_b=True, grad_c=True, sync=True)
    for got, want in zip(out, ref):
        assert H.norm_rel_err(got.cpu().numpy(), want) <= 1e-12


@pytest.mark.parametrize("N,pad,systems,dtype,M", [
    (8, 0, 90000, np.float64, 2), (8, 2, 90000, np.float64, 1), (12, 2, 33333, np.float64, 1),
    (12, 2, 29999, np.float64, 2), (40, 1, 70000, np.float64, 1), (40, 1, 60000, np.float64, 2),
    (12, 0, 16499, np.float32, 4), (12, 2, 16500, np.float32, 1), (64, 1, 40000, np.float32, 1),
    (64, 1, 30000, np.float32, 2), (64, 4, 40000, np.float32, 4)])
def test_adjoint_of_contiguous_systems_apart(N, pad, systems, dtype, M):
    """Rows per lane of short contiguous systems on rows apart from each other, against the
    oracle on a sample of the systems."""
    rng = np.random.default_rng(N + systems)
    n = (N + pad) * systems
    a, b, c, x = H.diag_dominant(rng, n, dtype)
    w = rng.standard_normal(n).astype(dtype)
    out = api.adjoint_strided_batch(*(dev(v) for v in (a, b, c, x, w)), solvedim=0,
                                    dims=[N, systems], pads=[N + pad, systems], grad_a=True,
                                    grad_b=True, grad_c=True, sync=True)
    assert api.last_config()[:2] == (4, M), api.last_config()
    out = [t.cpu().numpy() for t in out]
    for s in list(range(0, systems, 4999)) + [systems - 1]:
        i = slice(s * (N + pad), s * (N + pad) + N)
        ref = oracle.adjoint(*(v[i].astype(np.float64) for v in (a, b, c, x, w)), ndim=1,
                             solvedim=0, dims=[N])
        for got, want in zip(out, ref):
            assert H.norm_rel_err(got[i], want) <= (1e-12 if dtype == np.float64 else 1e-5), s


def test_adjoint_of_contiguous_planes_apart():
    """Gaps between planes count as gaps between rows do."""
    for dims, pads, M in (([16, 40, 1000], [16, 42, 1000], 1), ([16, 40, 1000], None, 2)):
        n = int(np.prod(pads or dims))
        a, c, x, w = (torch.rand(n, dtype=torch.float64, device="cuda") - 0.5 for _ in range(4))
        api.adjoint_strided_batch(a, 2 + a.abs() + c.abs(), c, x, w, solvedim=0, dims=dims,
                                  pads=pads or dims, grad_a=True, grad_b=True, grad_c=True,
                                  sync=True)
        assert api.last_config()[:2] == (4, M), (api.last_config(), pads)
