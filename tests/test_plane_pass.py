"""The plane pass (first two dims of a 3D plan in one launch) against the FP64
oracle and, in all four directions, against the plan of three single passes,
where it can go wrong: one-stage lines, planes with fewer lines than a
workgroup has wavefronts, odd and even extents in both dims, r2c / c2r of even and odd
length, BFFT chains, prime radices, both memory orders, extra dims.  On the CPU
through the host emulator, which runs the kernel's own phase functions; on the
device as planned.  Tolerances (relative L2): Float64 1e-13, Float32
5e-7 log2 N."""
import numpy as np
import pytest

from oracle import pipeline as OP
from tests.cases import CODE_NAMES, NP_DTYPES, meta_for, random_logical, tol_for

torch = pytest.importorskip("torch")

FUSED = 1 << 31   # emulator plans: first two dims fused
SIZES = [(2, 2, 2), (4, 2, 3), (3, 4, 2), (7, 13, 3), (14, 11, 2), (16, 12, 6), (15, 16, 5),
         (32, 20, 3), (36, 49, 2), (64, 64, 2), (63, 36, 2), (26, 81, 2), (78, 35, 2)]
SIZES += [(32, 33, 3), (36, 49, 18), (63, 36, 24), (26, 81, 22), (78, 35, 28)]   # the rule's two halves
KINDS = ["RFFT", "FFT", "BFFT"]


def fused(dims, kind):
    """x lines have a transform of two points or more; planes small, or many."""
    return not (kind == "RFFT" and dims[0] == 2) and (
        dims[0] * dims[1] <= 1088 or dims[2] * 100 >= dims[0] * dims[1])


@pytest.mark.parametrize("permute,extra", [(True, ()), (False, (2,))], ids=["perm", "noperm-extra"])
@pytest.mark.parametrize("real_type", [1, 0], ids=["F64", "F32"])
@pytest.mark.parametrize("dims", SIZES, ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("kind", KINDS)
def test_plane_pass_emulated(pf, emu, kind, dims, real_type, permute, extra):
    T = pf.Transforms
    tol = tol_for(CODE_NAMES[real_type], dims)
    meta, full = meta_for(T, dims, (getattr(T, kind)(),), CODE_NAMES[real_type], permute, extra)
    kinds = [t.code for t in full]
    dt_in, dt_out = NP_DTYPES[meta.eltype_in], NP_DTYPES[meta.eltype_out]
    rng = np.random.default_rng(0)
    x = random_logical(rng, tuple(dims) + extra, meta.eltype_in)
    xin = OP.memory_image(OP.to_memory(x, meta.perm_in)).astype(dt_in)
    wide = xin.astype(np.complex128 if np.iscomplexobj(xin) else np.float64)
    ref = OP.memory_image(OP.forward(meta, OP.from_image(wide, meta.mem_dims("in"))))
    y = random_logical(rng, ref.shape, meta.eltype_out).astype(dt_out)   # no symmetry
    if fused(dims, kind):
        assert emu.passes(dims, kinds, real_type, permute, extra, FUSED) == 2

    def both(direction, v):
        return [emu.run(dims, kinds, real_type, direction, v, permute, extra, flags=f)
                .view(dt_out if direction in (0, 4) else dt_in) for f in (FUSED, 0)]

    out, single = both(0, xin)
    assert OP.rel_l2(out, ref) <= tol
    back, _ = both(2, out)
    assert OP.rel_l2(back, wide) <= tol
    for direction, v in ((1, y), (2, y), (3, y), (4, xin)):
        got, want = both(direction, v)
        assert OP.rel_l2(got, want) <= tol, direction


def test_plane_pass_rule(pf, emu):
    """What keeps the single passes: other ranks, R2R and no transform in the
    first two dims, prime factors past 13, planes larger than the LDS, in place."""
    T = pf.Transforms
    for rt in (0, 1):
        for dims, trs, n in (((8, 9, 10), (T.FFT(),), 2),
                             ((8, 9, 10), (T.BRFFT(True),), 2),
                             ((8, 9, 10, 4), (T.FFT(),), 4),
                             ((8, 9, 10), (T.FFT(), T.FFT(), T.NoTransform()), 2),
                             ((8, 9, 10), (T.NoTransform(), T.FFT(), T.FFT()), 3),
                             ((8, 9, 10), (T.FFT(), T.NoTransform(), T.FFT()), 3),
                             ((17, 9, 10), (T.FFT(),), 3),
                             ((8, 19, 10), (T.FFT(),), 3),
                             ((8, 1, 10), (T.FFT(),), 3),
                             ((256, 256, 2), (T.FFT(),), 3),
                             ((8, 9, 10), (T.R2R(T.REDFT10), T.FFT(), T.FFT()), 3),
                             ((8, 9, 10), (T.FFT_(),), 3)):
            _, full = meta_for(T, dims, trs, CODE_NAMES[rt])
            got = emu.passes(dims, [t.code for t in full], rt, True, (), FUSED)
            assert got == n, (dims, trs, got)


@pytest.mark.gpu
@pytest.mark.parametrize("permute,extra", [(True, ()), (False, (2,))], ids=["perm", "noperm-extra"])
@pytest.mark.parametrize("real_type", [1, 0], ids=["F64", "F32"])
@pytest.mark.parametrize("dims", SIZES, ids=lambda d: "x".join(map(str, d)))
def test_plane_pass_device(pf, gpu, dims, real_type, permute, extra):
    from tests.test_gpu_parity import run_case
    T = pf.Transforms
    tol = tol_for(CODE_NAMES[real_type], dims)
    for kind in KINDS:
        err_f, err_b, meta = run_case(pf, dims, (getattr(T, kind)(),), real_type, permute, extra)
        if fused(dims, kind):
            assert meta.kernels[0].startswith("k_plane"), (kind, meta.kernels)
            assert meta.kernels[3].startswith("k_plane"), (kind, meta.kernels)
        assert err_f <= tol and err_b <= tol, (kind, err_f, err_b, tol)
