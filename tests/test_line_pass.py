"""The line pass against the FP64 oracle, where it can go wrong: every radix by
itself (lines of 2 to 16 points, one stage, no LDS), two and three stages, odd
r2c / c2r, tiles with fewer lines than they hold, both memory orders, extra
dims, long lines with one or two lines to a tile, prime factors of 17 to 61 (one,
two, a square), Bluestein lengths.  On the CPU through the host emulator, which runs the
kernel's own phase functions; on the device with the specialised kernels off,
so that every pass takes the line pass.  Tolerances (relative L2): Float64
1e-13, Float32 5e-7 log2 N."""
import pytest

from tests.cases import CODE_NAMES, tol_for
from tests.test_emulated import R2R_KINDS, emu_case

torch = pytest.importorskip("torch")

# first dim: the line length of interest; the others give partial tiles
SIZES = [(n, 5, 3) for n in range(2, 17)]            # one stage
SIZES += [(n, 37, 2) for n in (26, 33, 45, 98, 121, 143, 144, 169, 196, 225, 256)]   # two
SIZES += [(n, 19) for n in (315, 448, 1001, 2025, 4096)]   # three, and 4-stage 2 n of R2R
SIZES += [(3, 2, 130), (2, 70, 9)]                   # short lines, many of them
SIZES += [(n, 37, 2) for n in (17, 31, 34, 59, 61, 122, 289, 323)]   # primes 17 to 61
SIZES += [(n, 5, 3) for n in (67, 134, 257)] + [(1031, 3)]    # Bluestein


def cases_of(T, dims):
    yield "RFFT", (T.RFFT(),)
    yield "FFT", (T.FFT(),)
    if dims[0] <= 323:
        for k in R2R_KINDS:
            yield k, (T.R2R(getattr(T, k)),)


@pytest.mark.parametrize("permute,extra", [(True, ()), (False, (2,))], ids=["perm", "noperm-extra"])
@pytest.mark.parametrize("real_type", [1, 0], ids=["F64", "F32"])
@pytest.mark.parametrize("dims", SIZES, ids=lambda d: "x".join(map(str, d)))
def test_line_pass_emulated(pf, emu, dims, real_type, permute, extra):
    T = pf.Transforms
    tol = tol_for(CODE_NAMES[real_type], dims)
    for name, trs in cases_of(T, dims):
        err_f, err_b = emu_case(pf, emu, dims, trs, real_type, permute=permute, extra=extra)
        assert err_f <= tol and err_b <= tol, (name, err_f, err_b, tol)


@pytest.mark.gpu
@pytest.mark.parametrize("permute,extra", [(True, ()), (False, (2,))], ids=["perm", "noperm-extra"])
@pytest.mark.parametrize("real_type", [1, 0], ids=["F64", "F32"])
@pytest.mark.parametrize("dims", SIZES, ids=lambda d: "x".join(map(str, d)))
def test_line_pass_device(pf, gpu, dims, real_type, permute, extra):
    from tests.test_gpu_parity import run_case
    T = pf.Transforms
    tol = tol_for(CODE_NAMES[real_type], dims)
    for name, trs in cases_of(T, dims):
        err_f, err_b, meta = run_case(pf, dims, trs, real_type, permute, extra,
                                      flags=pf._lib.FLAG_GENERIC_ONLY)
        if name == "FFT" or (name == "RFFT" and dims[0] > 2):
            assert meta.kernels[0].startswith("k_line"), (name, meta.kernels)
        assert err_f <= tol and err_b <= tol, (name, err_f, err_b, tol)


@pytest.mark.parametrize("dims", [(6, 9, 10), (9, 7, 8), (10, 9, 7), (7, 6, 9), (6, 5, 7, 8)],
                         ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("kind", ["RFFT", "FFT"])
def test_intermediate_orders(pf, emu, dims, kind):
    """Odd and even extents in every place: the order of each intermediate is
    chosen by them, and no choice may change the result."""
    T = pf.Transforms
    for rt in (1, 0):
        tol = tol_for(CODE_NAMES[rt], dims)
        err_f, err_b = emu_case(pf, emu, dims, (getattr(T, kind)(),), rt)
        assert err_f <= tol and err_b <= tol, (err_f, err_b)
