"""C ABI of libdiagpu.so on the CPU: every symbol include/diagpu.h declares is
exported, and argument errors come back as status codes before any HIP call
(none of these calls reaches the GPU)."""
import ctypes as C
import re
from pathlib import Path

import pytest

from diagpu_amd import _lib

ROOT = Path(__file__).resolve().parents[1]


def declared_symbols():
    text = (ROOT / "include" / "diagpu.h").read_text()
    return sorted(set(re.findall(r"DIAGPU_API\s+[\w\s\*]+?\b(diagpu_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    names = declared_symbols()
    assert len(names) >= 8
    for name in names:
        assert hasattr(lib, name), name
        assert name in _lib.PROTOTYPES, f"{name} has no ctypes prototype"
    assert set(_lib.PROTOTYPES) == set(names)


def test_status_names():
    lib = _lib.load()
    assert lib.diagpu_abi_version() >= 100
    for code, name in [(0, b"DIAGPU_OK"), (1, b"DIAGPU_ERR_ARG"), (5, b"DIAGPU_ERR_CAPACITY")]:
        assert lib.diagpu_status_name(code) == name


def _status(name, *args):
    return getattr(_lib.load(), name)(*args)


def test_spmv_argument_errors():
    V = _lib.ReconViewF32
    fake = C.c_void_p(0x1000)   # never dereferenced: validation fails first
    assert _status("diagpu_spmv_recon_f32", None, fake, 4, fake, None) == _lib.ERR_ARG
    assert b"R is NULL" in _lib.load().diagpu_last_error()
    v = V(-1, 4, 1, fake.value, fake.value)
    assert _status("diagpu_spmv_recon_f32", C.byref(v), fake, 4, fake, None) == _lib.ERR_ARG
    v = V(4, 4, 1, None, fake.value)
    assert _status("diagpu_spmv_recon_f32", C.byref(v), fake, 4, fake, None) == _lib.ERR_ARG
    v = V(4, 4, 1, fake.value, None)
    assert _status("diagpu_spmv_recon_f32", C.byref(v), fake, 4, fake, None) == _lib.ERR_ARG
    v = V(4, 4, 1, fake.value, fake.value)
    assert _status("diagpu_spmv_recon_f32", C.byref(v), None, 4, fake, None) == _lib.ERR_ARG
    assert _status("diagpu_spmv_recon_f32", C.byref(v), fake, 4, None, None) == _lib.ERR_ARG
    assert _status("diagpu_spmv_recon_f32", C.byref(v), fake, -1, fake, None) == _lib.ERR_ARG
    # rows == 0 is a successful no-op (tc_spmv_regdirect_kernel.cu:143)
    v = V(0, 4, 1, None, None)
    assert _status("diagpu_spmv_recon_f32", C.byref(v), None, 0, None, None) == _lib.OK
    w = _lib.ReconViewF64(0, 0, 0, None, None)
    assert _status("diagpu_spmv_recon_f64", C.byref(w), None, 0, None, None) == _lib.OK


def test_python_wrapper_rejects_bad_tensors():
    import torch
    from diagpu_amd.spmv import recon_view
    with pytest.raises(TypeError):
        recon_view(torch.zeros(2, dtype=torch.int32), torch.zeros(8), 4, 4)


def test_spgemm_argument_errors():
    lib = _lib.load()
    sz = C.c_size_t(0)
    assert lib.diagpu_spgemm_symbolic_workspace(0, 1, 1, C.byref(sz)) == _lib.ERR_ARG
    assert lib.diagpu_spgemm_symbolic_workspace(100, -1, 1, C.byref(sz)) == _lib.ERR_ARG
    assert lib.diagpu_spgemm_symbolic_workspace(100, 3, 4, None) == _lib.ERR_ARG
    assert lib.diagpu_spgemm_symbolic_workspace(1 << 20, 9, 7, C.byref(sz)) == _lib.OK
    # A lookup of 2n-1 int32 plus two bitmaps and a word prefix dominate
    assert sz.value >= 4 * (2 * (1 << 20) - 1) + 3 * 4 * ((2 * (1 << 20)) // 32)
    fake = C.c_void_p(0x1000)
    info = _lib.SpgemmInfo()
    args = [100, fake, fake, fake, 3, fake, fake, fake, 2, fake, fake, fake, 6, fake, fake, 6,
            None, fake, 1 << 20, C.byref(info), None]
    bad = list(args); bad[19] = None
    assert lib.diagpu_spgemm_symbolic(*bad) == _lib.ERR_ARG
    bad = list(args); bad[0] = 0
    assert lib.diagpu_spgemm_symbolic(*bad) == _lib.ERR_ARG
    bad = list(args); bad[1] = None
    assert lib.diagpu_spgemm_symbolic(*bad) == _lib.ERR_ARG
    bad = list(args); bad[13] = None
    assert lib.diagpu_spgemm_symbolic(*bad) == _lib.ERR_ARG
    bad = list(args); bad[18] = 16
    assert lib.diagpu_spgemm_symbolic(*bad) == _lib.ERR_CAPACITY
    assert b"workspace" in lib.diagpu_last_error()
    # the same call with the A-stationary records: both records pointers are
    # required, and the symbolic checks come before any HIP call
    rstat = C.c_int32(-1)
    fused = args[:19] + [fake, C.byref(rstat)] + args[19:]
    bad = list(fused); bad[19] = None
    assert lib.diagpu_spgemm_symbolic_astat(*bad) == _lib.ERR_ARG
    assert b"records" in lib.diagpu_last_error()
    bad = list(fused); bad[20] = None
    assert lib.diagpu_spgemm_symbolic_astat(*bad) == _lib.ERR_ARG
    assert b"records_status" in lib.diagpu_last_error()
    bad = list(fused); bad[18] = 16
    assert lib.diagpu_spgemm_symbolic_astat(*bad) == _lib.ERR_CAPACITY
    assert rstat.value == -1                  # untouched when the symbolic phase fails
    # numeric
    assert lib.diagpu_spgemm_numeric_f32(0, fake, fake, fake, fake, fake, 1, fake, fake, 1,
                                         fake, None) == _lib.ERR_ARG
    assert lib.diagpu_spgemm_numeric_f32(10, fake, fake, fake, fake, fake, 0, fake, fake, 0,
                                         fake, None) == _lib.OK      # no C diagonals: no-op
    assert lib.diagpu_spgemm_numeric_f32(10, fake, fake, None, fake, fake, 3, fake, fake, 1,
                                         fake, None) == _lib.ERR_ARG
    assert lib.diagpu_spgemm_numeric_f32(10, fake, fake, fake, fake, fake, 50, fake, fake, 1,
                                         fake, None) == _lib.ERR_ARG  # > 2n - 1 diagonals
    assert lib.diagpu_rowpacked_as_hm(0, fake, 1, fake, fake, None) == _lib.ERR_ARG
    assert lib.diagpu_rowpacked_as_hm(10, None, 1, fake, fake, None) == _lib.ERR_ARG
    assert lib.diagpu_rowpacked_as_hm(10, None, 0, None, None, None) == _lib.OK


def test_axpby_argument_errors():
    lib = _lib.load()
    fake = C.c_void_p(0x1000)
    args = [100, fake, fake, 2, fake, 1.0, fake, fake, 2, fake, 1.0, fake, fake, 3, fake, None]
    bad = list(args); bad[0] = 0
    assert lib.diagpu_dia_axpby_f32(*bad) == _lib.ERR_ARG
    bad = list(args); bad[13] = -1
    assert lib.diagpu_dia_axpby_f32(*bad) == _lib.ERR_ARG
    bad = list(args); bad[14] = None
    assert lib.diagpu_dia_axpby_f32(*bad) == _lib.ERR_ARG
    bad = list(args); bad[1] = None
    assert lib.diagpu_dia_axpby_f32(*bad) == _lib.ERR_ARG
    assert b"X arrays" in lib.diagpu_last_error()
    bad = list(args); bad[13] = 0
    assert lib.diagpu_dia_axpby_f32(*bad) == _lib.OK          # empty Z: no-op


def test_complex_and_krylov_argument_errors():
    fake = C.c_void_p(0x1000)   # never dereferenced: validation fails first
    V = _lib.ReconViewC64
    v = V(4, 4, 1, fake.value, fake.value)
    assert _status("diagpu_spmv_recon_c64", None, fake, 4, fake, None) == _lib.ERR_ARG
    assert _status("diagpu_spmv_recon_c64", C.byref(v), None, 4, fake, None) == _lib.ERR_ARG
    w = _lib.ReconViewF32(4, 4, 1, fake.value, fake.value)
    assert _status("diagpu_spmv_recon_f32_c64", C.byref(w), fake, 4, None, None) == _lib.ERR_ARG
    z = V(0, 0, 0, None, None)
    assert _status("diagpu_spmv_recon_c64", C.byref(z), None, 0, None, None) == _lib.OK

    b = C.c_size_t(0)
    assert _status("diagpu_expm_krylov_workspace", 100, 0, C.byref(b)) == _lib.ERR_ARG
    assert _status("diagpu_expm_krylov_workspace", 100, 65, C.byref(b)) == _lib.ERR_ARG
    assert _status("diagpu_expm_krylov_workspace", 0, 10, C.byref(b)) == _lib.ERR_ARG
    assert _status("diagpu_expm_krylov_workspace", 1000, 10, C.byref(b)) == _lib.OK
    assert b.value >= 10 * 1000 * 8
    info = _lib.KrylovInfo()
    sq = V(1000, 1000, 1, fake.value, fake.value)
    rect = V(1000, 999, 1, fake.value, fake.value)
    call = lambda view, m, ws_bytes, t=1.0: _status(
        "diagpu_expm_krylov_c64", C.byref(view), fake, t, m, fake, fake, ws_bytes, None, None,
        None, C.byref(info), None)
    assert call(rect, 10, b.value) == _lib.ERR_ARG                 # not square
    assert call(sq, 0, b.value) == _lib.ERR_ARG                    # m out of range
    assert call(sq, 10, b.value, float("nan")) == _lib.ERR_ARG     # t not finite
    assert call(sq, 10, b.value - 1) == _lib.ERR_CAPACITY          # workspace too small
    assert b"workspace" in _lib.load().diagpu_last_error()
    assert _status("diagpu_expm_krylov_f32", None, fake, 1.0, 10, fake, fake, b.value, None,
                   None, None, C.byref(info), None) == _lib.ERR_ARG
    assert _status("diagpu_promote_f32_c64", -1, fake, fake, None) == _lib.ERR_ARG
    assert _status("diagpu_promote_f32_c64", 5, None, fake, None) == _lib.ERR_ARG
    assert _status("diagpu_promote_f32_c64", 0, None, None, None) == _lib.OK
    band = _lib.BandInfo()
    assert _status("diagpu_spgemm_band_prepare", 0, fake, fake, 1, fake, fake, 1, fake, 1, fake,
                   C.byref(band), None) == _lib.ERR_ARG
    assert _status("diagpu_spgemm_band_prepare", 100, fake, fake, 70000, fake, fake, 1, fake, 1,
                   fake, C.byref(band), None) == _lib.ERR_ARG
    assert _status("diagpu_spgemm_band_prepare", 100, None, fake, 1, fake, fake, 1, fake, 1, fake,
                   C.byref(band), None) == _lib.ERR_ARG
    assert _status("diagpu_spgemm_band_prepare", 100, fake, fake, 1, None, fake, 1, fake, 1, fake,
                   C.byref(band), None) == _lib.ERR_ARG
    # numeric_band needs an eligible, consistent info (validated before any launch)
    band = _lib.BandInfo(0, 4, 256, 1, 4 * (3 * 256 + 2 * 260) + 16 * 7, 7)
    call = lambda nA, info: _status("diagpu_spgemm_numeric_band_f32", 100, fake, fake, nA, fake,
                                    fake, fake, 2, fake, fake, fake, 5, fake, fake, C.byref(info),
                                    fake, None)
    assert call(4, band) == _lib.ERR_CAPACITY    # lds_bytes does not match nA
    band.eligible = 0
    assert call(3, band) == _lib.ERR_CAPACITY
    # A-stationary kernel: argument checks before any HIP call or launch
    prep = lambda n, aoff, nA, nB, cptr, nC, npairs: _status(
        "diagpu_spgemm_astat_prepare", n, aoff, fake, nA, fake, fake, nB, fake, cptr, nC, fake,
        npairs, fake, None)
    assert prep(0, fake, 1, 1, fake, 1, 1) == _lib.ERR_ARG        # n < 1
    assert prep(10, fake, 0, 1, fake, 1, 1) == _lib.ERR_ARG       # no A diagonal
    assert prep(10, fake, 1, 0, fake, 1, 1) == _lib.ERR_ARG       # no B diagonal
    assert prep(10, None, 1, 1, fake, 1, 1) == _lib.ERR_ARG       # A offsets NULL
    assert prep(10, fake, 1, 1, None, 1, 1) == _lib.ERR_ARG       # pair_ptr NULL
    assert prep(10, fake, 1, 1, fake, 1, -1) == _lib.ERR_ARG      # negative entry count
    assert prep(10, fake, 1, 1, fake, 20, 1) == _lib.ERR_ARG      # c_ndiag > 2n - 1
    assert prep(10, fake, 1, 1, fake, 0, 1) == _lib.ERR_ARG       # entries without C
    astat = lambda nA, nC, n=100, npairs=1: _status("diagpu_spgemm_numeric_astat_f32", n, fake,
                                                    fake, nA, fake, fake, fake, fake, fake, nC,
                                                    fake, fake, npairs, fake, None)
    assert astat(0, 5) == _lib.ERR_ARG
    assert astat(3, 5, 1 << 30) == _lib.ERR_ARG     # n < 2^30 (C stores' 32-bit byte range)
    # the kernel reads metadata and records at 32-bit byte offsets
    assert astat(3, 1 << 29, 1 << 29) == _lib.ERR_ARG          # c_ndiag < 2^29
    assert astat(3, 5, 100, 1 << 28) == _lib.ERR_ARG           # n_pairs < 2^28
    assert astat(_lib.ASTAT_MAX_A + 1, 5) == _lib.ERR_CAPACITY
    assert astat(3, 200) == _lib.ERR_ARG           # c_ndiag > 2n - 1
    assert astat(3, 0) == _lib.OK                   # empty C: nothing to do
    astat_c = lambda nA, nC, n=100, npairs=1: _status("diagpu_spgemm_numeric_astat_c64", n, fake,
                                                      fake, nA, fake, fake, fake, fake, fake, nC,
                                                      fake, fake, npairs, fake, None)
    assert astat_c(0, 5) == _lib.ERR_ARG
    assert astat_c(3, 5, 1 << 30) == _lib.ERR_ARG
    assert astat_c(3, 1 << 29, 1 << 29) == _lib.ERR_ARG
    assert astat_c(3, 5, 100, 1 << 28) == _lib.ERR_ARG
    assert astat_c(_lib.ASTAT_MAX_A_C64 + 1, 5) == _lib.ERR_CAPACITY
    assert astat_c(3, 200) == _lib.ERR_ARG
    assert astat_c(3, 0) == _lib.OK
    # the fused (alpha A) B + sigma I entry points: the same checks, the same limits
    one = _lib.Complex64(1.0, 0.0)
    for name, a, s, cap in (("diagpu_spgemm_numeric_astat_scaled_f32", 2.0, 1.0, _lib.ASTAT_MAX_A),
                            ("diagpu_spgemm_numeric_astat_scaled_c64", one, one,
                             _lib.ASTAT_MAX_A_C64)):
        sc = lambda nA, nC, n=100, npairs=1: _status(name, n, fake, fake, nA, fake, a, fake,
                                                     fake, fake, fake, nC, fake, fake, npairs, s,
                                                     fake, None)
        assert sc(0, 5) == _lib.ERR_ARG
        assert sc(3, 5, 1 << 30) == _lib.ERR_ARG
        assert sc(3, 1 << 29, 1 << 29) == _lib.ERR_ARG
        assert sc(3, 5, 100, 1 << 28) == _lib.ERR_ARG
        assert sc(cap + 1, 5) == _lib.ERR_CAPACITY
        assert sc(3, 200) == _lib.ERR_ARG
        assert sc(3, 0) == _lib.OK
        bad = [100, fake, fake, 3, None, a, fake, fake, fake, fake, 5, fake, fake, 1, s, fake, None]
        assert _status(name, *bad) == _lib.ERR_ARG                # A values NULL


def test_astat_max_a_matches_header():
    """The Python constants mirror DIAGPU_ASTAT_MAX_A and _C64, and the
    staged rows of that many A diagonals (288 fp32; 144 complex64, the
    128-row blocks taken above 75 complex A diagonals) fit a workgroup's
    160 KiB of LDS, one more does not."""
    import re
    hdr = (Path(__file__).resolve().parents[1] / "include" / "diagpu.h").read_text()
    m = re.search(r"#define DIAGPU_ASTAT_MAX_A (\d+)", hdr)
    assert m and int(m.group(1)) == _lib.ASTAT_MAX_A
    assert 288 * _lib.ASTAT_MAX_A * 4 <= 160 * 1024 < 288 * (_lib.ASTAT_MAX_A + 1) * 4
    m = re.search(r"#define DIAGPU_ASTAT_MAX_A_C64 (\d+)", hdr)
    assert m and int(m.group(1)) == _lib.ASTAT_MAX_A_C64
    assert 144 * _lib.ASTAT_MAX_A_C64 * 8 <= 160 * 1024 < 144 * (_lib.ASTAT_MAX_A_C64 + 1) * 8


def test_symbolic_noalloc_rejects_beyond_scratch():
    """diagpu_spgemm_symbolic_noalloc: a workspace larger than the library's
    scratch array is DIAGPU_ERR_CAPACITY, reported before any HIP call (the
    fake pointers are never read)."""
    lib = _lib.load()
    n = 1 << 23
    ws = C.c_size_t(0)
    assert lib.diagpu_spgemm_symbolic_workspace(n, 3, 3, C.byref(ws)) == _lib.OK
    assert ws.value > _lib.SYMBOLIC_SCRATCH_BYTES
    fake = C.c_void_p(0x1000)
    info = _lib.SpgemmInfo()
    st = lib.diagpu_spgemm_symbolic_noalloc(n, fake, fake, fake, 3, fake, fake, fake, 3, fake,
                                            fake, fake, 9, fake, fake, 9, None, C.byref(info),
                                            None)
    assert st == _lib.ERR_CAPACITY
    assert b"scratch" in lib.diagpu_last_error()
    assert lib.diagpu_spgemm_symbolic_noalloc(n, fake, fake, fake, 3, fake, fake, fake, 3, fake,
                                              fake, fake, 9, fake, fake, 9, None, None,
                                              None) == _lib.ERR_ARG


@pytest.mark.parametrize("n", [1, 511, 20000, 500000, 500001, 1 << 22])
def test_krylov_workspace_sizes(n):
    """The size that a caller may have kept: m basis vectors, a partial sum per
    512 rows for the dot and for the norm, T_m's entries; the one-kernel steps
    ask for more up to n = 500000, by their own query."""
    up = lambda b: -(-b // 256) * 256
    b, f = C.c_size_t(0), C.c_size_t(0)
    for m in (1, 30, 64):
        assert _status("diagpu_expm_krylov_workspace", n, m, C.byref(b)) == _lib.OK
        tiles = -(-n // 512)
        assert b.value == up(8 * m * n) + 2 * up(8 * tiles) + up(8 * (2 * m + 1))
        assert _status("diagpu_expm_krylov_workspace_fused", n, m, C.byref(f)) == _lib.OK
        assert f.value - b.value == (up(16 * n) + 32768 if n <= 500000 else 0)
    assert _status("diagpu_expm_krylov_workspace_fused", 0, 1, C.byref(f)) == _lib.ERR_ARG
    assert _status("diagpu_expm_krylov_workspace_fused", 1, 65, C.byref(f)) == _lib.ERR_ARG
    assert _status("diagpu_expm_krylov_workspace_fused", 1, 1, None) == _lib.ERR_ARG


def test_package_modules_import():
    """Every module of the package imports on a host without a GPU (the GPU
    tests would otherwise be the first to meet a broken module)."""
    import importlib

    import diagpu_amd
    names = [f.stem for f in Path(diagpu_amd.__file__).parent.glob("*.py") if f.stem != "__init__"]
    assert {"spgemm", "chain", "spmv", "krylov", "workloads", "_lib", "build"} <= set(names)
    for name in names:
        importlib.import_module(f"diagpu_amd.{name}")


def test_full_choice_is_host_logic():
    """The contiguous-band rule: only whole contiguous products, only operands
    that fit in LDS, from the stated number of entries per C diagonal."""
    fn = _lib.load().diagpu_spgemm_full_choice

    def take(n, a0, na, b0, nb, cplx=0, contiguous=1, nc=None, pairs=None):
        sh = _lib.SpgemmShape(a0, a0 + na - 1, b0, b0 + nb - 1, contiguous)
        return fn(n, na, nb, na + nb - 1 if nc is None else nc,
                  na * nb if pairs is None else pairs, C.byref(sh), cplx)

    assert take(100000, -16, 33, -16, 33) == 1
    assert take(100000, -16, 33, -16, 33, contiguous=0) == 0
    assert take(100000, -16, 33, -16, 33, nc=64) == 0
    assert take(100000, -16, 33, -16, 33, pairs=1088) == 0
    assert take(20, -10, 21, -10, 21) == 0            # sums reach beyond +-19
    assert take(21, -10, 21, -10, 21) == 1
    assert take(100000, -3, 7, -3, 7) == 0 and take(100000, -3, 7, -3, 7, cplx=1) == 1
    assert take(5000, -2, 5, -2, 5) == 1 and take(5000, -1, 3, -1, 3) == 0
    assert take(5000, -34, 69, -3, 7) == 1 and take(5000, -35, 70, -3, 7) == 0
    assert take(5000, -3, 7, -2000, 4000) == 0        # beyond LDS
    assert fn(100, 3, 3, 5, 9, None, 0) == 0


@pytest.mark.parametrize("n,na,nb,cplx,full", [
    # fp32 below 10000 rows: wide C of few entries stays with the general kernels
    (4200, 3, 49, 0, 0), (9999, 5, 37, 0, 0), (8000, 49, 5, 0, 0), (4200, 7, 5, 0, 0),
    (4200, 7, 37, 0, 0), (4200, 37, 7, 0, 1), (4200, 7, 7, 0, 1), (4200, 5, 29, 0, 1),
    (4095, 3, 49, 0, 1), (4200, 9, 37, 0, 1), (4096, 21, 21, 0, 1),
    # more than 64 C diagonals in more workgroups than CUs
    (8192, 17, 49, 0, 1), (8193, 17, 49, 0, 0), (14999, 21, 49, 0, 0), (15000, 21, 49, 0, 1),
    (12500, 33, 33, 0, 1), (9000, 17, 48, 0, 1), (17000, 17, 49, 0, 1),
    (94475, 21, 11, 0, 0), (100003, 15, 15, 0, 1),
    # complex: one C diagonal per wave of the A-stationary kernel, one round of blocks
    (32768, 7, 7, 1, 1), (32769, 7, 7, 1, 0), (65504, 9, 8, 1, 0), (65505, 9, 8, 1, 1),
    (50000, 9, 9, 1, 1)])
def test_full_choice_where_the_general_kernels_are_faster(n, na, nb, cplx, full):
    """The measured lines of the automatic choice, on both sides."""
    a0, b0 = -(na // 2), -(nb // 2)
    sh = _lib.SpgemmShape(a0, a0 + na - 1, b0, b0 + nb - 1, 1)
    assert _lib.load().diagpu_spgemm_full_choice(n, na, nb, na + nb - 1, na * nb, C.byref(sh),
                                                 cplx) == full


def test_full_argument_errors():
    f = C.c_void_p(0x1000)   # never dereferenced: validation fails first
    name = "diagpu_spgemm_numeric_full_f32"
    ok = (100, -1, 3, f, f, -1, 3, f, f, f, 5, f, None)
    for at, bad in ((0, 0), (2, 0), (3, None), (4, None), (6, 0), (8, None), (9, None), (10, 4),
                    (11, None), (1, -100), (5, 98)):
        args = list(ok)
        args[at] = bad
        assert _status(name, *args) == _lib.ERR_ARG, at
    assert _status(name, 10000, -100, 201, f, f, -1, 3, f, f, f, 203, f, None) == _lib.ERR_CAPACITY
    assert _status("diagpu_spgemm_symbolic_shape", 4, f, f, f, 1, f, f, f, 1, f, f, f, 1, f, f, 1,
                   None, f, 1 << 20, None, None, None, C.byref(_lib.SpgemmInfo()), None) == _lib.ERR_ARG


def test_chain_plans_argument_errors():
    name = "diagpu_chain_plans"
    off = (C.c_int32 * 3)(-1, 0, 1)
    bad = (C.c_int32 * 3)(-1, 1, 0)
    need, info = C.c_size_t(0), (_lib.ChainStep * 2)()
    buf = C.create_string_buffer(1 << 16)
    ok = (100, 3, off, 3, off, 2, buf, len(buf), C.byref(need), info)
    assert _status(name, *ok) == _lib.OK and need.value > 0
    for at, v, code in ((0, 0, _lib.ERR_ARG), (1, 0, _lib.ERR_ARG), (2, None, _lib.ERR_ARG),
                        (2, bad, _lib.ERR_OFFSET), (4, bad, _lib.ERR_OFFSET), (5, 0, _lib.ERR_ARG),
                        (6, None, _lib.ERR_ARG), (8, None, _lib.ERR_ARG), (9, None, _lib.ERR_ARG),
                        (0, 1, _lib.ERR_OFFSET)):
        args = list(ok)
        args[at] = v
        assert _status(name, *args) == code, (at, v)
    assert _status(name, 100, 3, off, 3, off, 2, None, 0, C.byref(need), info) == _lib.ERR_CAPACITY
    assert _status(name, 100, 3, off, 3, off, 2, buf, need.value, C.byref(need), info) == _lib.OK
    assert _status(name, 100, 3, off, 3, off, 2, buf, need.value - 1, C.byref(need),
                   info) == _lib.ERR_CAPACITY
    long = (C.c_int32 * 200)(*range(-100, 100))
    big = (_lib.ChainStep * 1)()
    assert _status(name, 9000, 200, long, 200, long, 1, None, 0, C.byref(need),
                   big) == _lib.ERR_OVERFLOW


@pytest.mark.parametrize("n,h,s,steps", [
    (10, [0], [0], 3), (10, [-9, 9], [-9, 9], 2), (50, [-7, -1, 0, 1, 7], [-7, 0, 3], 4),
    (40, [-13, 2, 5], [-39, -20, 0, 38], 5), (9, [-3, 1, 4], [-8, -2, 0, 5, 8], 6),
    (5000, [-300, -17, -1, 0, 1, 17, 300], [-300, -17, -1, 0, 1, 17, 300], 4),
    (100000, [5, 90000], [-99999, -5, 7], 3),
    (5000000, [-4000000, -3, 0, 5, 900000], [-2500000, 0, 7, 3000000], 3)])
def test_chain_plans_match_the_reference_planners(oracle, n, h, s, steps):
    """Every array against the oracle's restatement of the reference planners:
    C structure, pair_ptr, and each record against its GPair (A index, range
    of C positions where both operands hold an element, B index of position 0)."""
    import numpy as np
    ha, sa = np.array(h, np.int32), np.array(s, np.int32)
    info, need = (_lib.ChainStep * steps)(), C.c_size_t(0)
    fn = _lib.load().diagpu_chain_plans
    args = (n, len(h), ha.ctypes.data, len(s), sa.ctypes.data, steps)
    assert fn(*args, None, 0, C.byref(need), info) == _lib.ERR_CAPACITY
    buf = np.zeros(need.value, np.uint8)
    assert fn(*args, buf.ctypes.data, buf.size, C.byref(need), info) == _lib.OK
    at = lambda o, c, dt: buf[o: o + c * np.dtype(dt).itemsize].view(dt)
    layout = lambda o: (o, (n - np.abs(o.astype(np.int64))).astype(np.int32))
    starts = lambda ln: np.concatenate([[0], np.cumsum(ln.astype(np.int64))[:-1]])
    a_off, a_len = layout(ha)
    a_st = starts(a_len)
    b_off = sa
    for t in range(steps):
        b_off, b_len = layout(b_off)
        b_st = starts(b_len)
        c_off, c_len, c_st, nnz = oracle.c_structure(n, a_off, b_off)
        ptr, pairs = oracle.pairs_only(n, a_off, a_len, a_st, b_off, b_len, b_st, c_off)
        x = info[t]
        assert (x.c_ndiag, x.c_nnz, x.n_pairs) == (len(c_off), nnz, ptr[-1])
        assert x.max_pairs == np.diff(ptr).max() and x.b_extent == b_len.sum()
        assert x.has_main == (0 in c_off) and x.b_in_range == 1
        assert np.array_equal(at(x.c_off, x.c_ndiag, np.int32), c_off)
        assert np.array_equal(at(x.c_len, x.c_ndiag, np.int32), c_len)
        assert np.array_equal(at(x.c_starts, x.c_ndiag, np.int64), c_st)
        assert np.array_equal(at(x.pair_ptr, x.c_ndiag + 1, np.int64), ptr)
        rec = at(x.records, 4 * x.n_pairs + 4, np.int32)
        r = rec[:-4].reshape(-1, 4)
        lo = np.maximum(0, np.maximum(-pairs["ash"], -pairs["bsh"]))
        hi = np.minimum(pairs["al"] - pairs["ash"], pairs["bl"] - pairs["bsh"])
        assert (lo < hi).all()
        assert np.array_equal(a_st[r[:, 0]], pairs["ab"].astype(np.int64))
        assert np.array_equal(r[:, 1], lo) and np.array_equal(r[:, 2], hi)
        assert np.array_equal(r[:, 3], pairs["bb"].astype(np.int64) + pairs["bsh"])
        assert rec[-4:].tolist() == [0, 0, h[0], h[-1]]
        b_off = c_off
