"""SpgemmPlan's calls into the library, with a stand-in for the library: what
reaches a kernel is the plan as it is at the call, also where the caller has
changed it since the symbolic phase (fewer entries: the A-stationary kernel
finds A's offset range behind the last of them)."""
import ctypes as C

import pytest
import torch

from diagpu_amd import _lib, spgemm
from diagpu_amd.spgemm import SpgemmPlan
from diagpu_amd.workloads import HM


class _Library:
    """Every entry point succeeds; the symbolic call reports a plan, and the
    arguments of numeric calls are kept."""

    def __init__(self, info, shape):
        self.info, self.shape, self.calls = info, shape, []

    def __getattr__(self, name):
        def fn(*args):
            self.calls.append((name, args))
            if name == "diagpu_spgemm_symbolic_shape":
                for at, src in ((-2, self.info), (-3, self.shape)):
                    p = C.cast(args[at], C.POINTER(type(src)))
                    C.memmove(p, C.byref(src), C.sizeof(src))
            if name == "diagpu_spgemm_full_choice":
                return int(args[4] == self.info.n_pairs)
            return 0
        return fn


def _hm(n, offs):
    o = torch.tensor(offs, dtype=torch.int32)
    ln = n - o.abs()
    st = torch.cumsum(ln, 0) - ln
    return HM(n, o, ln, st.to(torch.int64), torch.zeros(int(ln.sum())), list(offs))


@pytest.fixture
def plan(monkeypatch):
    n, offs = 5000, [-1, 0, 1]
    nnz = sum(n - abs(d) for d in range(-2, 3))
    info = _lib.SpgemmInfo(c_ndiag=5, c_nnz=nnz, n_pairs=9, max_pairs=3, useful_flops=0,
                           a_extent=3 * n - 2, b_extent=3 * n - 2)
    lib = _Library(info, _lib.SpgemmShape(-1, 1, -1, 1, 1))
    monkeypatch.setattr(_lib, "_lib", lib)
    monkeypatch.setattr(spgemm, "_check_dev", lambda t, dtype, name: None)
    A, B = _hm(n, offs), _hm(n, offs)
    p = SpgemmPlan(A, B, stream=7)
    p.test_lib, p.test_C = lib, torch.zeros(nnz)
    return p


def _numeric(p, kernel):
    p.test_lib.calls.clear()
    p.numeric(p.A.values, p.B.values, p.test_C, kernel=kernel)
    return p.test_lib.calls[-1]


def test_entry_count_is_read_at_the_call(plan):
    name, args = _numeric(plan, "astat")
    assert name == "diagpu_spgemm_numeric_astat_f32" and args[12] == 9
    plan.info.n_pairs = 4
    plan._astat = None
    name, args = _numeric(plan, "astat")
    assert name == "diagpu_spgemm_numeric_astat_f32" and args[12] == 4
    assert args[11] == plan._astat.data_ptr() and plan._astat.numel() == 4 * 4 + 4


def test_records_of_the_plan_as_built_are_not_used_for_another(plan):
    assert plan._astat is True
    plan.info.n_pairs = 4
    _, args = _numeric(plan, "astat")
    assert args[12] == 4 and args[11] == plan._astat.data_ptr()


def test_contiguous_band_kernel_only_for_the_plan_as_built(plan):
    assert _numeric(plan, "auto")[0] == "diagpu_spgemm_numeric_full_f32"
    plan.pairs[:32].zero_()                  # entries written, counts the same
    assert not plan.uses_full()
    assert _numeric(plan, "auto")[0] == "diagpu_spgemm_numeric_astat_f32"
    with pytest.raises(ValueError):
        _numeric(plan, "full")
    plan.symbolic()
    assert _numeric(plan, "auto")[0] == "diagpu_spgemm_numeric_full_f32"
    plan.info.n_pairs = 8                    # counts changed
    assert _numeric(plan, "auto")[0] == "diagpu_spgemm_numeric_astat_f32"


def test_prepare_leaves_no_set_up_to_the_general_kernel(plan, monkeypatch):
    """prepare() on a contiguous band: the kernel that kernel_for names has its
    set-up too, so forcing it later waits for nothing."""
    def eligible(n, *args):
        args[-2]._obj.eligible = 1
        return 0
    plan.n = 1 << 18
    monkeypatch.setattr(plan.test_lib, "diagpu_spgemm_band_prepare", eligible, raising=False)
    plan.info.n_pairs = 15                   # from 3 entries per C diagonal on
    plan._written = plan._state()
    plan.test_lib.info.n_pairs = 15
    assert plan.prepare() == "full" and plan.kernel_for() == "band"
    assert plan._band is not None and plan._band[1].eligible
    name, _ = _numeric(plan, "band")
    assert name == "diagpu_spgemm_numeric_band_f32"
