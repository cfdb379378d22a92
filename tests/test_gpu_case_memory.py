"""The device memory that a case takes against the figure that admission uses (mose_case_bytes): nothing is reserved
twice."""
import pytest

from mosegpu import Context, DeviceCase, cases, serve

pytestmark = pytest.mark.gpu

GRAIN = 4 << 20      # the allocator hands out whole 2 MiB pages; a case makes a few allocations beside its slab


def taken(case):
    """Bytes of device memory that creating the case takes, on a context whose kernels are loaded."""
    ctx = Context(case.tables)
    DeviceCase(ctx, case).destroy()
    before = ctx.info()["hbm_free"]
    dc = DeviceCase(ctx, case)
    out = before - ctx.info()["hbm_free"]
    dc.destroy()
    ctx.close()
    return out


def test_viscous_box_takes_no_more_than_stated(gpu_ready):
    case = cases.taylor_green(128, 1)
    # 98,304 connection records: their plan is 20 MB, all of it in use
    got, stated = taken(case), serve.case_bytes(case)
    print(f"case memory: {got} B taken, {stated} B stated", flush=True)
    assert got <= stated + GRAIN


def test_unplanned_records_take_nothing(gpu_ready):
    case = cases.riemann2d(700, 1)
    # 980,000 no-flux records of the one-cell direction that no stage reads: 94 MB of plan if they were planned
    got, stated = taken(case), serve.case_bytes(case)
    print(f"case memory: {got} B taken, {stated} B stated", flush=True)
    assert got <= stated - (80 << 20)


def test_plain_only_cases_plan_nothing(gpu_ready):
    """Residual smoothing runs the plain path: no plan in the stated figure, nor in what is taken."""
    case = cases.taylor_green(128, 1)
    planned = serve.case_bytes(case)
    case.scheme.irs, case.scheme.irs_beta, case.scheme.irs_njacobi = 1, 0.5, 2
    smoothing = (5 + 2 * 5) * case.layout.NC * 8      # the residual and the two sweeps
    got, stated = taken(case), serve.case_bytes(case)
    print(f"case memory: {got} B taken, {stated} B stated", flush=True)
    assert stated <= planned + smoothing - (18 << 20) + GRAIN
    assert got <= stated
