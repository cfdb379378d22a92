"""The chemistry kernels' two forms of the rates of progress against the oracle, bit for bit: mechanisms at the limits
of the two-round form (at most 20 reactions, 10 of them third body or falloff, whole orders summing to at most 2 on a
side) and past each of them (the general loops), in batches that leave teams and wavefronts partly idle."""
import dataclasses

import numpy as np
import pytest

from mosegpu import Context, DeviceChem, chem
from mosegpu.core import ThermoTables
from oracle_bind import OracleChem

pytestmark = pytest.mark.gpu

BASE = chem.h2_air_mechanism()
W = BASE.ns + 1


def with_rows(extra, order=None):
    """The mechanism with Arrhenius reactions appended after the other Arrhenius ones: extra = a list of (ni1 row,
    ni2 row, eps row, kf, kb)."""
    na = BASE.n_arrh
    put = lambda a, rows: np.ascontiguousarray(np.concatenate([a[:na], np.array(rows).reshape(-1, a.shape[1]), a[na:]]))
    return dataclasses.replace(
        BASE, ni1=put(BASE.ni1, [e[0] for e in extra]), ni2=put(BASE.ni2, [e[1] for e in extra]),
        eps=put(BASE.eps, [e[2] for e in extra]),
        kf=np.ascontiguousarray(np.concatenate([BASE.kf, [e[3] for e in extra]])),
        kb=np.ascontiguousarray(np.concatenate([BASE.kb, [e[4] for e in extra]])))


def slow_copy(q, scale=1e-3):
    return (BASE.ni1[q].copy(), BASE.ni2[q].copy(), BASE.eps[q].copy(), scale * BASE.kf[q], scale * BASE.kb[q])


def third_body(q):
    e = slow_copy(q)
    e[0][BASE.ns] = 1.0
    e[2][:BASE.ns] = 1.0
    return e


def ordered(q, **orders):
    e = slow_copy(q, 1e-6)
    for sp, nu in orders.items():
        e[0][chem.SPECIES.index(sp)] = nu
    return e


def lindemann():
    """The last Troe reaction as a Lindemann one."""
    return dataclasses.replace(BASE, troe=np.ascontiguousarray(BASE.troe[:1]), lind=np.ascontiguousarray(BASE.troe[1:, :3]))


def all_third_body():
    ni1, eps = BASE.ni1.copy(), BASE.eps.copy()
    new = np.flatnonzero(ni1[:BASE.n_arrh, BASE.ns] == 0)[:7]       # 4 + 2 + 7 = 13 in the first round: too many
    ni1[new, BASE.ns] = 1.0
    eps[new, :BASE.ns] = 1.0
    scale = np.ones(BASE.n_arrh)
    scale[new] = 1e-2
    return dataclasses.replace(BASE, ni1=ni1, eps=eps, kf=np.ascontiguousarray(BASE.kf * scale[:, None]),
                               kb=np.ascontiguousarray(BASE.kb * scale[:, None]))


MECHS = {
    "20-reactions": lambda: with_rows([slow_copy(2)]),
    "10-in-the-first-round": lambda: with_rows([third_body(1)]),
    "lindemann": lindemann,
    "21-reactions": lambda: with_rows([slow_copy(2), slow_copy(9)]),
    "32-reactions": lambda: with_rows([slow_copy(q) for q in range(13)]),
    "13-third-body": all_third_body,
    "order-3": lambda: with_rows([ordered(0, H=2.0)]),
    "four-species": lambda: with_rows([ordered(0, OH=1.0, H2O=1.0)]),
    "half-order": lambda: with_rows([ordered(1, O=0.5)]),
}


@pytest.mark.parametrize("method", [1, 2], ids=["rodas", "radau5"])
@pytest.mark.parametrize("name", list(MECHS))
def test_mechanism_forms(gpu_ready, name, method):
    mech = MECHS[name]()
    n = 45
    st = chem.h2_air_cells(n, seed=5, T_range=(1150.0, 2400.0))
    st[:9] = np.maximum(st[:9], 1e-9)
    print(f"mechanism {name}, method {method}, {n} cells", flush=True)
    ctx = Context(ThermoTables(mech.wm, mech.cp, mech.h, names=mech.names))
    dc = DeviceChem(ctx, mech, n)
    dc.upload(st)
    dc.advance(1e-7, chem.ode_opts(1e-7, 1e-11, method=method))
    dev, hr, idid, nstep = dc.download()
    dc.destroy()
    ctx.close()
    ref, hr_o, idid_o, nstep_o = OracleChem(mech, nthreads=8).advance(st, 1e-7, 1e-7, 1e-11, method=method)
    assert np.all(idid_o == 1)
    assert np.array_equal(idid, idid_o) and np.array_equal(nstep, nstep_o)
    assert np.array_equal(dev, ref) and np.array_equal(hr, hr_o)
