"""Members of a batch that are not stepped (lg_set_active): one seeded while
the others run starts from its own fields when it joins, and one that is
parked keeps its fields, to the bit.  No dynamic-model update and no disks."""
import numpy as np
import pytest

import lesgo_amd

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "w", "p", "RHSx", "RHSz", "RHSx_f", "dudz", "dvdz", "txz", "tyz", "tzz")


def cfg_of(precision="fp64", cfl=False):
    return lesgo_amd.Config(24, 16, 9, dt=1e-5, precision=precision, initu=False, dyn_init=100,
                            use_cfl_dt=cfl, cfl=0.05)


def fields(c, member):
    return {n: c.download(n, member=member) for n in FIELDS}


def assert_same(a, b):
    for n in a:
        assert np.array_equal(a[n], b[n]), n


@pytest.mark.parametrize("before", [1, 2])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_member_seeded_while_inactive_joins(precision, before):
    with lesgo_amd.Case(cfg_of(precision)) as a:
        a.seed_state(9, 0.1)
        a.step(3)
        want = fields(a, 0)
    with lesgo_amd.Case(cfg_of(precision), members=2) as b:
        b.set_active(1)
        b.seed_state(5, 0.1)
        b.seed_state(9, 0.1, member=1)
        b.step(before)
        b.set_active(2)
        b.step_graph(3)
        assert_same(want, fields(b, 1))


@pytest.mark.parametrize("cfl", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_parked_member_keeps_its_fields(precision, cfl):
    """Member 0 starts anew (from physical fields) and steps on while member 1
    is parked."""
    with lesgo_amd.Case(cfg_of(precision, cfl), members=2) as c:
        for m in range(2):
            c.seed_state(3 + m, 0.1, member=m)
        c.set_counters(0, 0)
        c.step(2)
        c.set_active(1)
        want = fields(c, 1)
        c.seed_state(8, 0.1, member=0)
        c.step(2)
        assert_same(want, fields(c, 1))


@pytest.mark.parametrize("away", [1, 2])
@pytest.mark.parametrize("cfl", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_parked_member_goes_on_where_it_was(precision, cfl, away):
    """The buffers that a step exchanges (RHS and RHS_f among them) change
    places under the parked member too: after an odd and an even number of
    the others' steps it reads back what it held and steps on as if it had
    never been away."""
    with lesgo_amd.Case(cfg_of(precision, cfl)) as a:
        a.seed_state(4, 0.1)
        a.step(3)
        mid = fields(a, 0)
        a.step(2)
        end = fields(a, 0)
    with lesgo_amd.Case(cfg_of(precision, cfl), members=2) as c:
        for m in range(2):
            c.seed_state(3 + m, 0.1, member=m)
        c.set_counters(0, 0)
        c.step(3)
        c.set_active(1)
        c.step(away)
        assert_same(mid, fields(c, 1))
        c.step(2)
        c.set_active(2)
        c.step_graph(2)
        assert_same(end, fields(c, 1))
