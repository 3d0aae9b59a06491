"""Coaxial batches beyond one launch: several launches of whole items, and items of more workgroups than a launch's."""
import numpy as np
import pytest

import ccoil_abi as abi
import oracle as O

pytestmark = pytest.mark.gpu


def _rows(z, n_ang, n_thk, blocks):
    c = O.make_coil(0.1, 0.05, 0.1, 100, 2.0, pos=(0, 0, z))
    return dict(use_fast=1, n_ang=n_ang, n_thk=n_thk, n_len=1, blocks=blocks, R=c.R, a=c.a, b=c.b, J=c.J, current=c.I,
                turns=float(c.N), frequency=c.freq, pos=tuple(c.pos), alpha=0.0, beta=0.0)


def _value(ctx, d, n, n_ang, n_thk, a_blk, r_blk, what=abi.PAIR_M | abi.PAIR_FT):
    """The primary's angular and the secondary's radial rule in blocks, the primary's thickness rule in one."""
    P = abi.CoilSet.from_rows([_rows(0.0, n_ang, n_thk, (a_blk, 1, 1))])
    S = abi.CoilSet.from_rows([_rows(d, n_ang, n_thk, (1, r_blk, 1))])
    i = np.zeros(n, dtype=np.int64)
    return ctx.pairs_zaxis(P, S, n, what, prim_index=i, sec_index=i)[0]


def test_one_item_of_many_workgroups(ctx):
    """1,100 x 31 blocks of 100 x 100 radial and angular nodes, 3.4e8; thirteen threads to each would be more than the 2^32
    threads of a launch. The value of two blocks, to the rounding of the second differences (1e-10 at this distance)."""
    got = _value(ctx, 0.25, 1, 100, 100, 31, 1100, abi.PAIR_M)
    ref = _value(ctx, 0.25, 1, 100, 100, 2, 2, abi.PAIR_M)
    assert abs(got["M"][0] - ref["M"][0]) <= 1e-10 * abs(ref["M"][0])


def test_items_over_several_launches(ctx):
    """60,000 touching pairs, whose rules stay whole: 4.6 million workgroups. All have the value of one."""
    got, one = _value(ctx, 0.1, 60000, 80, 20, 1, 1), _value(ctx, 0.1, 1, 80, 20, 1, 1)
    for k in ("M", "Fz"):
        assert np.all(got[k] == one[k][0]), k
