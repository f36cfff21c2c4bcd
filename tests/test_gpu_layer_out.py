"""What closes a step's layer (pi_k_layer_out_step): 8 and 16 rows a workgroup, rows of one or two more than fit, and waves with none, one and up to
nine pieces of the list of attention and expert columns, against float64."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl

pytestmark = pytest.mark.gpu


def bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def wide(u):
    return (u.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


@pytest.mark.parametrize("rows,ld_att,E,top,ld_act,T", [
    (8, 32, 0, 0, 0, 1), (9, 0, 1, 1, 32, 1), (1000, 544, 3, 2, 544, 5), (2048, 4096, 0, 0, 0, 16), (2048, 2048, 40, 6, 1408, 16), (2049, 256, 5, 2, 288, 3), (2056, 0, 9, 4, 1024, 2),
    (4096, 4096, 8, 6, 1408, 1), (4097, 512, 6, 3, 96, 7), (4100, 2048, 4, 4, 512, 16)])
def test_closing_a_layer(rows, ld_att, E, top, ld_act, T):
    L, rng = pl.init(), np.random.default_rng(rows + ld_att + E + T)
    x = rng.standard_normal((T, rows)).astype(np.float32)
    want, mag = x.astype(np.float64), np.abs(x).astype(np.float64)
    out, keep, s = pl.DevBuf.zeros(4 * T * rows), pl.DevBuf.zeros(4 * T * rows), pl.LayerOut()
    hold = [pl.DevBuf(host=x)]
    s.x, s.rows, s.T, s.out, s.keep = hold[0].ptr, rows, T, out.ptr, keep.ptr
    if ld_att:
        wo, att = bf16(rng.standard_normal((rows, ld_att))), bf16(rng.standard_normal((T, ld_att)))
        hold += [pl.DevBuf(host=wo), pl.DevBuf(host=att)]
        s.wo, s.att, s.ld_att = hold[-2].ptr, hold[-1].ptr, ld_att
        want, mag = want + wide(att) @ wide(wo).T, mag + np.abs(wide(att)) @ np.abs(wide(wo)).T
    if E:
        down, act = bf16(rng.standard_normal((E, rows, ld_act))), bf16(rng.standard_normal((T, top, ld_act)))
        ids = np.stack([rng.permutation(E)[:top] for _ in range(T)]).astype(np.int32)
        hold += [pl.DevBuf(host=down), pl.DevBuf(host=act), pl.DevBuf(host=ids)]
        s.down, s.act, s.ids, s.ld_act, s.top, s.n_expert = hold[-3].ptr, hold[-2].ptr, hold[-1].ptr, ld_act, top, E
        for e in range(E):
            t, k = np.nonzero(ids == e)
            if len(t):
                d, a = wide(down[e]), wide(act[t, k])
                want[t] += a @ d.T
                mag[t] += np.abs(a) @ np.abs(d).T
    print(rows, ld_att, E, top, ld_act, T, flush=True)
    pl.check(L.pi_k_layer_out_step(C.byref(s), None))
    got = out.download(np.float32).reshape(T, rows)
    n = ld_att + top * ld_act                                         # products of bf16 are exact in fp32: only their sum rounds
    assert (np.abs(got - want) <= (n / 8 + 32) * 2.0 ** -24 * mag).all()
    assert np.array_equal(keep.download(np.float32).reshape(T, rows), got)


@pytest.mark.parametrize("ld_att,E,top,ld_act,T", [(2048, 9, 3, 1408, 16), (32, 0, 0, 0, 1), (4096, 0, 0, 0, 5), (0, 5, 2, 288, 3), (544, 40, 6, 544, 16), (0, 2, 2, 4096, 7), (6144, 3, 1, 96, 2)])
def test_rows_a_workgroup_do_not_change_the_sums(ld_att, E, top, ld_act, T):
    """A matrix's first rows by themselves (8 rows a workgroup) and inside one of twice as many (16): the same bits."""
    L, rng = pl.init(), np.random.default_rng(ld_att + E + T)
    many, few = 4096, 1000                                            # 256 and 63 workgroups of 16 rows for 256 compute units
    wo, att = bf16(rng.standard_normal((many, max(ld_att, 32)))), bf16(rng.standard_normal((T, max(ld_att, 32))))
    down, act = bf16(rng.standard_normal((max(E, 1), many, max(ld_act, 32)))), bf16(rng.standard_normal((T, max(top, 1), max(ld_act, 32))))
    ids = np.stack([rng.permutation(max(E, 1))[:max(top, 1)] for _ in range(T)]).astype(np.int32)
    got = []
    for rows in (few, many):
        out, s = pl.DevBuf.zeros(4 * T * rows), pl.LayerOut()
        hold = [pl.DevBuf(host=np.ascontiguousarray(a)) for a in (wo[:rows], att, down[:, :rows], act, ids)]
        s.rows, s.T, s.out = rows, T, out.ptr
        if ld_att:
            s.wo, s.att, s.ld_att = hold[0].ptr, hold[1].ptr, ld_att
        if E:
            s.down, s.act, s.ids, s.ld_act, s.top, s.n_expert = hold[2].ptr, hold[3].ptr, hold[4].ptr, ld_act, top, E
        print(rows, ld_att, E, top, ld_act, T, flush=True)
        pl.check(L.pi_k_layer_out_step(C.byref(s), None))
        got.append(out.download(np.float32).reshape(T, rows)[:, :few])
    assert np.array_equal(*got) and got[0].any()
