"""The sparse FFN of a prompt chunk over the neurons that fire for one of its tokens (pi_k_ffn_union_f16), against float64."""
import ctypes as C

import numpy as np
import pytest

from powerinfer_amd import lib as pl

pytestmark = pytest.mark.gpu


def call(ff, rank, cols, T, gated, two, share, fill=None, split=True, silent=None):
    """share: of the neurons, how many may fire at all.  Factors of the predictor are small whole numbers, so that thresholds are met exactly."""
    L, rng = pl.init(), np.random.default_rng(ff + T + rank)
    up, gate, x, down = ((rng.standard_normal(s) / np.sqrt(s[1]) ** (s[0] != T)).astype(np.float16) for s in ((ff, cols), (ff, cols), (T, cols), (ff, cols)))
    fc2, hid = rng.integers(-3, 4, (ff, rank)).astype(np.float16), rng.integers(0, 3, (T, rank)).astype(np.float16)
    hid[:, 0] = 1
    fc2[rng.random(ff) >= share, 0] = -30000                              # never fires
    if silent is not None:                                                # exactly as many never fire, the others for some token or all of them
        fc2[:, 0] = 400
        fc2[rng.choice(ff, silent, replace=False), 0] = -30000
    a1, a2 = rng.standard_normal((2, T, cols)).astype(np.float32)
    lg = (hid.astype(np.float64) @ fc2.astype(np.float64).T).astype(np.float32)
    thr = 20.0
    active = ~(lg < thr)
    if fill is not None:
        up[~active.any(0)] = fill                                         # rows that nobody reads
        down[~active.any(0)] = fill
    b = [pl.DevBuf(host=np.ascontiguousarray(a)) for a in (fc2, hid, up, gate, down, x, a1, a2)]
    scratch, h, out, n = pl.DevBuf(L.pi_k_ffn_union_scratch(ff, T) + 64), pl.DevBuf(2 * T * ff + 64), pl.DevBuf(4 * T * cols + 64), pl.DevBuf(16)
    room = [pl.DevBuf(4 * T * cols + 64) for _ in range(3)]
    parts = (C.c_void_p * 3)(*(r.ptr for r in room)) if split else None
    for d in [scratch, h, out] + room:
        pl.check(L.pi_memset(d.ptr, 0xAB, d.nbytes))
    print(ff, rank, cols, T, gated, two, share, flush=True)
    pl.check(L.pi_k_ffn_union_f16(b[0].ptr, rank, b[1].ptr, b[2].ptr, b[3].ptr if gated else None, b[4].ptr, ff, cols, b[5].ptr, T, thr, scratch.ptr, h.ptr, parts, b[6].ptr,
                                  b[7].ptr if two else None, out.ptr, n.ptr, None))
    pl.sync()
    for d in [scratch, h, out] + room:
        assert (d.download(np.uint8)[-64:] == 0xAB).all()
    u, g = (x.astype(np.float64) @ w.T.astype(np.float64) for w in (up, gate))
    with np.errstate(invalid="ignore"):
        v = np.where(active, np.maximum(g, 0) * u if gated else np.maximum(u, 0), 0)
    want = np.where(active.any(0)[:, None], down, 0).astype(np.float64)
    # h is rounded to fp16 where the sums' own error leaves it, and the sums over the neurons are fp32's
    bound = 2.0 ** -10 * np.abs(v) @ np.abs(want) + 1e-4 * np.sqrt(max(1, active.sum(1).max())) * np.abs(v).max() * np.abs(want).max() * 2.0 ** -4
    want = v @ want + a1 + (a2 if two else 0)
    got = out.download(np.float32)[:T * cols].reshape(T, cols)
    assert n.download(np.int32)[0] == active[-1].sum()
    assert (np.abs(got - want) <= bound + 1e-6 * np.abs(want)).all(), float((np.abs(got - want) / (bound + 1e-6 * np.abs(want))).max())
    call.listed = scratch.download(np.int32)[-20]                         # (the last word but three ahead of the guard)
    return active.any(0).sum()


@pytest.mark.parametrize("gated,two", [(True, False), (False, True)])
@pytest.mark.parametrize("ff,rank,cols,T,share", [(256, 256, 256, 1, 1.0), (384, 320, 512, 17, 0.3), (1152, 256, 256, 63, 0.1), (640, 256, 256, 64, 1.0), (4352, 256, 512, 65, 0.5), (2176, 512, 768, 129, 0.02),
                                                  (1024, 256, 1280, 257, 0.9), (11008, 1024, 4096, 140, 0.4), (32768, 256, 256, 130, 0.6), (512, 256, 4096, 2100, 0.7)])
def test_matches_float64(ff, rank, cols, T, share, gated, two):
    call(ff, rank, cols, T, gated, two, share)


@pytest.mark.parametrize("gated,two", [(True, False), (False, True)])
@pytest.mark.parametrize("ff,T,share", [(4224, 20, 0.5), (5120, 70, 0.5), (4352, 150, 0.9), (2304, 257, 1.0)])
def test_matches_float64_of_8192_columns(ff, T, share, gated, two):
    """A row's sum begins at a column stage that goes with its place, in the list or (the last) among all neurons: places from 2048 on begin elsewhere."""
    call(ff, 256, 8192, T, gated, two, share)


# 160 and 192 units of the down projection for 256 workgroups: in three parts from 72 stages on (4608 listed neurons) where all are 192 and more, in four from 96 (6144) of 256, whole otherwise
@pytest.mark.parametrize("ff,cols,T,silent", [(12288, 4096, 1200, 0), (12288, 4096, 1200, 12288 - 4608), (12288, 4096, 1200, 12288 - 4480), (12160, 4096, 1200, 0), (16384, 4096, 1500, 512),
                                              (16384, 4096, 1500, 16384 - 6144), (16384, 4096, 1500, 16384 - 6016), (16256, 4096, 1500, 0), (12288, 8192, 520, 1000)])
def test_units_that_do_not_fill_the_chip(ff, cols, T, silent):
    call(ff, 256, cols, T, False, True, 1.0, silent=silent)


@pytest.mark.parametrize("gated,two", [(True, False), (False, True)])
@pytest.mark.parametrize("T,silent", [(300, 513), (300, 512), (300, 0), (530, 257), (530, 256)])
def test_around_the_share_from_which_all_neurons_are_gone_through(T, silent, gated, two):
    """8192 neurons: where no more than 512 stay silent (256 from 513 tokens on) bits and rows are gone through as they lie; beyond that the rows of silent ones are not read (NaN)."""
    listed = silent > (256 if T > 512 else 512)
    assert call(8192, 256, 256, T, gated, two, 1.0, silent=silent, fill=np.nan if listed else None) == 8192 - silent
    assert call.listed == ((8192 - silent + 127) // 128 * 128 if listed else 8192)


@pytest.mark.parametrize("ff,rank,cols,T", [(640, 256, 256, 64), (1024, 256, 4096, 600), (11008, 1024, 4096, 140)])
def test_without_room_for_parts(ff, rank, cols, T):
    call(ff, rank, cols, T, True, False, 0.5, split=False)


def test_no_neuron_fires():
    assert call(1024, 256, 512, 200, True, False, 0.0) == 0


def test_rows_of_neurons_that_never_fire_are_not_read():
    """NaN in the rows of up and down of neurons that no token fires."""
    assert 0 < call(1408, 256, 512, 150, True, True, 0.3, fill=np.nan) < 1408


def test_what_it_refuses():
    L = pl.init()
    d = pl.DevBuf.zeros(1 << 20)
    go = lambda rank=256, ff=256, cols=256, T=3, at=d.ptr: L.pi_k_ffn_union_f16(at, rank, d.ptr, d.ptr, None, d.ptr, ff, cols, d.ptr, T, 0.0, d.ptr, d.ptr, None, d.ptr, None, d.ptr, None, None)  # noqa: E731
    assert go(rank=128) != 0 and go(ff=128) != 0 and go(ff=300) != 0 and go(ff=32768 + 128) != 0 and go(cols=384) != 0 and go(T=0) != 0 and go(at=None) != 0 and go(at=d.ptr + 8) != 0


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("off", [None, 4, 8])
def test_parts_that_it_refuses(which, off):
    """A null among the three buffers, or one off 16 bytes: refused ahead of every launch, so that nothing is written."""
    L = pl.init()
    d, out = pl.DevBuf.zeros(1 << 20), pl.DevBuf.zeros(1 << 12)
    pl.check(L.pi_memset(out.ptr, 0xAB, out.nbytes))
    at = [d.ptr + (1 << 18) * (k + 1) for k in range(3)]
    at[which] = None if off is None else at[which] + off
    assert L.pi_k_ffn_union_f16(d.ptr, 256, d.ptr, d.ptr, None, d.ptr, 256, 256, d.ptr, 3, 0.0, d.ptr, d.ptr, (C.c_void_p * 3)(*at), d.ptr, None, out.ptr, None, None) != 0
    pl.sync()
    assert (out.download(np.uint8) == 0xAB).all()
