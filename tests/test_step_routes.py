"""How one token's step goes through its matrices, on the CPU (fake_hip): by streams of rows where these are the faster way, in tiles where those are."""
import fake_hip

CALLS = """
from powerinfer_amd import lib as pl
L, P = pl.load(), 1 << 20
def closing(rows, ld_att, top=0, ld_act=0, T=1):
    s = pl.LayerOut()
    s.rows, s.T, s.out = rows, T, P
    if ld_att:
        s.wo, s.att, s.ld_att = P, P, ld_att
    if top:
        s.down, s.act, s.ids, s.ld_act, s.top, s.n_expert = P, P, P, ld_act, top, 8
    F.fake_clear_counts()
    assert L.pi_k_layer_out_step(C.byref(s), None) == 0
    return count("layer_out_one"), count("layer_out_step")
def first(top, ff, cols, T=1):              # workgroups; ff gate rows and as many up rows
    assert L.pi_k_mix_up_step(None, None, P, 8, ff, cols, 0.9, 1.7, P, T, P, P, top, P, (ff + 31) // 32 * 32, None) == 0
    return F.fake_grid()
"""


def test_closing_a_layer():
    fake_hip.run(CALLS + """
for a in ((2049, 4096), (4096, 4096), (12288, 4096), (1, 4128), (256, 6144), (8192, 4128), (4096, 11008), (2048, 2048, 6, 1408), (4096, 2048, 2, 1024), (4096, 4096, 8, 2048),
          (2048, 2048, 2, 704), (1024, 1056, 2, 1024), (12288, 2048)):
    assert closing(*a) == (1, 0), a
for a in ((4096, 4064), (2048, 4096), (8192, 4096), (2048, 2048), (64, 64), (256, 256, 8, 128), (1024, 1024, 4, 512), (1024, 1024, 2, 1024), (8192, 3072), (12288, 2016), (16385, 6144), (4096, 32768), (4096, 4096, 6, 1408, 2)):
    assert closing(*a) == (0, 1), a
""")


def test_first_matrices_of_experts():
    fake_hip.run(CALLS + """
tiles = lambda top, ff: (2 * ff + 15) // 16 * top
for top, ff, cols in ((1, 16, 2048), (6, 704, 2048), (4, 896, 2048), (6, 1408, 2048), (1, 4097, 2048), (1, 6144, 2048), (1, 12800, 2048), (6, 1408, 1024), (6, 1408, 5120)):
    assert first(top, ff, cols) == tiles(top, ff), (top, ff, cols)
for top, ff, cols, want in ((8, 1024, 2048, 512), (8, 959, 2048, 512), (4, 1024, 2048, 512), (1, 6145, 2048, 512), (1, 9217, 2048, 512), (1, 12801, 2048, 512), (6, 2816, 2048, 512),
                            (1, 1, 4096, 1), (6, 1408, 4096, 512), (2, 64, 8192, 128)):
    assert first(top, ff, cols) == want, (top, ff, cols)
assert first(6, 1408, 4096, T=2) == 2 * tiles(6, 1408)
""")
