"""CPU audit of the kpair GEMM's memory accesses (q4_gemm_kpair.hip), as
test_access_audit.py does for the other kernels: the kernel's index arithmetic restated
in numpy and checked against the buffers and LDS arrays it addresses, over every tile
height, odd shapes, two-plane handles and K splits."""

import numpy as np
import pytest
from test_access_audit import OOB, REC, REC_SB, chk_buf, in_sb_part, in_tile_part, layout, tile_of

LANE = np.arange(64)
COL, KQ = LANE & 15, LANE >> 4


def audit_kpair(m, n, k, kmt, splits, kx=None):
    L = layout(n, k)
    kx = kx or k
    gx, groups, gp = kx // 64, L["g"], L["gp"]
    bm = 16 * kmt
    mtiles, ntiles = -(-m // bm), -(-n // 256)
    octets = -(-groups // 8)
    per = -(-octets // splits)
    g_split = per * 8
    splits = -(-octets // per)
    xbytes = m * kx * 2
    slot = 4 * bm * 8  # 16-byte units of an x slot
    ycount = np.zeros((splits, m, n), np.int32) if m * n * splits <= 2_000_000 else None
    nwg = mtiles * ntiles
    for bid in range(nwg) if nwg <= 24 else sorted({0, 1, nwg // 2, nwg - 2, nwg - 1}):
        mt, nt = tile_of(bid, nwg, mtiles, ntiles)
        for y in range(splits):
            g0 = y * g_split
            g1 = min(groups, g0 + g_split)
            assert g0 < g1 and g0 % 8 == 0
            p_end = (g1 + 1) // 2
            seen = np.zeros(groups, np.int32)
            for s in range(g0 // 4, -(-g1 // 4)):
                filled = np.zeros(slot, np.int32)
                for wave in range(8):
                    st, wn = wave >> 2, wave & 3
                    rbw = nt * 16 + wn * 4
                    for u in range(kmt):
                        b = 8 * u + wave
                        h4, rb8 = divmod(b, 2 * kmt)
                        g = 4 * s + h4
                        row = mt * bm + rb8 * 8 + (LANE >> 3)
                        c = (LANE & 7) ^ ((4 * (rb8 & 1) + (LANE >> 4)) & 7)
                        # the position of chunk c in its row is c ^ ((row >> 1) & 7)
                        r = rb8 * 8 + (LANE >> 3)
                        assert (((LANE & 7) ^ ((r >> 1) & 7)) == c).all()
                        voff = (row * kx + 8 * c) * 2
                        assert (voff < 2 ** 32).all()
                        if g < g1:
                            src = g - gx if g >= gx else g
                            chk_buf("kpair x", np.where(voff < xbytes, voff + src * 128, OOB), 16, xbytes, xbytes)
                            assert ((voff < xbytes) == (row < m)).all()
                        filled[b * 64 + LANE] += 1
                    p = 2 * s + st
                    if p < p_end:
                        for j in range(4):
                            rb = rbw + ((j + 2 * st) & 3)
                            off = rb * gp * REC + LANE * 16
                            assert (off < 2 ** 32).all() and ((off < L["rec_bytes"]) == (rb < L["nb"])).all()
                            ok = off < L["rec_bytes"]
                            assert not ok.any() or in_tile_part(off[ok] + p * REC, 16)
                            chk_buf("kpair w", np.where(ok, off + p * REC, OOB), 16, L["rec_bytes"], L["rec_bytes"])
                            so = rb * gp * REC + COL * 8
                            ok = so < L["sb_bytes"]
                            assert (ok == (rb < L["nb"])).all()
                            assert not ok.any() or in_sb_part(so[ok] + p * REC, 8)
                            chk_buf("kpair s", np.where(ok, so + p * REC, OOB), 8, L["sb_bytes"], L["sb_bytes"])
                        if wn == 0:
                            seen[2 * p:min(2 * p + 2, groups)] += 1
                    for jj in range(2):  # the scale/bias words of the step's groups, the wave's own half
                        po = 2 * s + (KQ >> 1)
                        rb = rbw + 2 * st + jj
                        off = np.where(po < p_end, rb * gp * REC + po * REC + COL * 8 + (KQ & 1) * 4, OOB)
                        if rb >= L["nb"]:
                            assert (off >= L["sb_bytes"]).all()
                        ok = off < L["sb_bytes"]
                        assert not ok.any() or in_sb_part(off[ok], 4)
                        chk_buf("kpair bias words", off, 4, L["sb_bytes"], L["sb_bytes"])
                    # operand reads of every row tile, and of the X_g row tiles
                    for hh in range(2):
                        for i in list(range(kmt)) + [min(wn + 4 * q, kmt - 1) for q in range((kmt + 3) // 4)]:
                            for h in range(2):
                                rd = st * 2 * bm * 8 + COL * 8 + (hh * bm + 16 * i) * 8 + ((4 * h + KQ) ^ ((COL >> 1) & 7))
                                assert (rd >= 0).all() and (rd < slot).all()
                assert (filled == 1).all(), "every 16-byte unit of the slot is loaded once"
            assert (seen[g0:g1] == 1).all() and seen.sum() == g1 - g0, "every group once, by one set"
            # the exchange, and the stores of both sets' halves
            assert 3 * kmt * 2 * 64 + (kmt * 2 - 1) * 64 + 63 < slot
            row0 = mt * bm
            rows = min(m - row0, bm)
            for st in range(2):
                for wn in range(4):
                    for j in range(2):
                        rb = nt * 16 + wn * 4 + 2 * st + j
                        nn = rb * 16 + COL
                        for i in range(kmt):
                            for e in range(4):
                                r = 16 * i + 4 * KQ + e
                                off = np.where(nn < n, 4 * KQ * n * 4 + nn * 4, OOB) + (16 * i + e) * n * 4
                                ok = off < rows * n * 4
                                assert (ok == ((r < rows) & (nn < n))).all()
                                if ycount is not None:
                                    np.add.at(ycount, (y, (row0 + r)[ok], nn[ok]), 1)
    if ycount is not None and nwg <= 24:
        assert (ycount == 1).all(), "every output of every split is stored once"
    assert (2 * slot + 2 * kmt * 64) * 16 <= 160 * 1024


@pytest.mark.parametrize("kmt", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("m,n,k,kx", [(1, 16, 64, None), (45, 300, 640, None), (113, 130, 576, None), (200, 257, 1088, None),
                                      (224, 512, 3840, None), (100, 40, 1152, 576), (33, 272, 1280, 640)])
def test_kpair_accesses(m, n, k, kx, kmt):
    for splits in (1, 2, 3):
        audit_kpair(m, n, k, kmt, splits, kx)
