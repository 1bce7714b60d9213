"""Host model of the swizzled input rings of the chain GEMM (xg_gemm_kernel) and the wide grouped GEMM (gw_gemm_kernel),
k_prefill.hip: a copy by hand of the formulas for every lane's source address and LDS destination, checked so that each
fragment read finds the 16 bytes meant for it, every read and write stays in its row, array and ring, and the reads of 8
consecutive lanes lie in different banks. XG_NW, XG_MS, GP_NW, GW_MT and GW_GR are read from the source; the formulas are
not, so a change of the kernels' addressing has to be made here too (the GPU tests hold the kernels themselves)."""
import os
import re

import numpy as np
import pytest

from conftest import ROOT

TEXT = open(os.path.join(ROOT, "glm-flash-lite_amd", "csrc", "k_prefill.hip")).read()
LANE = np.arange(64)


def _const(name):
    return int(re.search(r"constexpr int %s = (\d+);" % name, TEXT).group(1))


@pytest.mark.parametrize("ms", [16, 32, 64])
def test_chain_gemm_input_ring(ms):
    nw, row = _const("XG_NW"), 8 * 16 * 4
    assert ms <= _const("XG_MS") and ms % nw == 0
    ring = np.full((ms, row // 4), -1)                       # source dword of slot row sl held at each LDS dword
    for wave in range(nw):
        for r in range(ms // nw):
            sl = wave * (ms // nw) + r
            vo = (((LANE >> 2) ^ (sl & 7)) << 4) + (LANE & 3) * 4
            for h in range(row // 256):
                src = h * 256 + vo
                assert src.min() >= 0 and src.max() + 4 <= row
                ring[sl, (h * 256 + 4 * LANE) // 4] = src // 4
    assert (np.sort(ring, axis=1) == np.arange(row // 4)).all()   # each row is a permutation of its own bytes
    j, n = LANE >> 4, LANE & 15
    for t8 in range(8):
        for b in range(ms // 16):
            at = (t8 >> 2) * 256 + (16 * b + n) * row + (((4 * (t8 & 3) + j) ^ (n & 7)) << 4)
            for i in range(4):
                assert (ring.reshape(-1)[at // 4 + i] == t8 * 16 + 4 * j + i).all()
            for g in range(8):                                # 8 lanes read 8 different 16-byte groups of banks
                assert len(set((at[8 * g:8 * g + 8] // 16) % 16)) == 8
        for m in range(ms):                                   # the single-slot chains' broadcast reads
            at = (t8 >> 2) * 256 + m * row + (((4 * (t8 & 3) + j) ^ (m & 7)) << 4)
            assert (ring.reshape(-1)[at // 4] == t8 * 16 + 4 * j).all()


@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 79, 80, 81, 159, 160])
def test_wide_gemm_input_ring(T):
    mt, nw, gr, kdim = _const("GW_MT"), _const("GP_NW"), _const("GW_GR"), 512
    row = gr * 16 * 2
    assert mt % (2 * nw) == 0 and T <= mt
    un = (LANE & 31) >> 2
    x1 = (un >> 1) * 64 + (un & 1) * 16 + (LANE & 3) * 4
    x2 = x1 + (LANE >> 5) * kdim * 2
    for g in range(4):
        ring = np.full(mt * row // 4, -1)
        for wave in range(nw):
            for k in range(mt // 2 // nw):
                pr = wave + nw * k
                if 2 * pr >= T:
                    continue
                sw = ((pr & 6) << 5) | ((pr & 1) << 4)
                src = ((x2 if 2 * pr + 1 < T else x1) ^ sw) + 2 * pr * kdim * 2 + (g >> 1) * 256 + (g & 1) * 32
                assert src.min() >= 0 and src.max() + 4 <= T * kdim * 2      # inside the pass's rows
                dst = pr * 2 * row + 4 * LANE
                assert dst.max() + 4 <= mt * row
                ring[dst // 4] = src // 4
        q, i16 = LANE >> 4, LANE & 15
        for rp in range(gr // 2):
            for mb in range((T + 15) // 16):
                at = mb * 16 * row + ((i16 * row + (((2 * q) ^ (i16 >> 1)) << 4)) ^ (rp << 4))
                slot = mb * 16 + i16
                ok = slot < T
                # stored group g / 2 of 8 tile rows: [q][8 tile rows][4] fp16; this half's row pair rp
                want = slot * kdim * 2 + (g >> 1) * 256 + q * 64 + (g & 1) * 32 + rp * 16
                for i in range(4):
                    assert (ring[at // 4 + i][ok] == (want // 4 + i)[ok]).all()
                for lanes in range(8):
                    assert len(set((at[8 * lanes:8 * lanes + 8] // 16) % 16)) == 8
