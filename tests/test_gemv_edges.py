"""The baseline GEMV kernel at the edges of its loads: rows that end inside a lane's 16 bytes, rows shorter
than one load, K around whole segments and superchunks, one and two row tiles, and the digit split of
every fp16 value.  GPU results are bit for bit the oracle's exact sum."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import c_oracle
from tests.test_gemv import _run, bits, make_gemv


def test_digit_split_of_every_fp16():
    """split_fixed in float32 (w4a16_gemv.hip): hi * 2^24 + lo is a * 2^24 for every finite fp16, and the
    bytes it leaves are the six balanced base-256 digits."""
    h = np.arange(65536, dtype=np.uint16).view(np.float16)
    f = h[np.isfinite(h)].astype(np.float32)
    magic = np.float32(8388608 + 4227200)
    m = (f + np.float32(0.00196)) + magic
    assert np.all((m >= 2**23) & (m < 2**24))
    d = f - (m - magic)
    lo = d.astype(np.float64) * 2.0**24 + 8421504.0                      # the fma: exact in float32
    assert np.all(lo == np.round(lo)) and lo.min() >= 0 and lo.max() < 2**24
    lo, hb = lo.astype(np.int64), m.view(np.uint32).astype(np.int64) & 0xFFFFFF
    X = np.round(f.astype(np.float64) * 2.0**24).astype(np.int64)
    assert np.array_equal((hb - 0x408080) * 2**24 + lo - 0x808080, X)
    digits = [((lo >> (8 * j)) & 255) - 128 for j in range(3)] + [(hb & 255) - 128, ((hb >> 8) & 255) - 128,
                                                                 ((hb >> 16) & 255) - 64]
    assert np.array_equal(sum(dj * 256**j for j, dj in enumerate(digits)), X)
    assert all(dj.min() >= -128 and dj.max() <= 127 for dj in digits)


@pytest.mark.parametrize("kw", list(range(4, 40)) + [511, 513, 514, 515, 897])
def test_row_tail_words_emulated(kw):
    """The lane's words wi .. wi + 3 of a row of kw words: loaded from min(wi, kw - 4), shifted when the
    superchunk crosses the row's end; every word inside the row must come out in its place."""
    row = np.arange(1, kw + 1)
    for p in range(-(-kw // 16)):
        crosses = 16 * (p + 1) > kw and kw % 4 != 0
        for g in range(4):
            wi = 16 * p + 4 * g
            s = min(wi, kw - 4)
            w = row[s:s + 4]
            assert len(w) == 4                                           # in bounds
            if crosses:
                sh = wi - s
                if sh & 1:
                    w = np.array([w[1], w[2], w[3], w[3]])
                if sh & 2:
                    w = np.array([w[2], w[3], w[2], w[3]])
            inside = [e for e in range(4) if wi + e < kw]
            assert [w[e] for e in inside] == [row[wi + e] for e in inside]


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(1, 8), (17, 24), (16, 32), (33, 40), (15, 120), (16, 136), (31, 1016), (40, 2056),
                                 (8200, 2056), (8192, 4072), (9000, 4096), (50, 4104), (20, 8184), (5, 8192), (37, 8200),
                                 (19, 12312), (3, 16400), (2, 131080),
                                 (4097, 32), (4112, 40), (4100, 1016), (4113, 1024), (4096, 1024), (4097, 1032), (8177, 2048),
                                 (8200, 2040), (20490, 1160),
                                 (18, 3072), (33, 3080), (17, 3064)])
@pytest.mark.parametrize("w_off,a_off", [(0, 0), (1, 1), (3, 4)])
def test_gemv_edges(N, K, w_off, a_off):
    print(f"gemv N={N} K={K} w_off={w_off} a_off={a_off}", flush=True)
    W, A, sW, zW = make_gemv(N, K, 11, special=True)
    C = _run(W, A, sW, zW, w_offset=w_off, a_offset=a_off).cpu().numpy()
    assert np.array_equal(bits(C), bits(c_oracle.gemv(W, A, sW, zW, exact=True)))


def test_single_segment_kernels_load_only_what_they_multiply(tmp_path):
    """A wave waits for every load it issued.  Up to K = 1024, 2048 and 3072 the longest segment gives a wave one, two and
    three superchunks, so those instantiations request as many pieces of 16 bytes per row tile, and one of A."""
    import os
    import re
    import subprocess
    import sys
    from tests import test_isa_hazards as hz
    if not os.path.exists(hz.HIPCC):
        pytest.skip("hipcc not available")
    sys.path.insert(0, os.path.join(hz.ROOT, "w4a16-gemm_amd"))
    import build
    flags = [f for f in build.compile_flags("w4a16_gemv.hip") if f != "-fPIC"]
    out = tmp_path / "gemv.s"
    subprocess.run([hz.HIPCC, *flags, "-S", "--cuda-device-only", os.path.join(hz.CSRC, "w4a16_gemv.hip"), "-o", str(out)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    seen = {}
    for name, lines in hz._kernels(out.read_text()).items():
        m = re.search(r"gemv_kernelILb0ELb1ELi(\d)ELb0ELi(\d)EE", name)      # 16-byte loads of A, one segment
        if m:
            text = "\n".join(lines)
            seen[int(m[1]), int(m[2])] = text[:text.index("s_barrier")].count("global_load_dwordx4")
    assert seen == {(rt, pw): 1 + rt * pw for rt, pw in ((1, 1), (1, 2), (1, 3), (1, 4), (2, 1), (2, 2))}
