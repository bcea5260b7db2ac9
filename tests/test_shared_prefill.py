"""The alternative prefill tiles (w4a16_internal.h): prefill_group_kernel_shared (kSharedTable, ids 1..6),
small-batch prefill whose producer waves dequantise into LDS fragments that other waves multiply, and
prefill_padded_kernel (kPaddedCfg, ids 7..10), the wide tiles for K / 64 that their step does not divide.

CPU: the planner's choice, and an emulation of the kernel's index math (weights -> fragments -> MFMA
operands, x staging, stage walk over odd chunk counts and segments, every address in bounds) against
the oracle's dequantisation.  GPU: every tile forced at the edges of its range, bit for bit against
variant 4 of the same problem, and within the tolerance of the oracle.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from oracle import quant
from tests._helpers import assert_close, gemm, make_problem, ref_gemm, torch_cuda
from tests.test_abi_host import MI355X, Limits, _check, lib, plan  # noqa: F401  (lib is a fixture)

# id: n16 blocks, 16-token tiles, blocks and token tiles per multiplying wave, producer waves
TILES = {1: (2, 1, 1, 1, 8), 2: (2, 2, 2, 1, 8), 3: (4, 1, 2, 1, 12), 4: (4, 2, 2, 2, 12), 5: (4, 3, 2, 3, 8),
         6: (4, 4, 2, 2, 8)}


@pytest.mark.parametrize("M,N,K,want", [
    (17, 4096, 4096, 1), (32, 4096, 4096, 1), (33, 4096, 4096, 2), (64, 4096, 4096, 2), (65, 4096, 4096, 4),
    (32, 6144, 4096, 2), (32, 14336, 4096, 4), (48, 14336, 4096, 5), (64, 14336, 4096, 6), (192, 4096, 4096, 5),
    (24, 10240, 4096, 3 + 1), (16, 14352, 4096, 3), (5, 10256, 1024, 0), (32, 4096, 512, 0), (24, 28672, 4096, 0),
    (512, 4096, 4096, 0), (32, 4096, 14336, 0), (1, 4112, 4160, 1), (37, 4112, 4160, 3), (256, 4112, 4160, 7),
    (1, 28672, 14400, 3), (4096, 4112, 4160, 9), (1024, 4112, 4160, 9), (2048, 14336, 4160, 10), (513, 4112, 4160, 7),
    (1024, 28672, 14400, 8), (513, 6144, 4224, 7), (256, 14336, 4224, 7), (2048, 14336, 4224, 0), (256, 28672, 14464, 9),
    (64, 4112, 14464, 0), (134, 28544, 10880, 9), (271, 18304, 8576, 9), (2048, 28672, 8192, 0)])
def test_planner_choice(lib, M, N, K, want):
    rc, p, err = plan(lib, M=M, N=N, K=K, G=64)
    assert rc == 0 and p.kernel >= 1, err
    assert p.decode_variant == want
    assert _check(lib, p) == 0
    if want:
        p.decode_variant = 11                      # no such tile
        assert _check(lib, p) == 1


@pytest.mark.parametrize("N", [256, 4112, 28672])
@pytest.mark.parametrize("M", [17, 64, 512, 2048])
def test_short_k_keeps_the_tiled_kernel(lib, M, N):
    """The padded tiles lose to prefill_kernel on the shortest K (measured at alt_select)."""
    one_round = -(-M // 64) * -(-N // 128) <= 256
    for chunks in (1, 2, 3, 5, 6, 7):
        rc, p, err = plan(lib, M=M, N=N, K=64 * chunks, G=64)
        assert rc == 0, err
        if chunks < 3 or (chunks < 6 and not one_round):
            assert p.decode_variant == 0, chunks
        elif chunks % 2:
            assert p.kernel <= 4 and p.decode_variant > 0, chunks


@pytest.mark.parametrize("M,N,want", [
    (44, 3952, {16: 2, 18: 0, 20: 0, 22: 0, 24: 2, 26: 2, 64: 2, 128: 2}),           # tile 2: whole stages, or from 24
    (704, 256, {32: 2, 36: 2, 128: 2}), (1024, 256, {28: 2, 32: 2, 34: 0, 52: 0, 128: 0}),   # and at most 22 groups
    (67, 6272, {16: 0, 22: 0, 64: 0, 128: 0}), (97, 4880, {18: 5, 64: 5}), (1078, 480, {24: 5, 40: 5}),
    (106, 5856, {16: 0, 18: 0, 20: 6, 22: 0, 24: 6, 26: 0, 28: 6, 64: 6}),
    (24, 2048, {16: 1, 18: 1, 22: 1, 128: 1}), (79, 3328, {16: 4, 18: 4, 22: 4, 128: 4})])
def test_shared_tiles_only_where_they_win(lib, M, N, want):
    """One K chain, an even number of chunks: the lines of shared_wins, measured on either side."""
    got = {chunks: plan(lib, M=M, N=N, K=64 * chunks, G=64)[1].decode_variant for chunks in want}
    assert got == want


def test_alternative_tiles_ask_for_no_scratch(lib):
    rng = np.random.default_rng(5)
    long = 0
    for _ in range(4000):
        chunks = int(rng.integers(1, 480))
        M, N = int(2 ** rng.uniform(4, 11)), 16 * int(2 ** rng.uniform(6, 10.8))
        rc, p, err = plan(lib, M=M, N=N, K=64 * chunks, G=64)
        assert rc == 0, err
        if p.kernel >= 1 and p.decode_variant:
            long += chunks > 128 and chunks % 2 == 0
            assert (p.workspace_bytes, p.counter_slots, p.splits) == (0, 0, 1), (M, N, chunks, p.kernel, p.decode_variant)
            assert _check(lib, p) == 0
    assert long >= 10


def test_override_that_does_not_fit_is_ignored(lib, monkeypatch):
    M, N, K = 256, 4112, 14400                                           # odd K / 64, several segments
    auto = plan(lib, M=M, N=N, K=K, G=64)[1].decode_variant
    assert auto > 0
    for value, want in (("10", auto), ("11", auto), ("-3", auto), ("x", 0), ("0", 0), ("3", 3), ("9", 9)):
        monkeypatch.setenv("W4A16_PREFILL_SHARED", value)                # id 10 has one K chain only
        assert plan(lib, M=M, N=N, K=K, G=64)[1].decode_variant == want, value
    monkeypatch.setenv("W4A16_PREFILL", "3")                             # both: the tile runs, based on config 3
    p = plan(lib, M=M, N=N, K=K, G=64)[1]
    assert (p.kernel, p.decode_variant) == (3, 9)
    monkeypatch.setenv("W4A16_PREFILL_SHARED", "10")
    p = plan(lib, M=M, N=N, K=K, G=64)[1]
    assert (p.kernel, p.decode_variant) == (3, 0)
    monkeypatch.delenv("W4A16_PREFILL_SHARED")
    p = plan(lib, M=M, N=N, K=K, G=64)[1]
    assert (p.kernel, p.decode_variant) == (3, 0)


def test_route_sweep_forces_every_alternative_tile(lib, monkeypatch):
    import os
    import sys
    import types
    from tests._helpers import PKG
    monkeypatch.syspath_prepend(PKG)
    import route_sweep

    def info(M, N, K, G):
        p = plan(lib, M=M, N=N, K=K, G=G)[1]
        return {"kernel": p.kernel, "decode_variant": p.decode_variant, "splits": p.splits, "kernel_name": ""}

    for var in route_sweep.OVERRIDES:                                    # stray values are cleared
        monkeypatch.setenv(var, "2")
    labels = [label for label, _, _ in route_sweep.forced_plans(types.SimpleNamespace(plan_info=info), 8, 4112, 4160, 64)]
    assert labels == ["p1", "p2", "p3", "p4"] + [f"s{i}" for i in range(1, 11)]
    labels = [label for label, _, _ in route_sweep.forced_plans(types.SimpleNamespace(plan_info=info), 8, 4096, 4096, 64)]
    assert labels and all(label.startswith("d") for label in labels)
    assert not any(var in os.environ for var in route_sweep.OVERRIDES)
    sys.modules.pop("route_sweep", None)


def test_forced_variants_and_small_devices_take_no_shared_tile(lib):
    for v in (1, 2, 3, 4):
        rc, p, err = plan(lib, M=32, N=4096, K=4096, G=128, variant=v)
        assert rc == 0 and p.kernel == v and p.decode_variant == 0, err
    rc, p, err = plan(lib, M=32, N=4096, K=4096, G=128, limits=Limits(256, 64 * 1024, 1024, 942))
    assert rc == 0 and p.decode_variant == 0, err


def _segments(KC):
    if KC <= 128:
        return KC
    s = -(-KC // 64)
    return 2 * -(-KC // (2 * s))


@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("M,N,K,G", [(1, 16, 64, 64), (17, 80, 192, 64), (50, 48, 640, 128), (5, 96, 8256, 64)])
def test_index_math_emulated(tile, M, N, K, G):
    nb_t, tm, cb, ct, np_w = TILES[tile]
    P, RG = np_w // nb_t, 2 * tm
    KC, NBLK = K // 64, N // 16
    seg = _segments(KC)
    rng = np.random.default_rng(K + N + tile)
    q = rng.integers(0, 16, (N, K), dtype=np.uint8)
    s = rng.uniform(0.002, 0.02, (K // G, N)).astype(np.float16)
    x = rng.standard_normal((M, K)).astype(np.float16)
    words = quant.pack_int4(q).view(np.uint32).reshape(NBLK, KC, 32, 4)
    W = quant.dequantize_w4(q, s, G)
    lane = np.arange(64)
    cc, t, g = lane >> 5, (lane >> 3) & 3, lane & 7
    kb, li = lane >> 4, lane & 15
    gm, gn = -(-M // (16 * tm)), -(-NBLK // nb_t)
    XCH, ASZ = tm * 16 * 144, np_w * 4096
    XSZ = 2 * P * XCH

    def deq(w, par, sc):                            # dq_frag: words (2h, 2h + 1) of one nibble parity
        out = []
        for d in (w[0], w[0] >> np.uint32(8), w[1], w[1] >> np.uint32(8)):
            for sh in (4 * par, 16 + 4 * par):
                out.append((np.float16(int(d >> np.uint32(sh)) & 15) - np.float16(8)) * sc)
        return out

    for tile_i in sorted({0, gm * gn - 1}):
        m0, nb0 = tile_i % gm * 16 * tm, tile_i // gm * nb_t
        y = np.zeros((16 * tm, 16 * nb_t))
        k0, end = 0, min(seg, KC)
        while k0 < KC:
            xs = np.full(XSZ // 2, np.nan, np.float16)
            frag = np.full(ASZ // 2, np.nan, np.float16)
            for pw in range(np_w):
                blk, pr = pw // P, pw % P
                nb = min(nb0 + blk, NBLK - 1)
                kc = min(k0 + 2 * pr, KC - 1)
                for l in range(64):
                    c = kc + (int(cc[l]) if kc + 1 < KC else 0)
                    w = words[nb, c, 4 * g[l] + t[l]]
                    row = (kc * 64) // G + (int(cc[l]) if G == 64 and kc + 1 < KC else 0)
                    for h in range(2):
                        for par in range(2):
                            a = (blk * P + pr) * 4096 + (2 * h + par) * 1024 + l * 16
                            frag[a // 2:a // 2 + 8] = deq(w[2 * h:2 * h + 2], par, s[row, nb * 16 + g[l] + 8 * par])
                for i in range(2 * P * RG // np_w):
                    ident = i * np_w + pw
                    xc = ident // RG
                    for l in range(64):
                        lr, qq = (ident - xc * RG) * 8 + (l >> 3), l & 7
                        src = x[min(m0 + lr, M - 1), min(k0 + xc, KC - 1) * 64 + qq * 8:][:8]
                        a = xc * XCH + lr * 144 + (qq >> 2) * 64 + (qq & 3) * 4
                        for e in range(4):
                            xs[a // 2 + 8 * e:a // 2 + 8 * e + 2] = src[2 * e:2 * e + 2]
            for c in range(min(2 * P, end - k0)):
                for wave in range(nb_t * tm // (cb * ct)):
                    cb0, ct0 = wave % (nb_t // cb) * cb, wave // (nb_t // cb) * ct
                    for h in range(2):
                        for b in range(cb):
                            for j in range(ct):
                                aa = ((cb0 + b) * P + (c >> 1)) * 4096 + (c & 1) * 512 + h * 2048 + (li >> 3) * 1024 + \
                                    kb * 128 + (li & 7) * 16
                                ba = c * XCH + ((ct0 + j) * 16 + li) * 144 + kb * 16 + h * 64
                                A = np.zeros((16, 32))
                                B = np.zeros((16, 32))
                                for l in range(64):
                                    A[li[l], kb[l] * 8:kb[l] * 8 + 8] = frag[aa[l] // 2:aa[l] // 2 + 8]
                                    B[li[l], kb[l] * 8:kb[l] * 8 + 8] = xs[ba[l] // 2:ba[l] // 2 + 8]
                                y[(ct0 + j) * 16:(ct0 + j) * 16 + 16, (cb0 + b) * 16:(cb0 + b) * 16 + 16] += B @ A.T
            k0 += 2 * P
            if k0 >= end:
                k0, end = end, min(end + seg, KC)
        rows, cols = min(16 * tm, M - m0), min(16 * nb_t, N - nb0 * 16)
        ref = x[m0:m0 + rows].astype(np.float64) @ W[nb0 * 16:nb0 * 16 + cols].astype(np.float64).T
        # float64 sums of the same exact products in two orders: K * 2^-53 of the mass
        mass = np.abs(x[m0:m0 + rows].astype(np.float64)) @ np.abs(W[nb0 * 16:nb0 * 16 + cols].astype(np.float64)).T
        assert np.all(np.abs(y[:rows, :cols] - ref) <= 2 * K * 2.0**-53 * mass)


# Edges: one chunk, a stage of each tile (2 np / nb chunks) exactly and +- one chunk, odd and even counts,
# K > 8192 (segments, the last one shorter), one n16 block, a partly filled column tile, M at and
# around the token tiles, several rounds of workgroups.
@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("M,N,K,G", [(1, 16, 64, 64), (16, 32, 128, 128), (17, 80, 192, 64), (33, 64, 256, 128),
                                     (31, 48, 320, 64), (32, 272, 384, 128), (49, 144, 448, 64), (64, 512, 512, 128),
                                     (65, 4112, 576, 64), (7, 4112, 4160, 64), (100, 1040, 4096, 128),
                                     (37, 4112, 4160, 64), (40, 528, 8256, 64), (20, 208, 14400, 64),
                                     (130, 256, 14336, 128), (300, 2064, 1088, 64)])
def test_shared_tiles_bitwise_equal(monkeypatch, tile, M, N, K, G):
    torch = torch_cuda()
    import w4a16_opt
    x, q, scales, Wp, key = make_problem(M, N, K, G, seed=M + K)
    want = gemm(Wp, x, scales, variant=4)
    monkeypatch.setenv("W4A16_PREFILL_SHARED", str(tile))
    if M <= 16 and N % 64 == 0 and K % 512 == 0:
        pytest.skip("decode route")
    info = w4a16_opt.plan_info(M, N, K, G)
    print(f"shared tile {tile}: M={M} N={N} K={K} G={G} {info['kernel_name']}", flush=True)
    assert info["decode_variant"] == tile and "prefill_group_kernel_shared" in info["kernel_name"], info
    nb, tm, cb, ct, producers = TILES[tile]
    assert (info["grid"], info["block"]) == (-(-M // (16 * tm)) * -(-(N // 16) // nb), 64 * (producers + nb * tm // (cb * ct)))
    y = gemm(Wp, x, scales)
    assert torch.equal(y, want)
    assert_close(y, ref_gemm(x, q, scales, G, key))


# Padded steps: K / 64 from one chunk to one past whole steps of 2 and 4, one chain and segments (the last
# one odd), tails in M and N.  The 128 x 512 tile (id 10) has no second accumulator set.
@pytest.mark.gpu
@pytest.mark.parametrize("tile", [7, 8, 9, 10])
@pytest.mark.parametrize("M,N,K,G", [(1, 16, 64, 64), (65, 528, 128, 128), (130, 272, 192, 64), (129, 1040, 320, 64),
                                     (300, 2064, 384, 128), (64, 512, 448, 64), (513, 4112, 4160, 64),
                                     (128, 256, 8128, 64), (100, 272, 8256, 64), (200, 528, 14400, 64),
                                     (150, 144, 14464, 128)])
def test_padded_tiles_bitwise_equal(monkeypatch, tile, M, N, K, G):
    torch = torch_cuda()
    import w4a16_opt
    if tile == 10 and K > 8192:
        pytest.skip("one K chain only")
    x, q, scales, Wp, key = make_problem(M, N, K, G, seed=M + K)
    want = gemm(Wp, x, scales, variant=4)
    monkeypatch.setenv("W4A16_PREFILL_SHARED", str(tile))
    info = w4a16_opt.plan_info(M, N, K, G)
    print(f"padded tile {tile}: M={M} N={N} K={K} G={G} {info['kernel_name']}", flush=True)
    assert info["decode_variant"] == tile and "prefill_padded_kernel" in info["kernel_name"], info
    bm, bn, waves = {7: (64, 128, 4), 8: (128, 128, 4), 9: (128, 256, 8), 10: (128, 512, 8)}[tile]
    assert (info["grid"], info["block"], info["splits"]) == (-(-M // bm) * -(-N // bn), 64 * waves, 1)
    y = gemm(Wp, x, scales)
    assert torch.equal(y, want)
    assert_close(y, ref_gemm(x, q, scales, G, key))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(37, 4112, 4160), (24, 4096, 4096), (513, 4112, 4160)])
def test_rows_keep_to_themselves(M, N, K):
    """Infinities and NaN in one token row stay in that row; the other rows keep their bits."""
    torch = torch_cuda()
    x, q, scales, Wp, key = make_problem(M, N, K, 64, seed=3)
    y = gemm(Wp, x, scales)
    x2 = x.clone()
    x2[5, K - 1] = float("inf")
    x2[9, 0] = float("nan")
    y2 = gemm(Wp, x2, scales)
    keep = [m for m in range(M) if m not in (5, 9)]
    assert torch.equal(y2[keep], y[keep])
    v4 = gemm(Wp, x2, scales, variant=4)
    assert torch.equal(torch.isnan(y2), torch.isnan(v4)) and torch.equal(torch.isinf(y2), torch.isinf(v4))
    assert torch.isnan(y2[9]).all()


def test_padded_kernels_leave_pending_loads_alone(tmp_path):
    """The check of test_isa_hazards on the padded kernels: no instruction touches the register of an
    in-flight asm load before its wait."""
    import os
    import subprocess
    import sys
    from tests import test_isa_hazards as hz
    if not os.path.exists(hz.HIPCC):
        pytest.skip("hipcc not available")
    sys.path.insert(0, os.path.join(hz.ROOT, "w4a16-gemm_amd"))
    import build
    src = "w4a16_prefill_wide.hip"
    flags = [f for f in build.compile_flags(src) if f != "-fPIC"]
    out = tmp_path / "wide.s"
    subprocess.run([hz.HIPCC, *flags, "-S", "--cuda-device-only", os.path.join(hz.CSRC, src), "-o", str(out)], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    ks = {k: v for k, v in hz._kernels(out.read_text()).items() if "prefill_padded_kernel" in k}
    assert len(ks) == 7, list(ks)
    assert not {k: v[:5] for k, v in ((k, hz.check_kernel(v)) for k, v in ks.items()) if v}
