"""The wide matrix-core kernels (bf16 / int8: 9..64 activation rows; int4: 1..64): every output row equal bit for bit to the same row computed alone
by the one-row kernel at the same K order, and to the oracle, at the edges of its tiles: a single weight row, partial
blocks of 16 weight rows, partial activation blocks, activation tiles in separate workgroups, waves without a segment,
split K, the SiLU epilogue's odd last pair, unaligned output rows."""

from __future__ import annotations

import pytest
import torch

from byteprof_amd import _lib
from byteprof_amd.optim import skinny as S

from .helpers import check_against_oracle, make_weights, oracle_weights, randn_x

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _mf(kind, x, args, waves, split, rb=1, xs=0):
    m, k = x.shape
    n = args[0].shape[0]
    y = torch.full((m, n), 7.0, dtype=torch.bfloat16, device=DEV)
    ws = torch.empty(max(1, split * m * n), dtype=torch.float32, device=DEV)
    sc, sdt = (args[1].data_ptr(), _lib.TORCH_DT[args[1].dtype]) if kind == "int8" else (None, 0)
    _lib.check(_lib.lib().bp_skinny_mf(S._KIND_CODE[kind], x.data_ptr(), args[0].data_ptr(), sc, sdt, y.data_ptr(), m, n,
                                       k, rb, waves, split, xs, ws.data_ptr(), ws.numel() * 4, _lib.stream_ptr(DEV)),
               "bp_skinny_mf")
    return y


@pytest.mark.parametrize("kind", ["bf16", "int8"])
@pytest.mark.parametrize("n,segs,waves,split", [(1, 3, 4, 1), (15, 1, 2, 1), (17, 9, 8, 1), (250, 5, 1, 1),
                                                (1000, 16, 4, 2), (1026, 7, 2, 3), (4100, 4, 4, 1), (9000, 2, 1, 1)])
def test_rows_equal_the_one_row_kernel(kind, n, segs, waves, split):
    k = segs * S.k_segment(kind)
    _, args = make_weights(kind, n, k, seed=n + segs)
    w_np = oracle_weights(kind, args)
    x = randn_x(64, k, seed=segs)
    ones = torch.cat([_mf(kind, x[r:r + 1].contiguous(), args, waves, split) for r in range(64)])
    for m in (9, 10, 16, 17, 31, 33, 48, 49, 64):
        xm = x[:m].contiguous()
        got = _mf(kind, xm, args, waves, split)
        assert torch.equal(got.view(torch.int16), ones[:m].view(torch.int16)), m
    check_against_oracle(got, x, w_np)


@pytest.mark.parametrize("kind", ["bf16", "int8"])
@pytest.mark.parametrize("ffn", [1, 129, 2050])
def test_silu_rows_equal_the_one_row_kernel(kind, ffn):
    k, waves = 6 * S.k_segment(kind), 4
    _, args = make_weights(kind, 2 * ffn, k, seed=ffn)
    x = randn_x(16, k, seed=3)
    sc, sdt = (args[1].data_ptr(), _lib.TORCH_DT[args[1].dtype]) if kind == "int8" else (None, 0)

    def silu(rows):
        out = torch.full((rows.shape[0], ffn), 7.0, dtype=torch.bfloat16, device=DEV)
        _lib.check(_lib.lib().bp_skinny_mf_silu(S._KIND_CODE[kind], rows.data_ptr(), args[0].data_ptr(), sc, sdt,
                                                out.data_ptr(), rows.shape[0], ffn, k, 1, waves, 0,
                                                _lib.stream_ptr(DEV)), "silu")
        return out

    ones = torch.cat([silu(x[r:r + 1].contiguous()) for r in range(16)])
    for m in (9, 11, 16):
        assert torch.equal(silu(x[:m].contiguous()).view(torch.int16), ones[:m].view(torch.int16)), m


def _rows(kind, x, args, waves, split, epi):
    """bp_skinny_mf_rows of all rows of x in one call."""
    m, k = x.shape
    n = args[0].shape[0] // (1 + epi)
    y = torch.full((m, n), 7.0, dtype=torch.bfloat16, device=DEV)
    ws = torch.empty(max(1, split * m * n), dtype=torch.float32, device=DEV)
    sc, sdt = (args[1].data_ptr(), _lib.TORCH_DT[args[1].dtype]) if kind == "int8" else (None, 0)
    _lib.check(_lib.lib().bp_skinny_mf_rows(S._KIND_CODE[kind], x.data_ptr(), args[0].data_ptr(), sc, sdt, y.data_ptr(), m,
                                            n, k, waves, split, epi, ws.data_ptr(), ws.numel() * 4,
                                            _lib.stream_ptr(DEV)), "bp_skinny_mf_rows")
    return y


def _by_eight(kind, x, args, waves, split, epi):
    """The same rows eight at a time: launches of the 8-row kernel."""
    return torch.cat([_rows(kind, x[r:r + 8].contiguous(), args, waves, split, epi) for r in range(0, x.shape[0], 8)])


@pytest.mark.parametrize("kind", ["bf16", "int8"])
@pytest.mark.parametrize("waves", [1, 2, 4, 8])
def test_every_tile_of_the_rule_runs_and_equals_the_8_row_kernel(kind, waves):
    """Every (rp, mb) tile that the rule picks for 17..64 rows of any number of weight rows is compiled for every wave
    count and both epilogues: launched once at the smallest size that has it, each row equal bit for bit to the 8-row
    kernel's, and the plain product to the oracle. The rule never sends 8 rows or fewer to the wide kernel."""
    L, code, seg = _lib.lib(), S._KIND_CODE[kind], S.k_segment(kind)
    k = 2 * waves * seg  # two segments a wave: no straight-line kernel
    tiles = {}
    for n in (2, 30, 300, 2048, 4096, 6144, 8192, 12000, 16384, 20000, 33000):
        assert all(L.bp_skinny_mf_wide(code, m, n, k, waves, 1, 0) == 0 for m in range(1, 9))
        for m in range(9, 65):
            t = L.bp_skinny_mf_wide(code, m, n, k, waves, 1, 0)
            assert t > 0 and t // 256 in (1, 2, 4) and 1 <= t % 256 <= 4, (n, m, t)
            if t not in tiles or n * m < tiles[t][0] * tiles[t][1]:
                tiles[t] = (n, m)
    assert {t // 256 for t in tiles} == {1, 2, 4}, tiles
    for t, (n, m) in tiles.items():
        _, args = make_weights(kind, n, k, seed=n + m)
        x = randn_x(m, k, seed=m)
        for epi in (0, 1):
            if epi == 1 and m <= 16:  # the SiLU launches of up to 16 rows: test_silu_rows_equal_the_one_row_kernel
                continue
            got, want = _rows(kind, x, args, waves, 1, epi), _by_eight(kind, x, args, waves, 1, epi)
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (t, n, m, epi)
        if n <= 2048:
            check_against_oracle(_rows(kind, x, args, waves, 1, 0), x, oracle_weights(kind, args))


@pytest.mark.parametrize("kind", ["bf16", "int8"])
@pytest.mark.parametrize("n,segs,waves,split,epi", [(70, 5, 4, 1, 0), (70, 5, 4, 1, 1), (1030, 9, 2, 2, 0),
                                                    (6150, 4, 4, 1, 1), (6150, 8, 8, 2, 0)])
def test_mf_rows_past_64_rows(kind, n, segs, waves, split, epi):
    """bp_skinny_mf_rows, one launch for a prompt's rows: 5 to 16 activation blocks, several activation tiles per weight
    tile, a last one of one row, the split reduce over all rows; each row equal bit for bit to the 8-row kernel's."""
    k = segs * S.k_segment(kind)
    _, args = make_weights(kind, n, k, seed=n)
    x = randn_x(256, k, seed=segs)
    want = _by_eight(kind, x, args, waves, split, epi)
    for m in (65, 97, 127, 160, 255, 256):
        got = _rows(kind, x[:m].contiguous(), args, waves, split, epi)
        assert torch.equal(got.view(torch.int16), want[:m].view(torch.int16)), m


@pytest.mark.parametrize("n,groups,tile,waves,split,epi", [(70, 5, 16, 4, 1, 0), (300, 9, 32, 8, 2, 0), (300, 3, 32, 2, 1, 1),
                                                           (4100, 4, 64, 1, 1, 0), (22, 3, 16, 4, 1, 0)])
def test_int4_rows_past_64_rows(n, groups, tile, waves, split, epi):
    """bp_skinny_int4_rows past 64 rows, the VALU kernel's shapes (n % 4 != 0: 16 rows a launch inside) among them."""
    k = groups * S.GROUP
    w = (torch.randn(n * (1 + epi), k, generator=torch.Generator(device=DEV).manual_seed(n), device=DEV) * 0.02).to(
        torch.bfloat16)
    packed, scale, zero = S.quantize_int4(w, tile)
    x = randn_x(256, k, seed=n)
    ws = torch.empty(split * 256 * n, dtype=torch.float32, device=DEV)

    def rows(xm):
        y = torch.full((xm.shape[0], n), 7.0, dtype=torch.bfloat16, device=DEV)
        _lib.check(_lib.lib().bp_skinny_int4_rows(xm.data_ptr(), packed.data_ptr(), scale.data_ptr(),
                                                  _lib.TORCH_DT[scale.dtype], zero.data_ptr(), y.data_ptr(), xm.shape[0], n,
                                                  k, tile, waves, split, epi, ws.data_ptr(), ws.numel() * 4,
                                                  _lib.stream_ptr(DEV)), "bp_skinny_int4_rows")
        return y

    ones = torch.cat([rows(x[r:r + 1].contiguous()) for r in range(256)])
    for m in (65, 97, 127, 160, 255, 256):
        got = rows(x[:m].contiguous())
        assert torch.equal(got.view(torch.int16), ones[:m].view(torch.int16)), m
    if epi == 0:
        check_against_oracle(ones, x, S.dequantize("int4", packed, scale, zero).cpu().numpy())


@pytest.mark.parametrize("tile_rows", [16, 32, 64])
@pytest.mark.parametrize("n,groups,waves,split,sdt", [(4, 1, 4, 1, None), (68, 3, 2, 1, torch.float16),
                                                      (300, 9, 8, 2, torch.float32), (1000, 32, 1, 1, None),
                                                      (17000, 2, 4, 1, None), (132, 16, 4, 1, torch.float16),
                                                      (132, 64, 4, 2, None)])
def test_int4_rows_equal_the_one_row_launch(tile_rows, n, groups, waves, split, sdt):
    """bp_skinny_int4_rows at 1..64 rows (one and two activation blocks per workgroup, one and several activation tiles,
    partial weight tiles, waves without a group): each row equal bit for bit to its own launch. In 16-row tiles the 16-row
    kernel takes the one-row launch from 4 groups a wave on, and up to 7 rows from 8 groups on: both sides of those lines."""
    k = groups * S.GROUP
    w = (torch.randn(n, k, generator=torch.Generator(device=DEV).manual_seed(n), device=DEV) * 0.02).to(torch.bfloat16)
    packed, scale, zero = S.quantize_int4(w, tile_rows)
    scale = scale if sdt is None else scale.to(sdt)
    x = randn_x(64, k, seed=n)
    ones = torch.cat([S.skinny_mm(x[r:r + 1].contiguous(), packed, scale, zero, cfg=(waves, split)) for r in range(64)])
    for m in (2, 3, 5, 7, 8, 9, 16, 17, 32, 33, 49, 64):
        got = S.skinny_mm(x[:m].contiguous(), packed, scale, zero, cfg=(waves, split))
        assert torch.equal(got.view(torch.int16), ones[:m].view(torch.int16)), m
    check_against_oracle(got, x, S.dequantize("int4", packed, scale, zero).cpu().numpy())
