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


def test_the_rule_takes_every_tile_it_may_pick():
    """Every tile of the rule is compiled for every wave count: a launch of each row count at sizes on both sides of its
    lines returns success, and the rule never sends 8 rows or fewer to the wide kernel."""
    L = _lib.lib()
    for kind in (0, 1):
        seg = 64 if kind == 0 else 128
        for n in (1, 300, 2048, 4096, 6144, 16384, 100352):
            for m in (1, 8, 9, 10, 11, 17, 33, 49, 64):
                for waves in (1, 2, 4, 8):
                    code = L.bp_skinny_mf_wide(kind, m, n, 32 * seg, waves, 1, 0)
                    assert (code == 0) if m <= 8 else (code // 256 in (0, 1, 2, 4) and code % 256 <= 4)
                    assert m <= 10 or code > 0


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
