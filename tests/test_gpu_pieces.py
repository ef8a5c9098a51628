"""The fused kernel's two ways through a call: pieces (16, 32 or 64 rows whose key tiles are split
over a block's waves, where that many rows do not fill the chip) and the blocks that stream
every tile. Both follow one contract, so every P byte equals the oracle's on either way; the
outputs differ by the order of the binary32 sums (helpers.output_bound). The shapes sit at the
edges of the choice on a 256-CU chip (rows and key tiles), with ragged last pieces, last tiles that a split has alone
and splits without a tile.
"""
import numpy as np
import pytest
import torch

import vcx
from helpers import bits, cosine, dtype_name, make_qkv, output_bound
from oracle import vc_oracle as o

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

MODES = {  # name: (expcast, smooth, channel scale)
    "folded": (True, False, True), "unfused": (True, True, True), "block": (True, True, False),
    "control": (False, False, True), "control_smooth": (False, True, True),
}
ROUTES = [  # D, H, Nq, Nk: the way taken (folded: the folded encode's own way)
    (64, 1, 37, 1100),    # 1 group x 8 splits, the second step has one tile
    (64, 2, 2048, 130),   # too few tiles: streaming blocks; folded: 256 pieces of one group exactly
    (64, 2, 2049, 129),   # too few tiles; folded: 2 groups x 4 splits
    (64, 2, 2048, 520),   # 256 pieces of one group exactly, five tiles
    (64, 2, 2049, 420),   # 2 groups x 4 splits, one tile each
    (64, 2, 2049, 300),   # three tiles: streaming blocks; folded: a split has no tile
    (64, 5, 2047, 300),   # streaming blocks
    (64, 5, 2047, 3000),  # 4 groups x 2 splits from 24 tiles on
    (64, 5, 2047, 1000),  # 8 tiles: folded and block only
    (64, 9, 1100, 420),   # 4 groups x 2 splits: 81 streaming blocks would not deal out evenly
    (64, 9, 2047, 300),   # streaming blocks
    (64, 1, 20, 17000),   # more than a chunk of 16 tiles per split
    (128, 1, 37, 1100),   # 2 groups x 4 splits
    (128, 1, 200, 20),    # up to eight pieces, at one tile too
    (64, 1, 120, 130),    # and at D64 at two
    (128, 4, 2048, 130),  # too few tiles; folded: 256 pieces of two groups exactly
    (128, 4, 2048, 500),  # 256 pieces of two groups exactly
    (128, 4, 2049, 257),  # too few tiles; folded: 4 groups x 2 splits
    (128, 4, 2049, 500),  # 4 groups x 2 splits: 68 streaming blocks would not deal out evenly
    (128, 5, 2047, 1000),  # 80 would: pieces for per-block V scales only
    (128, 9, 2047, 300),  # streaming blocks
    (128, 1, 20, 8900),   # more than a chunk of 16 tiles per split
]


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("route", ROUTES, ids=lambda r: "D%d_%dx%dx%d" % r)
def test_p_bytes_and_output_on_either_way(route, mode):
    D, H, Nq, Nk = route
    dtype = torch.float16 if mode == "control" else torch.bfloat16
    print("case: pieces", route, mode, flush=True)
    expcast, smooth, channel = MODES[mode]
    q, k, v = make_qkv(1, H, Nq, Nk, D, dtype, seed=Nq + Nk, kind="outlier" if smooth else "normal")
    q8, qs, k8, ks, _ = vcx.prepare_qk(q.to(DEV), k.to(DEV))
    v8, vs, means = vcx.prepare_v(v.to(DEV), smooth=smooth, channel_scale=channel)
    args = (q8, k8, v8, qs, ks, vs, means if smooth else None, expcast, smooth, 0 if dtype == torch.float16 else 1,
            D ** -0.5)
    options = dict(channel_scale=channel, affine=mode == "folded")
    out, codes = vcx.forward(*args, **options, p_rows=(0, Nq))
    plain = vcx.forward(*args, **options, out=torch.full_like(out, float("nan")))
    assert torch.equal(out, plain)  # the dump changes nothing, and every row is written
    # the oracle on 16-row groups (the folded encode decides per group) from both ends and between
    rows = np.unique(np.r_[0:min(48, Nq), Nq // 32 * 16:min(Nq // 32 * 16 + 16, Nq), max(0, Nq // 16 * 16 - 32):Nq])
    identity = np.broadcast_to(np.arange(Nk), (1, H, Nk))
    st = o.prepare(bits(q), bits(k), bits(v), v_smooth=smooth, permutation=identity, dtype=dtype_name(dtype),
                   expcast=expcast, v_scale_mode="channel" if channel else "block")
    eout, ecodes = o.reference(st, query_indices=rows, return_codes=True, affine=mode == "folded")
    np.testing.assert_array_equal(codes.cpu().numpy()[:, :, rows], ecodes)
    got = out.float().cpu().numpy()[:, :, rows]
    err, bound = output_bound(got, eout)
    if not channel:
        # the mean term's factor mean * vs goes into its MFMA as RN_f16: off by at most 2^-11 of itself
        # in each tile, and the output is a mean of the tiles' terms. Either way of a call measures
        # 1.008 of the bound without this at [1,9,1100 x 420,64], one element in 58000.
        bound += 2.0 ** -11 * np.abs(st["means"].astype(np.float64) * st["vs"]).max(axis=2, keepdims=True)
    assert np.all(err <= bound), float((err / bound).max())
    assert cosine(got, eout) >= 0.9999


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("expcast,affine", [(True, True), (True, False), (False, False)])
def test_fp8_scores_give_the_same_bytes_on_either_way(D, expcast, affine):
    # 9 heads x 2047 rows stream every tile; one head and three heads of the same payload run as
    # pieces (of one or two groups), nine heads x 1100 rows as pieces of four. The scores come
    # from the same MFMAs, so every P byte is the same.
    print("case: pieces fp8", D, expcast, affine, flush=True)
    q, k, v = (x.to(DEV) for x in make_qkv(1, 9, 2047, 1100, D, torch.bfloat16, seed=17))
    q8, qs, k8, ks, _ = vcx.prepare_qk_fp8(q, k)
    v8, vs, _ = vcx.prepare_v(v)

    def run(n, rows):
        part = [x[:, :n].contiguous() for x in (q8, k8, v8, qs, ks, vs)]
        part[0], part[3] = part[0][:, :, :rows].contiguous(), part[3][:, :, :(rows + 63) // 64].contiguous()
        return vcx.forward_fp8(*part, expcast, 1, D ** -0.5, affine=affine, p_rows=(0, rows))

    out, codes = run(9, 2047)
    for n, rows in ((1, 2047), (3, 2047), (1, 70), (9, 1100)):
        got, part = run(n, rows)
        assert torch.equal(part, codes[:, :n, :rows])
        err, bound = output_bound(got.float().cpu().numpy(), out[:, :n, :rows].float().cpu().numpy())
        assert np.all(err <= 2 * bound), float((err / bound).max())  # two roundings of the output
