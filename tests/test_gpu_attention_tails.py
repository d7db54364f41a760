"""Edges of the attention kernel's tile: every count of key tiles from one to
nine (odd counts padded to even ones, pipelines shorter than their LDS ring)
against last query tiles that leave zero to seven waves without a row.
Same tolerance as the other attention tests."""

from __future__ import annotations

import pytest
import torch

from h3_flash_amd import _ext, flash_attn_func
from oracle.attention import sdpa_reference
from tests.test_gpu_attention import _varlen_workspace, assert_parity

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _qkv(B, Sq, Sk, H, seed):
    g = torch.Generator().manual_seed(seed)
    mk = lambda S: torch.randn((B, S, H, 128), generator=g).to(torch.bfloat16)
    return mk(Sq), mk(Sk), mk(Sk)


@pytest.mark.parametrize("Sk", [1, 64, 65, 128, 190, 256, 257, 320, 384, 447, 512, 513, 576])
@pytest.mark.parametrize("Sq", [1, 33, 256, 257, 300, 480])
def test_key_tiles_and_idle_waves(Sq, Sk):
    q, k, v = _qkv(1, Sq, Sk, 3, Sq * 1000 + Sk)
    out, lse = flash_attn_func(q.to(DEV), k.to(DEV), v.to(DEV), split_tail=False)
    torch.cuda.synchronize()
    ref_out, ref_lse = sdpa_reference(q, k, v)
    assert_parity(out.cpu(), lse.cpu(), ref_out, ref_lse, f"{Sq}x{Sk}")


# At most 32 rows past the whole query tiles: one workgroup per (batch, head)
# after the tiles, or (43 x 6 whole tiles on 256 CUs: 2 over) fewer workgroups
# that take several; beside the queued and the static split, with strided
# views, and with keys from fewer than one per wave to many rounds.
@pytest.mark.parametrize(
    "B, H, Sq, Sk, split",
    [(1, 2, 257, 3, True), (2, 3, 288, 700, True), (1, 40, 1560, 300, True), (1, 43, 1552, 64, True),
     (1, 40, 1537, 100, False), (3, 5, 520, 33, False), (1, 20, 3590, 640, True)],
)
def test_rows_past_the_whole_tiles(B, H, Sq, Sk, split):
    q, k, v = _qkv(B, Sq, Sk, H, Sq + Sk)
    view = torch.empty((B, Sq, H + 1, 128), dtype=torch.bfloat16, device=DEV)[:, :, 1:]
    view.copy_(q)
    out, lse = flash_attn_func(view, k.to(DEV), v.to(DEV), split_tail=split)
    torch.cuda.synchronize()
    rows = sorted({0, Sq // 256 * 256 - 1, *range(Sq // 256 * 256, Sq)})
    ref_out, ref_lse = sdpa_reference(q[:, rows], k, v)
    assert_parity(out.cpu()[:, rows], lse.cpu()[:, :, rows], ref_out, ref_lse, f"{B}x{H}x{Sq}x{Sk}")


# The ragged rows become units only in launches whose tiles all run whole:
# where the tiles are cut into key-range pieces the ragged ones are cut with
# them (the rows equal those of a call with 40 rows more, which has as many
# tiles and no units), and whole tiles stay whole without them.
@pytest.mark.parametrize("H, Sq, Sk", [(8, 2064, 2064), (20, 1296, 1296), (2, 2064, 17000), (16, 1040, 300)])
def test_ragged_rows_of_a_split_launch(H, Sq, Sk):
    q, k, v = (x.to(DEV) for x in _qkv(1, Sq + 40, Sk, H, Sq + Sk))
    got = flash_attn_func(q[:, :Sq], k, v)
    more = flash_attn_func(q, k, v)
    assert torch.equal(got[0], more[0][:, :Sq]) and torch.equal(got[1], more[1][..., :Sq])


@pytest.mark.parametrize("H, Sq, Sk", [(16, 2832, 2832), (8, 5904, 300)])
def test_whole_tiles_beside_ragged_rows_stay_whole(H, Sq, Sk):
    q, k, v = (x.to(DEV) for x in _qkv(1, Sq, Sk, H, Sq + Sk))
    got, whole = flash_attn_func(q, k, v), flash_attn_func(q, k, v, split_tail=False)
    n = Sq // 256 * 256
    assert torch.equal(got[0][:, :n], whole[0][:, :n]) and torch.equal(got[1][..., :n], whole[1][..., :n])


# Units alone: one key, fewer blocks than waves, a last block of one key, no
# keys, many blocks; packed segments with empty ones and unequal key lengths.
@pytest.mark.parametrize("B, H, Sq, Sk", [(1, 1, 1, 1), (2, 3, 33, 0), (1, 4, 31, 257), (1, 5, 640, 640), (3, 2, 70, 225), (1, 2, 32, 2048)])
def test_short_attention(B, H, Sq, Sk):
    q, k, v = _qkv(B, Sq, Sk, H, 7 * Sq + Sk)
    out, lse = flash_attn_func(q.to(DEV), k.to(DEV), v.to(DEV))
    torch.cuda.synchronize()
    if Sk == 0:
        assert (out == 0).all() and (lse == float("-inf")).all()
        return
    ref_out, ref_lse = sdpa_reference(q, k, v)
    assert_parity(out.cpu(), lse.cpu(), ref_out, ref_lse, f"{B}x{H}x{Sq}x{Sk}")


def _runs_as_units(Sq, Sk, H, offsets=None):
    """Whether the call launches without a workspace (asked for, one would be
    named where tiles are cut into pieces)."""
    q, k, v = (torch.zeros((1, S, H, 128), dtype=torch.bfloat16, device=DEV) for S in (Sq, Sk, Sk))
    out, s = torch.empty_like(q), H * 128
    cq, ck, longest = (None, None, 0) if offsets is None else offsets
    rc = _ext.attn_fwd(
        DEV, _ext.ABI_VERSION, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), 0, 1, H, Sq, Sk, 128,
        *(Sq * s, s, 128), *(Sk * s, s, 128), *(Sk * s, s, 128), *(Sq * s, s, 128), 0, 0, 0.1, 0,
        *((0, 0, 0, 0) if cq is None else (cq.data_ptr(), ck.data_ptr(), cq.numel() - 1, longest)),
        0, _ext.H3A_WORKSPACE_ASK,
    )
    assert rc in (_ext.H3A_OK, _ext.H3A_NEED_WORKSPACE)
    torch.cuda.synchronize()
    return rc == _ext.H3A_OK


# Units pass all keys of their head: over long key ranges tiles in key-range
# pieces are shorter, few units or many.
@pytest.mark.parametrize(
    "H, Sq, Sk, units",
    [(1, 64, 2500, True), (5, 640, 640, True), (1, 64, 8000, False), (1, 1, 50000, False), (4, 256, 4000, False), (16, 1, 20000, False)],
)
def test_units_by_key_range(H, Sq, Sk, units):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the rule was timed on a 256-CU part")
    assert _runs_as_units(Sq, Sk, H) == units


@pytest.mark.parametrize(
    "H, qlens, klens, units",
    [(5, [1900, 30, 400], [30000, 26000, 24000], False), (1, [60, 3], [60000, 40000], False), (2, [500, 20, 300], [900, 800, 700], True)],
)
def test_packed_units_by_key_range(H, qlens, klens, units):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the rule was timed on a 256-CU part")
    cq, ck = (torch.tensor([0, *torch.tensor(x).cumsum(0).tolist()], dtype=torch.int32, device=DEV) for x in (qlens, klens))
    assert _runs_as_units(sum(qlens), sum(klens), H, (cq, ck, max(qlens))) == units


@pytest.mark.parametrize("qlens, klens", [([5, 0, 64, 33], [70, 9, 0, 300]), ([1], [1]), ([200, 31, 32], [200, 31, 32])])
def test_short_packed_segments(qlens, klens):
    H = 3
    q, k, v = _qkv(1, sum(qlens), sum(klens), H, sum(qlens))
    cq, ck = (torch.tensor([0, *torch.tensor(x).cumsum(0).tolist()], dtype=torch.int32) for x in (qlens, klens))
    out, lse = flash_attn_func(
        q.to(DEV), k.to(DEV), v.to(DEV), cu_seqlens_q=cq.to(DEV), cu_seqlens_k=ck.to(DEV), max_seqlen_q=max(qlens)
    )
    torch.cuda.synchronize()
    for (a, b), (c, d) in zip(zip(cq[:-1], cq[1:]), zip(ck[:-1], ck[1:])):
        if a == b:
            continue
        if c == d:
            assert (out[:, a:b] == 0).all() and (lse[:, :, a:b] == float("-inf")).all()
            continue
        ref_out, ref_lse = sdpa_reference(q[:, a:b], k[:, c:d], v[:, c:d])
        assert_parity(out[:, a:b].cpu(), lse[:, :, a:b].cpu(), ref_out, ref_lse, f"rows {a}:{b}")


def _overflowed_block(Sq, Sk, H, row, block, seed):
    """q, k, v in which the scores of query row `row` against the 32 keys of
    `block` overflow fp32 to -inf, all other scores being ordinary: the row
    lives in dims 0..63 (where the other keys are tiny), the others in 64..127."""
    q, k, v = _qkv(1, Sq, Sk, H, seed)
    q[..., :64], k[..., :64] = 0, k[..., :64] * 1e-18
    q[:, row, :, :64], q[:, row, :, 64:] = 1e18, 0
    k[:, 32 * block : 32 * block + 32, :, :64] = -1e20
    return q, k, v


# Each wave of a unit starts on its own block of keys: one row whose scores
# there are all -inf, while the wave's other rows have finite ones, keeps the
# weights of the finite blocks that follow. Units of a dense call and of a
# packed one (48 keys leave the later waves without keys), and the ragged rows
# beside whole tiles.
@pytest.mark.parametrize(
    "Sq, Sk, H, row, block, packed",
    [(64, 600, 2, 5, 0, False), (64, 600, 2, 40, 3, False), (40, 48, 3, 39, 0, False), (1296, 300, 40, 1290, 1, False),
     (64, 600, 2, 5, 0, True), (64, 600, 2, 40, 3, True), (40, 48, 3, 39, 0, True)],
)
def test_units_keep_rows_with_a_block_of_overflowed_scores(Sq, Sk, H, row, block, packed):
    q, k, v = _overflowed_block(Sq, Sk, H, row, block, Sq + Sk + block)
    kw = {}
    if packed:
        kw = dict(cu_seqlens_q=torch.tensor([0, Sq], dtype=torch.int32, device=DEV),
                  cu_seqlens_k=torch.tensor([0, Sk], dtype=torch.int32, device=DEV), max_seqlen_q=Sq)
    out, lse = flash_attn_func(q.to(DEV), k.to(DEV), v.to(DEV), **kw)
    torch.cuda.synchronize()
    rows = list(range(row // 32 * 32, min(Sq, row // 32 * 32 + 32)))
    ref_out, ref_lse = sdpa_reference(q[:, rows], k, v)
    assert torch.isfinite(ref_lse).all()
    assert_parity(out.cpu()[:, rows], lse.cpu()[:, :, rows], ref_out, ref_lse, f"{Sq}x{Sk} block {block}")


# Scores that grow from block to block by far more than fp32 exponents hold
# (every rescale taken), that shrink, and one key far above all others: units
# of a dense and a packed call, ragged rows, and the pieces of a last round.
@pytest.mark.parametrize("H, Sq, Sk, packed", [(2, 64, 700, False), (2, 64, 700, True), (40, 1296, 400, False), (20, 3500, 700, False)])
@pytest.mark.parametrize("kind", ["rising", "falling", "peak"])
def test_units_and_pieces_on_extreme_scores(H, Sq, Sk, packed, kind):
    q, k, v = _qkv(1, Sq, Sk, H, Sq + Sk)
    q[..., 0], k[..., 0] = 8.0, 0.0
    ramp = torch.linspace(0, 3000, Sk).to(torch.bfloat16)  # scores up to 2,100
    k[..., 0] = {"rising": ramp, "falling": ramp.flip(0), "peak": torch.eye(1, Sk)[0].roll(Sk // 2).to(torch.bfloat16) * 3000}[kind][:, None]
    kw = dict(cu_seqlens_q=torch.tensor([0, Sq], dtype=torch.int32, device=DEV), max_seqlen_q=Sq,
              cu_seqlens_k=torch.tensor([0, Sk], dtype=torch.int32, device=DEV)) if packed else {}
    out, lse = flash_attn_func(q.to(DEV), k.to(DEV), v.to(DEV), **kw)
    torch.cuda.synchronize()
    h, rows = [0, H - 1], sorted({0, Sq // 2, max(0, Sq - Sq % 256 - 8), max(0, Sq - Sq % 256 - 1), Sq - 2, Sq - 1})
    ref_out, ref_lse = sdpa_reference(q[:, rows][:, :, h], k[:, :, h], v[:, :, h])
    m = (out.cpu()[:, rows][:, :, h].float() - ref_out).abs().max().item()
    assert m <= 2e-2, m
    # scores of thousands: their fp32 sum over 128 products carries 2^-24 of it a term
    assert ((lse.cpu()[:, h][..., rows] - ref_lse).abs() <= 1e-3 + 2.0**-18 * ref_lse.abs()).all()


# A NaN in one query row, and in one key: NaN where the row or the key takes part
# and nowhere else, as from the tiles.
@pytest.mark.parametrize("H, Sq, Sk, row", [(2, 64, 300, 5), (40, 1296, 100, 1290)])
def test_nan_stays_in_its_rows(H, Sq, Sk, row):
    q, k, v = (x.to(DEV) for x in _qkv(1, Sq, Sk, H, 11))
    clean, _ = flash_attn_func(q, k, v)
    q[0, row, 1, 7] = float("nan")
    out, _ = flash_attn_func(q, k, v)
    bad = torch.zeros((1, Sq, H), dtype=torch.bool, device=DEV)
    bad[0, row, 1] = True
    assert torch.isnan(out[bad]).all() and torch.equal(out[~bad], clean[~bad])
    q[0, row, 1, 7], k[0, Sk // 2, 1, 3] = 0.0, float("nan")
    out, _ = flash_attn_func(q, k, v)
    assert torch.isnan(out[:, :, 1]).all() and torch.equal(out[:, :, 0], clean[:, :, 0])


# Queued last rounds over short key ranges (pieces of a few key tiles).
@pytest.mark.parametrize("H, Sq, Sk", [(20, 3500, 1500), (40, 2048, 2048), (70, 1024, 1300)])
def test_last_round_pieces_of_short_key_ranges(H, Sq, Sk):
    q, k, v = _qkv(1, Sq, Sk, H, Sk)
    out, lse = flash_attn_func(q.to(DEV), k.to(DEV), v.to(DEV))
    torch.cuda.synchronize()
    h = [0, H - 1]
    ref_out, ref_lse = sdpa_reference(q[:, :, h], k[:, :, h], v[:, :, h])
    assert_parity(out.cpu()[:, :, h], lse.cpu()[:, h], ref_out, ref_lse, f"{H}x{Sq}x{Sk}")


# Those tiles would otherwise hold their sums in fp32 to the one final rounding:
# their pieces' partial results do too, so the last tiles are as near the 64-bit
# result as in the launch that cuts nothing (a rounding of the partial results
# to bf16 raises the error by a quarter or more).
@pytest.mark.parametrize("H, Sq, Sk", [(20, 3500, 1500), (40, 2048, 2048), (70, 1024, 1300)])
def test_last_round_pieces_are_as_near_the_exact_result(H, Sq, Sk):
    q, k, v = _qkv(1, Sq, Sk, H, H + Sk)
    rows = slice(Sq - Sq % 256 - 256 * 2, Sq - Sq % 256)
    err = {}
    qh, kh, vh = (x[0, :, H - 1].double() for x in (q, k, v))
    exact = torch.softmax(qh[rows] @ kh.T * 128**-0.5, dim=-1) @ vh
    for split in (True, False):
        out, _ = flash_attn_func(q.to(DEV), k.to(DEV), v.to(DEV), split_tail=split)
        got = out[0, rows, H - 1].double().cpu()
        err[split] = ((got - exact).norm() / exact.norm()).item()
    assert err[True] <= 1.03 * err[False], err


# Persistent launches that order their segments by key length: more segments
# than a wave has lanes, empty ones first, last and in between, equal lengths,
# query and key lengths in different orders, and fewer tiles than CUs (0.9, 6.3,
# 5.5 and 5.9 rounds of tiles, which the planned list does not take). The same
# tiles as one workgroup each, so the same bits.
@pytest.mark.parametrize(
    "qlens, klens, H",
    [([0, 300, 0, 257, 700, 1, 0], None, 28), ([700 - 7 * i if i % 3 else 0 for i in range(90)], None, 12),
     ([256, 1000, 40, 600], [900, 64, 700, 1], 150), ([40] * 130 + [600] * 3, None, 16)],
)
def test_persistent_order_by_length(qlens, klens, H):
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert _varlen_workspace(qlens, H, klens) == 256
    own, klens = klens is not None, qlens if klens is None else klens
    q, k, v = _qkv(1, sum(qlens), sum(klens), H, sum(klens))
    cq, ck = (torch.tensor([0, *torch.tensor(x).cumsum(0).tolist()], dtype=torch.int32, device=DEV) for x in (qlens, klens))
    kw = dict(cu_seqlens_q=cq, cu_seqlens_k=ck if own else cq, max_seqlen_q=max(qlens))
    got = flash_attn_func(q.to(DEV), k.to(DEV), v.to(DEV), **kw)
    whole = flash_attn_func(q.to(DEV), k.to(DEV), v.to(DEV), split_tail=False, **kw)
    torch.cuda.synchronize()
    assert torch.equal(got[0], whole[0]) and torch.equal(got[1], whole[1])
    a, b = qlens[0] + qlens[1], klens[0] + klens[1]
    rows, keys = slice(qlens[0], a), slice(klens[0], b)
    ref_out, ref_lse = sdpa_reference(q[:, rows, :2], k[:, keys, :2], v[:, keys, :2])
    assert_parity(got[0][:, rows, :2].cpu(), got[1][:, :2, rows].cpu(), ref_out, ref_lse, "second segment")
