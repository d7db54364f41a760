"""Edges of the attention kernel's tile: every count of key tiles from one to
nine (odd counts padded to even ones, pipelines shorter than their LDS ring)
against last query tiles that leave zero to seven waves without a row.
Same tolerance as the other attention tests."""

from __future__ import annotations

import pytest
import torch

from h3_flash_amd import flash_attn_func
from oracle.attention import sdpa_reference
from tests.test_gpu_attention import assert_parity

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
