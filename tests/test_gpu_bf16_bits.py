"""Bits of the bf16 variant's results. Layers amplify a last-bit change of one before
them (to 5e-3 of a pair's outputs at full depth), so the order of the sums, the
K ranges and the rounding of the rotary embedding are part of the result: the
checksums below are those of the kernels that these launches ran on at first
(128 x 128 tiles cut in K below 432 of them, 256 x 128 tiles from 512 on), at
launches of each kind."""
import zlib

import pytest

import gsplat_hip as G
from gpu_util import case, dev, empty, host, stream

pytestmark = pytest.mark.gpu

CONFIG = dict(patch=16, enc_dim=256, enc_depth=2, enc_heads=4, enc_mlp=1024, dec_dim=256, dec_depth=2,
              dec_heads=4, dec_mlp=768, dpt_feat=64, dpt_dims=[32, 64, 96, 128], dpt_hooks=[0, 1, 2, 2],
              head_mid=32, lf_hidden=512, desc_dim=24, precision=1)


def pair_checksums(G, gh, gw, B):
    cfg = G.default_config(img_h=16 * gh, img_w=16 * gw, **CONFIG)
    H, W = cfg.img_h, cfg.img_w
    m = G.Mastr(cfg, B)
    m.init_seeded(3, 0.02, 0.1)
    img = [dev(G.seed_uniform(5, f"view{v}", B * 3 * H * W).reshape(B, 3, H, W)) for v in (1, 2)]
    out = [empty(B, H, W, c) for _ in (1, 2) for c in (3, 1, 24)]
    m.pair(*img, B, *out, stream())
    sums = [zlib.crc32(host(t).tobytes()) for t in out]
    m.close()
    return sums


@pytest.mark.parametrize("gh,gw,B,want", [
    (24, 32, 1, [1422295998, 2484651131, 4188531315, 3029966134, 4121427180, 4116017546]),
    (10, 14, 3, [445955100, 3989443969, 1321205750, 3795348864, 2242763045, 3235586239]),
    (32, 32, 8, [569314930, 796536553, 326184468, 2363269199, 1384152564, 2291890367]),
    (32, 32, 16, [2095336937, 2000849046, 1549416659, 3646738341, 3572239314, 250354727]),
])
def test_bf16_pair_bits(gh, gw, B, want):
    case(f"bf16 pair bits {gh}x{gw} B={B}")
    assert pair_checksums(G, gh, gw, B) == want
