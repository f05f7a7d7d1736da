"""The forms that attention kernels get for a launch's size, seen in the emitted parameters (no GPU needed)."""
import pytest

from test_gemm_forms import defines


@pytest.mark.parametrize("heads,s,br,pair", [(112, 512, 64, 1), (32, 2048, 64, 1), (90, 384, 64, 1), (48, 1024, 64, 1), (80, 448, 64, 0), (40, 1344, 64, 0),
                                             (100, 576, 128, 0), (80, 600, 128, 0), (112, 353, 128, 0), (64, 777, 128, 0), (32, 1024, 128, 0), (256, 640, 128, 0)])
def test_fp32_attention_under_the_mask_halves_its_query_tiles_in_pairs(heads, s, br, pair):
    """Launches of 256 to 512 workgroups of 128 queries: halves that pair up, or an odd number of halves that fill the part once and
    two thirds; never with a last tile partly filled, nor on fewer or more workgroups."""
    d = defines("fmha_f32", B=1, H=heads, S=s, D=128, CAUSAL=1, SCALE=0.1, FILL=1)
    assert int(d["FF_WAVES"]) * 32 == br and (br == 128 or d["FF_PAIR"] == str(pair)), d
    d = defines("fmha_f32", B=1, H=heads, S=s, D=128, CAUSAL=1, SCALE=0.1)
    assert d["FF_WAVES"] == "4"


@pytest.mark.parametrize("heads,s,d,br,pair", [(60, 1024, 128, 256, 0), (80, 768, 128, 256, 0), (64, 600, 128, 256, 0), (200, 256, 128, 256, 0),
                                               (16, 2048, 128, 128, 0), (32, 2048, 128, 128, 2), (60, 1024, 64, 128, 0), (32, 2048, 64, 128, 2),
                                               (300, 1024, 128, 256, 2), (64, 333, 128, 128, 0), (24, 1608, 96, 128, 0)])
def test_masked_16_bit_attention_on_small_launches(heads, s, d, br, pair):
    """Queries per workgroup and pairs of query tiles by how many workgroups the launch has: one round of 256
    queries by themselves at head dim 128 rather than almost two of 128."""
    d = defines("fmha_bf16", B=1, H=heads, S=s, D=d, CAUSAL=1, SCALE=0.1, FILL=1)
    assert (int(d["FA_BR"]), int(d["FA_PAIR"])) == (br, pair), d
