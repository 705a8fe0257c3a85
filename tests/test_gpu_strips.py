"""Strip length and workgroup size of the span attention forward: every choice gives the same bits."""
import pytest
import torch

import sparseattention_amd as sa
from sparseattention_amd import _lib
from sparseattention_amd.ops import functional as fn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture
def knobs():
    def set_knobs(sb, wpb):
        assert _lib.lib().hsa_attn_tile_tune(sb, wpb, -1, -1) == 0
    yield set_knobs
    assert _lib.lib().hsa_attn_tile_tune(0, 0, -1, -1) == 0


# automatic choices: four wavefronts instead of six, six with strips of two / four / eight, five, seven,
# eight where nothing divides, three at 128 channels, part heads, a sequence of one block, short strips
@pytest.mark.parametrize("case", [(5, 1024, 12, 64, 13), (4, 2048, 6, 64, 16), (3, 2048, 12, 64, 16), (8, 2048, 12, 64, 16),
                                  (2, 8192, 10, 64, 16), (6, 2048, 7, 64, 16), (5, 1024, 11, 64, 24), (3, 4096, 6, 128, 16),
                                  (3, 2048, 8, 96, 16), (1, 16, 4, 32, 5), (2, 64, 3, 64, 40), (1, 128, 1, 64, 8)])
@pytest.mark.parametrize("causal", [True, False])
def test_strip_choice_same_bits(case, causal, knobs):
    B, N, H, D, R = case
    g = torch.Generator(device=DEV).manual_seed(N + H)
    mk = lambda n: torch.randn(B, n, H, D, generator=g, device=DEV).to(torch.bfloat16)
    q, k, v = mk(N), mk(2 * N - 1), mk(2 * N - 1)
    t = sa.build_tree_topology(N, causal, device=DEV)
    mask = t["forward_mask"] if causal else None
    run = lambda: fn.attention_forward(q, k, v, t["forward_idx"], mask, R)
    auto = run()
    gather = fn.attention_forward(q, k, v, t["forward_idx"], mask, R, algo="gather")
    # weights rounded to 8 bits once: 2^-9 of sums of size 1 to 4, as in the other tests of this kernel
    assert (auto.float() - gather.float()).abs().max() <= 2e-2
    for sb in (1, 2, 4, 8):
        for wpb in (0, 4):
            knobs(sb, wpb)
            assert torch.equal(run(), auto), (sb, wpb)
    knobs(0, 0)
