"""The sampler's moves connect the space: from the default config of a shape every compiled config that is legal there
is reached, also where the default is a block 192 or 16 wide (CPU only)."""

from collections import deque

import pytest

import kernel_library as kl
from autotune.search import FAMILY_VARIANTS, Atom, IllegalMove, TileMDP
from kernel_library.config import TileConfig

# Shapes whose defaults are 192 wide (both matmuls), powers of two, split, non-temporal, and 16, 32 and 64 wide (fp32).
SHAPES = [("matmul_lhsT_rhs", (2056, 4032, 8520)), ("matmul_lhsT_rhs", (2048, 2048, 2048)),
          ("matmul_lhsT_rhs", (16, 4096, 4096)), ("matmul_lhs_rhs", (1000, 5000, 4104)),
          ("matmul_lhs_rhs", (64, 4096, 1024)), ("rmsnorm_matmul", (8, 4096, 4096)),
          ("matmul_lhsT_rhs_f32", (256, 512, 512)), ("matmul_lhsT_rhs_f32", (1000, 1501, 777)),
          ("matmul_lhsT_rhs_f32", (4096, 4096, 4096))]


def _closure(mdp):
    root = mdp.reset()
    seen, q = {root.name}, deque([root])
    while q:
        s = q.popleft()
        for a in mdp.atoms:
            try:
                n = mdp.step(s, a)
            except IllegalMove:
                continue
            if n.name not in seen:
                seen.add(n.name)
                q.append(n)
    return seen


@pytest.mark.parametrize("fam,shape", SHAPES)
def test_every_compiled_config_is_reached(fam, shape):
    seen = _closure(TileMDP(fam, *shape, prebuilt_only=True))
    legal = [c for c in kl.compiled_configs(fam) if c.variant in FAMILY_VARIANTS[fam] and kl.check(fam, c, *shape)[0] == 0]
    assert legal
    assert not [c.name for c in legal if c.name not in seen]


@pytest.mark.parametrize("prebuilt_only", [True, False])
def test_192_is_left_and_reached(prebuilt_only):
    mdp = TileMDP("matmul_lhs_rhs", 1000, 5000, 4104, prebuilt_only)
    wide, base = (TileConfig.from_name(f"bm128_bn{n}_bk32_w4_s4_v1") for n in (192, 128))
    assert mdp.step(base, Atom("block_n", "wider")) == wide
    assert mdp.step(wide, Atom("block_n", "narrower")) == base
    assert mdp.step(wide, Atom("block_n", "wider")).block_n == 256
    with pytest.raises(IllegalMove):
        mdp.step(base, Atom("block_n", "narrower"))  # what halving reaches is left to it
    with pytest.raises(IllegalMove):
        mdp.step(TileConfig(96, 128, 32, 4, 4, variant=1), Atom("block_m", "wider"))


def test_a_variant_move_lands_on_the_nearest_compiled_config():
    mdp = TileMDP("matmul_lhsT_rhs_f32", 4096, 4096, 4096, prebuilt_only=True)
    s = TileConfig.from_name("bm64_bn64_bk16_w4_s2_v3")
    assert mdp.step(s, Atom("variant", "=1")) == TileConfig.from_name("bm64_bn64_bk16_w4_s1_v1")
    assert mdp.step(s, Atom("variant", "=0")) == TileConfig.from_name("bm64_bn64_bk16_w4_s1")
    small = TileConfig.from_name("bm16_bn16_bk32_w4_s2_v3")
    assert mdp.step(small, Atom("waves", "x2")).waves == 8
    assert mdp.step(small, Atom("block_m", "x2")).block_m == 32
