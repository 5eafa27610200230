"""Pair sizes at and around the kernels' tile edges, down to one token.

The kernels tile pairs in 16-, 64- and 128-row blocks, keys in 32-key blocks
padded to 64, and the contraction in 128- and 256-wide tiles (rows padded to
128).  Every module is compared with the oracle at N on either side of those
edges, including N = 1 and 2 (a single pair row, a single key block mostly
padding), in fp32 arithmetic (max-abs <= 1e-4) and bf16 arithmetic under
autocast with an fp32 z (the bench's mode; the bf16 tier on the update).
The token mask pads the last token where N > 2, so every size also has a
fully masked row and column.
"""

import pytest
import torch

from helpers import assert_bf16, assert_fp32, params_of, say, seeded, token_pair_mask
from oracle import reference as ref
from opendde_amd.pairformer import PairformerBlock
from opendde_amd.triangular import (TriangleAttention, TriangleMultiplicationIncoming,
                                    TriangleMultiplicationOutgoing)

pytestmark = pytest.mark.gpu
DEV = "cuda"
SIZES = [1, 2, 3, 15, 16, 33, 63, 65, 127, 129, 255, 257]


def _inputs(n, seed):
    z = torch.randn(n, n, 128, generator=torch.Generator().manual_seed(seed))
    mask = token_pair_mask(n, 1 if n > 2 else 0)
    return z, mask


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("kind", ["att_start", "att_end", "mul_out", "mul_in"])
def test_module_sizes(n, kind):
    say(f"[gpu] size sweep {kind} n={n}")
    z, mask = _inputs(n, 1000 + n)
    if kind.startswith("att"):
        mod = seeded(TriangleAttention(128, 32, 4, starting=kind == "att_start"), n, 0.1)
        exp = ref.triangle_attention(z, mask, params_of(mod), 4, starting=kind == "att_start")
        run = lambda m, x: m(x, mask.to(DEV), triangle_attention="hip")  # noqa: E731
    else:
        mod = seeded((TriangleMultiplicationOutgoing if kind == "mul_out"
                      else TriangleMultiplicationIncoming)(128, 128), n, 0.1)
        exp = ref.triangle_multiplication(z, mask, params_of(mod), outgoing=kind == "mul_out")
        run = lambda m, x: m(x, mask.to(DEV), triangle_multiplicative="hip")  # noqa: E731
    mod = mod.to(DEV)
    with torch.no_grad():
        got = run(mod, z.to(DEV))
        assert_fp32(got, exp, f"{kind} n={n}")
        with torch.autocast("cuda", dtype=torch.bfloat16):
            got16 = run(mod, z.to(DEV))
    assert got16.dtype == torch.float32
    assert_bf16(got16, exp, f"{kind} bf16 n={n}")


@pytest.mark.parametrize("n", [1, 2, 17, 65, 129])
def test_block_sizes(n):
    """A whole block (c_s 384, 16 single heads) in fp32 and in the bench's mode."""
    say(f"[gpu] size sweep block n={n}")
    z, mask = _inputs(n, 2000 + n)
    s = torch.randn(n, 384, generator=torch.Generator().manual_seed(3000 + n))
    blk = seeded(PairformerBlock(n_heads=16, c_z=128, c_s=384), 4000 + n, 0.05)
    se, ze = ref.pairformer_block(s, z, mask, params_of(blk), no_heads_pair=4, n_heads=16)
    blk = blk.to(DEV)
    with torch.no_grad():
        sg, zg = blk(s.to(DEV), z.to(DEV), mask.to(DEV), triangle_multiplicative="hip",
                     triangle_attention="hip", inplace_safe=True)
        assert_fp32(zg, ze, f"block n={n} z")
        assert_fp32(sg, se, f"block n={n} s")
        with torch.autocast("cuda", dtype=torch.bfloat16):
            sb, zb = blk(s.to(DEV), z.to(DEV), mask.to(DEV), triangle_multiplicative="hip",
                         triangle_attention="hip", inplace_safe=True)
    assert_bf16(zb - z.to(DEV), ze - z, f"block bf16 n={n} z update")
    assert_bf16(sb - s.to(DEV), se - s, f"block bf16 n={n} s update")


@pytest.mark.parametrize("n,c", [(66, 64), (129, 64), (191, 64), (256, 64), (319, 64), (384, 64),
                                 (385, 64), (450, 64), (513, 64), (577, 64), (190, 384),
                                 (321, 384), (449, 384)])
@pytest.mark.parametrize("outgoing", [True, False])
def test_multiplication_plane_sizes(n, c, outgoing):
    """Planes rounded up to 64 and every tile of the contraction, with whole
    and partial last tiles (Np 128 to 640), over a workspace of NaN: rows that
    no projection writes must not reach the result."""
    say(f"[gpu] plane sizes n={n} c={c} out={outgoing}")
    z = torch.randn(n, n, c, generator=torch.Generator().manual_seed(n + c))
    mask = token_pair_mask(n, 2)
    cls = TriangleMultiplicationOutgoing if outgoing else TriangleMultiplicationIncoming
    mod = seeded(cls(c, c), n, 0.1 if c == 64 else 0.05)
    exp = ref.triangle_multiplication(z, mask, params_of(mod), outgoing=outgoing)
    mod, zd, md = mod.to(DEV), z.to(DEV), mask.to(DEV)

    def run(autocast):
        torch.cuda.empty_cache()
        dirty = torch.full((1 << 28,), float("nan"), device=DEV)
        del dirty  # its block serves the call's workspace
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            return mod(zd, md, triangle_multiplicative="hip")

    assert_bf16(run(True), exp, f"planes bf16 n={n} c={c} out={outgoing}")
    if c == 64:
        assert_fp32(run(False), exp, f"planes n={n} c={c} out={outgoing}")


@pytest.mark.parametrize("rows", [4095, 4097, 16417, 90001])
@pytest.mark.parametrize("inplace", [False, True])
def test_transition_rows_c384(rows, inplace):
    """The wide transition's forms by row count (tiles up to 4096 rows, then 32
    and from 90001 rows 64 rows a wave), with rows that end inside a wave."""
    from opendde_amd.pairformer import Transition
    say(f"[gpu] transition rows={rows} inplace={inplace}")
    mod = seeded(Transition(384, 4), rows, 0.04)
    x = torch.randn(rows, 384, generator=torch.Generator().manual_seed(rows))
    exp = ref.transition(x, params_of(mod))
    mod, xg = mod.to(DEV), x.to(DEV)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        got = mod.hip_apply(xg, out=xg, add_residual=True) if inplace else mod.hip_apply(xg)
    assert_bf16(got.cpu() - x if inplace else got, exp, f"transition rows={rows} inplace={inplace}")


@pytest.mark.parametrize("n", [96, 111, 112, 160, 192, 193])
@pytest.mark.parametrize("tf32", [False, True])
@pytest.mark.parametrize("c", [64, 128])
def test_staged_f32_sizes(n, tf32, c):
    """The fp32 and three-part kernels with weights staged in LDS, one and two
    rows per workgroup, on either side of their sizes, in place."""
    say(f"[gpu] staged f32 n={n} tf32={tf32} c={c}")
    z = torch.randn(n, n, c, generator=torch.Generator().manual_seed(n + c))
    mask = token_pair_mask(n, 3)
    att = seeded(TriangleAttention(c, 32, c // 32), n, 0.1)
    mul = seeded(TriangleMultiplicationIncoming(c, c), n, 0.1)
    ea = ref.triangle_attention(z, mask, params_of(att), c // 32)
    em = ref.triangle_multiplication(z, mask, params_of(mul), outgoing=False)
    old = torch.backends.cuda.matmul.allow_tf32
    torch.backends.cuda.matmul.allow_tf32 = tf32
    try:
        with torch.no_grad():
            for mod, exp, what in ((att, ea, "attention"), (mul, em, "multiplication")):
                zd = z.to(DEV)
                got = mod.to(DEV).hip_apply(zd, mask.to(DEV), out=zd, add_residual=True)
                assert got.data_ptr() == zd.data_ptr()
                assert_fp32(zd, z + exp, f"staged {what} n={n} tf32={tf32} c={c}")
    finally:
        torch.backends.cuda.matmul.allow_tf32 = old


@pytest.mark.parametrize("rows", [4096, 6655, 6656, 9217, 16384, 16385])
@pytest.mark.parametrize("tf32", [False, True])
@pytest.mark.parametrize("c", [64, 128])
def test_transition_f32_staged_rows(rows, tf32, c):
    """The fp32 transition's forms on either side of their row counts: weight
    fragments, 64 rows (in two hidden halves for true fp32) and 128 rows."""
    from opendde_amd.pairformer import Transition
    say(f"[gpu] transition f32 rows={rows} tf32={tf32} c={c}")
    x = torch.randn(rows, c, generator=torch.Generator().manual_seed(rows + c))
    mod = seeded(Transition(c, 4), 11, 0.07 * (128 / c) ** 0.5)
    exp = ref.transition(x, params_of(mod))
    old = torch.backends.cuda.matmul.allow_tf32
    torch.backends.cuda.matmul.allow_tf32 = tf32
    try:
        xg = x.to(DEV)
        with torch.no_grad():
            mod.to(DEV).hip_apply(xg, out=xg, add_residual=True)
        assert_fp32(xg, x + exp, f"transition f32 rows={rows} tf32={tf32} c={c}")
    finally:
        torch.backends.cuda.matmul.allow_tf32 = old
