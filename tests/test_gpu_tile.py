"""GPU: the expert projections as tiles on bf16 MFMA (all batches but single tokens and those of the
grouped GEMM) against the oracle on every row: token tiles of 1..64 rows, row blocks and K-groups with
remainders, one and several tiles per expert.  Bars as the other forwards': f32 rows 1e-4 (two bf16
terms, 2^-17 per value), bf16 rows 2e-2."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = {"f32": 1e-4, "bf16": 2e-2}


@pytest.mark.parametrize("D,F,E,K,n,dtype,layout,flags", [
    (256, 256, 2, 2, 17, "f32", "interleaved", 3),     # the smallest batch: 17 tokens in both tiles
    (200, 100, 3, 2, 100, "f32", "halves", 3),         # partial K-groups on both sides, odd feature blocks
    (96, 72, 5, 3, 333, "f32", "interleaved", 1),      # one K-group, rows below a row block
    (256, 256, 1, 1, 129, "f32", "interleaved", 3),    # tiles of 64, 64 and 1 token
    (640, 1152, 8, 2, 250, "f32", "interleaved", 2),   # 5 and 9 K-groups
    (33, 40, 4, 2, 70, "f32", "interleaved", 3),       # D not a multiple of 4 or 8
    (2880, 2880, 32, 4, 130, "f32", "interleaved", 3),
    (256, 264, 4, 2, 33, "bf16", "interleaved", 3),    # 33 features past a row block
    (50, 31, 6, 2, 60, "bf16", "halves", 0),           # odd F: the last value of a row segment alone
    (2880, 2880, 128, 4, 63, "bf16", "interleaved", 3),
    (2880, 2880, 32, 4, 17, "bf16", "interleaved", 3),
    # the grouped GEMM at both sides of its first sizes and of its tiles of 2, 3 and 4 token columns
    (256, 256, 1, 1, 79, "bf16", "interleaved", 3),
    (256, 256, 1, 1, 96, "bf16", "interleaved", 3),
    (256, 256, 1, 1, 112, "bf16", "interleaved", 3),
    (640, 1152, 3, 1, 97, "bf16", "interleaved", 3),
    (2200, 520, 2, 2, 97, "bf16", "halves", 3),
    # decode sizes: one tile of up to 16 tokens per active expert
    (256, 256, 2, 2, 16, "f32", "interleaved", 3),     # full tiles
    (200, 100, 3, 3, 2, "bf16", "halves", 3),          # partial K-groups
    (33, 40, 40, 32, 16, "f32", "interleaved", 3),     # the most segment entries (16 x 32)
    (640, 1152, 256, 8, 7, "bf16", "interleaved", 1),  # the most experts
    (50, 31, 6, 2, 11, "f32", "interleaved", 0),
    (2880, 2880, 32, 4, 2, "f32", "interleaved", 3),
    (1024, 2048, 64, 16, 1, "bf16", "interleaved", 3), # one token: the GEMVs, without K-parts in gate_up
])
def test_forward_tiles_all_rows(oracle, D, F, E, K, n, dtype, layout, flags):
    from burnext_amd import moe, synth
    print(f"tile case D={D} F={F} E={E} K={K} n={n} {dtype} {layout} flags={flags}", flush=True)
    L = synth.make_layer(D, F, E, K, seed=41, dtype=dtype, gate_up_layout=layout, ue8_offset=14, with_gamma=True)
    x = synth.make_tokens(n, D, seed=42, dtype=dtype)
    layer = moe.MoeLayer(L)
    y = layer.forward(moe.to_device_x(x, dtype), flags=flags).float().cpu().numpy()
    layer.close()
    y_ref, _, _ = oracle.moe_forward(L, x, apply_rmsnorm=bool(flags & 1), add_residual=bool(flags & 2))
    res = x if flags & 2 else 0
    assert np.isfinite(y).all()
    assert oracle.max_abs_rel(y, y_ref) <= TOL[dtype] and oracle.max_abs_rel(y - res, y_ref - res) <= TOL[dtype]
