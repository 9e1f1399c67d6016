"""GPU: the matrix-core router (from 20480 logits on) bit for bit against the oracle's fixed reduction
order, at rows below, on and past the 512-column steps, expert and token counts around the 16 x 16
tiles, every pair of row types; and the normalised rows it writes, through a forward."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,E,n,xdt,wdt,norm,gamma", [
    (8, 16, 1280, "f32", "f32", True, False),
    (24, 256, 81, "bf16", "bf16", True, True),
    (504, 17, 1205, "f32", "bf16", True, False),
    (512, 33, 640, "bf16", "f32", False, False),
    (520, 130, 159, "bf16", "bf16", False, False),
    (1032, 31, 673, "f32", "f32", True, True),
    (3080, 100, 209, "bf16", "bf16", True, True),
    (4104, 64, 321, "f32", "bf16", True, False),
])
def test_route_matrix_core_bitexact(oracle, D, E, n, xdt, wdt, norm, gamma):
    from burnext_amd import moe, synth
    assert n * E >= 20480
    print(f"router case D={D} E={E} n={n} x {xdt} w {wdt} norm={norm} gamma={gamma}", flush=True)
    L = synth.make_layer(D, 32, E, 3, seed=7, dtype=wdt, with_gamma=gamma)
    x = synth.make_tokens(n, D, seed=8, dtype=xdt)
    x[::7] *= 300.0  # rows of other magnitudes
    x = synth.round_bf16(x) if xdt == "bf16" else x
    layer = moe.MoeLayer(L)
    idx, _, lg = layer.route(moe.to_device_x(x, xdt), flags=1 if norm else 0)
    ref = oracle.route_logits(x, L.router_w_f32, L.router_b_f32, L.gamma_f32, L.rms_eps, norm)
    got = lg.cpu().numpy()
    layer.close()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), np.max(np.abs(got - ref))
    assert np.array_equal(idx.cpu().numpy(), oracle.topk_softmax(ref, 3)[0])


@pytest.mark.parametrize("D,E,n,dtype,flags", [(40, 128, 161, "f32", 3), (520, 40, 513, "bf16", 3), (520, 40, 1100, "f32", 2),
                                               (200, 200, 103, "bf16", 1)])
def test_forward_after_matrix_core_router(oracle, D, E, n, dtype, flags):
    """The rows the router writes for the expert tiles (f32, bf16) and the grouped GEMM (two terms)."""
    from burnext_amd import moe, synth
    print(f"router rows case D={D} E={E} n={n} {dtype} flags={flags}", flush=True)
    L = synth.make_layer(D, 96, E, 2, seed=9, dtype=dtype, with_gamma=True)
    x = synth.make_tokens(n, D, seed=10, dtype=dtype)
    layer = moe.MoeLayer(L)
    y = layer.forward(moe.to_device_x(x, dtype), flags=flags).float().cpu().numpy()
    layer.close()
    y_ref, _, _ = oracle.moe_forward(L, x, apply_rmsnorm=bool(flags & 1), add_residual=bool(flags & 2))
    res = x if flags & 2 else 0
    assert oracle.max_abs_rel(y - res, y_ref - res) <= (1e-4 if dtype == "f32" else 2e-2)
