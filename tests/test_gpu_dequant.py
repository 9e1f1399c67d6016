"""GPU: the dequant hook over widths, sizes and alignments of every dispatch branch, bit for bit
against the oracle (cols a multiple of 8, even, odd; spans that end inside a store; source and
output at odd addresses)."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out_dtype", ["f32", "bf16"])
@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 7), (3, 8), (5, 2), (37, 30), (33, 31), (9, 32), (65, 33), (70, 1000),
                                       (1, 8), (1, 9), (2, 11), (5, 15), (301, 129), (11, 2818), (7, 2817), (13, 4104)])
def test_dequant_shapes(oracle, rows, cols, out_dtype):
    from burnext_amd import _native as N
    from burnext_amd import moe
    rng = np.random.default_rng(rows * 10007 + cols)
    experts, ue8 = 2, 14
    bpr, gpr = (cols + 1) // 2, (cols + 31) // 32
    blocks = rng.integers(0, 256, (experts * rows, bpr), dtype=np.uint8)
    scales = rng.integers(0, 255, (experts * rows, gpr), dtype=np.uint8)  # stored: true exponent + 14 mod 256
    scales[(scales.astype(np.int32) - ue8) & 255 == 255] = 20
    ref = oracle.dequant_matrix(blocks, scales, experts * rows, cols, ue8)
    desc = moe.QuantLinearMxFp4Desc.for_matrix(experts, rows, cols, ue8).c()
    el, code = (4, N.BURNEXT_F32) if out_dtype == "f32" else (2, N.BURNEXT_BF16)
    n = experts * rows * cols
    for src_off, out_off in ((0, 0), (1, 0), (0, el), (3, el)):  # bytes past an aligned address
        src = torch.zeros(blocks.size + 16, dtype=torch.uint8, device="cuda")
        src[src_off:src_off + blocks.size] = torch.from_numpy(blocks.ravel()).cuda()
        sc = torch.from_numpy(scales.ravel()).cuda()
        out = torch.full((n * el + 64,), 0xA5, dtype=torch.uint8, device="cuda")
        N.check(N.lib().burnext_mxfp4_dequant(ctypes.byref(desc), ctypes.c_void_p(src.data_ptr() + src_off),
                                              ctypes.c_void_p(sc.data_ptr()), ctypes.c_void_p(out.data_ptr() + out_off),
                                              code, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        host = out.cpu().numpy()
        got = host[out_off:out_off + n * el].view(np.uint32 if el == 4 else np.uint16)
        want = ref.ravel().view(np.uint32)
        assert np.array_equal(got, want if el == 4 else (want >> 16).astype(np.uint16)), (src_off, out_off)
        assert (host[:out_off] == 0xA5).all() and (host[out_off + n * el:] == 0xA5).all()  # nothing beside it
