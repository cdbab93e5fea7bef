"""The weight gradient's tile-to-tile pipeline (smoe_gemm_wgrad.hip): a
workgroup that walks several tiles loads each one's first row group during
the epilogue of the tile before it.  A call over all experts, more tiles than
workgroups, must give the bytes of one call per expert (at most one tile per
workgroup, nothing loaded ahead) in every output mode, with experts that have
no rows, one row group, and more groups than one scale chunk, and with tiles
at both edges of dW.  One expert's gradient is held to the exact sum of the
dequantised operands."""
import pytest
import torch

from smoe import ops
from smoe import workloads as W

pytestmark = pytest.mark.gpu

COUNTS = [0, 5, 128, 129, 0, 0, 300, 1024, 1025, 1, 700, 0, 127, 2200, 256, 0] * 3


@pytest.mark.parametrize("scale", ["fp32", "pow2"])
@pytest.mark.parametrize("N,K", [(784, 528), (512, 768), (2048, 256)])
def test_tiles_loaded_ahead_equal_single_tiles(dev, N, K, scale):
    print("[wgrad ring]", N, K, scale, flush=True)
    E, R = len(COUNTS), sum(COUNTS)
    assert E * -(-N // 256) * -(-K // 256) > 256  # several tiles a workgroup
    off = W.offsets_from_counts(COUNTS, dev)
    dy, x = W.tokens(R, N, device=dev, seed=N), W.tokens(R, K, device=dev, seed=K + 1)
    aq, as_, pad, ld = ops.quant_cols(dy, off, col_scale=scale)
    bq, bs, _, _ = ops.quant_cols(x, off, col_scale=scale)
    base = W.tokens(E * N, K, device=dev, seed=5).view(E, N, K)
    for dt in (torch.float32, torch.bfloat16):
        for acc in (False, True):
            start = base.to(dt) if acc else torch.full((E, N, K), 3.0, dtype=dt, device=dev)
            whole, each = start.clone(), start.clone()
            args = dict(accumulate=acc, e8m0=scale == "pow2")
            ops.grouped_gemm_fp8_wgrad(aq, as_, bq, bs, pad, ld, out=whole, **args)
            for e in range(E):
                ops.grouped_gemm_fp8_wgrad(aq, as_, bq, bs, pad[e:e + 2].clone(), ld, out=each[e:e + 1], **args)
            as_int = torch.int32 if dt is torch.float32 else torch.int16
            assert torch.equal(whole.view(as_int), each.view(as_int)), (dt, acc)
            if dt is torch.float32 and not acc:
                e = COUNTS.index(1025)
                p0, p1 = int(pad[e]), int(pad[e + 1])
                deq = lambda q, s: (q.view(torch.float8_e4m3fn)[:, p0:p1].double()
                                    * s[:, p0 // 128:p1 // 128].double().repeat_interleave(128, 1))
                a, b = deq(aq, as_), deq(bq, bs)
                # fp32 sums of 9 row groups: far below 2^-16 of the summed magnitudes
                bound = (a.abs() @ b.abs().t()) * 2.0 ** -16
                assert ((whole[e].double() - a @ b.t()).abs() <= bound + 1e-30).all()
