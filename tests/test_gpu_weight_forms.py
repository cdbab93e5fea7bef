"""One-launch weight forms against the launches they replace, byte for byte:
quantise + pack, and transpose + pack, on whole and edge 128x128 blocks (N and
K multiples of 16), both scale rules; the plain transpose against torch's."""
import pytest
import torch

from smoe import ops
from smoe import workloads as W

pytestmark = pytest.mark.gpu

u8 = lambda t: t.contiguous().view(torch.uint8)


@pytest.mark.parametrize("E,N,K", [(2, 256, 512), (3, 144, 1024), (1, 16, 528), (2, 1536, 2048), (1, 5760, 2880),
                                   (2, 512, 656)])
@pytest.mark.parametrize("scale", ["amax", "pow2"])
def test_one_launch_forms(dev, E, N, K, scale):
    print("[weights]", E, N, K, scale, flush=True)
    w = W.weights(E, N, K, device=dev, seed=N + K)
    w[0, :3] *= 50
    wq, ws = ops.quantize_weight_blockwise(w, scale=scale)
    q, s, p = ops.quantize_pack_weight(w, scale=scale)
    assert torch.equal(u8(q), u8(wq)) and torch.equal(s, ws)
    assert torch.equal(p.data, ops.pack_weight_fp8(wq).data)
    wqT, wsT = ops.transpose_blockwise(wq, ws, k=K)
    ref = torch.zeros((E, K, ops.pad128(N)), dtype=torch.uint8, device=dev)
    ref[:, :, :N] = u8(wq)[:, :, :K].transpose(1, 2)
    assert torch.equal(u8(wqT), ref) and torch.equal(wsT, ws.transpose(1, 2))
    if not ops._packable(K, ops.pad128(N)):
        with pytest.raises(ValueError):
            ops.transpose_blockwise(wq, ws, k=K, pack=True)
        return
    pT, sT = ops.transpose_blockwise(wq, ws, k=K, pack=True)
    assert torch.equal(pT.data, ops.pack_weight_fp8(wqT).data) and torch.equal(sT, wsT)


def test_quantise_and_pack_refuses_uncovered_shapes(dev):
    with pytest.raises(ValueError):
        ops.quantize_pack_weight(W.weights(1, 128, 256, device=dev))
