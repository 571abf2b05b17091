"""The flow network at sizes where its cost volumes run one, three and nine
displacement rows a block, with odd levels and more than one pair: a pair's
flows have the same bits alone and in a batch, and a level-6 flow agrees with
the float64 network."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("W,H", [(64, 64), (129, 65), (321, 190), (700, 450)])
def test_batched_pairs_equal_single_ones(cuda, dtype, W, H):
    import torch
    vsc = importlib.import_module("video-stream-consistency_amd")
    rng = np.random.default_rng(W + H)
    base = rng.integers(0, 256, (H // 8 + 3, W // 8 + 3, 4), dtype=np.uint8).repeat(8, 0).repeat(8, 1)
    frames = [torch.from_numpy(np.ascontiguousarray(base[k:k + H, k:k + W])).to(cuda) for k in range(3)]
    net = vsc.FlowNet(W, H, 1, dtype, seed=5, slots=3)
    for k in range(3):
        net.extract(frames[k], k)
    print(f"flow network {dtype} {W}x{H}", flush=True)
    both = [x.clone() for x in net.flow([(1, 2), (1, 0)])]
    alone = [net.flow([p])[0].clone() for p in ((1, 2), (1, 0))]
    for a, b in zip(both, alone):
        assert torch.isfinite(a).all() and torch.equal(a, b)
    net.close()


@pytest.mark.parametrize("W,H", [(130, 70), (700, 450)])
def test_level6_flow_against_float64(cuda, W, H):
    import torch
    from oracle import pwcnet_light as pw
    vsc = importlib.import_module("video-stream-consistency_amd")
    rng = np.random.default_rng(W)
    base = rng.integers(0, 256, (H // 8 + 3, W // 8 + 3, 4), dtype=np.uint8).repeat(8, 0).repeat(8, 1)
    im = [np.ascontiguousarray(base[k:k + H, k:k + W]) for k in (0, 2)]
    net = vsc.FlowNet(W, H, 1, "f32", seed=3, slots=2)
    for k in range(2):
        net.extract(torch.from_numpy(im[k]).to(cuda), k)
    net.flow([(0, 1)])
    got = net.intermediate(1, 6).cpu().numpy()
    P = pw.unpack_params(net.params())
    fa, fb = (pw.extractor(P, pw.preprocess(x, 1)[0]) for x in im)
    ref = pw.decoder(P, 6, fa[5], fb[5])[0][0].permute(1, 2, 0).numpy()
    # the tolerance of the library's own smoke check of this level
    assert float(np.max(np.abs(got - ref)) / (np.max(np.abs(ref)) + 1e-3)) < 2e-5
    net.close()
