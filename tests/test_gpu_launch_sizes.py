"""Calls whose work takes more threads than one launch holds (2^32): large
batches, many table rows, many (sample, table) items.  References in torch on
the device, over all samples where they are cheap."""
import pytest
import torch

from test_gpu_fc import make_dm

pytestmark = pytest.mark.gpu


def anchors_of(T, Nc, I, dev, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.stack([torch.randperm(I, generator=g)[:2] for _ in range(T * Nc)]).to(torch.int32).flatten().to(dev)


def test_weight_gradient_rows(cuda_device):
    """2^28 table rows."""
    B, I, T, Nc, O = 2, 32, 1 << 16, 12, 1
    E = 1 << Nc
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(5)
    g = torch.randn(B * O, device=dev, generator=gen)
    idx = torch.randint(0, E, (B * T,), device=dev, dtype=torch.int32, generator=gen)
    md, mi = torch.ones(B * T, device=dev), torch.zeros(B * T, dtype=torch.int32, device=dev)
    W = torch.zeros(T * E * O, device=dev)
    x = torch.randn(B * I, device=dev, generator=gen)
    anchors = anchors_of(T, Nc, I, dev, 5)
    dm = make_dm(I, O, T, Nc)
    dm.forward_step(W, B, x, anchors, torch.zeros(B * O, device=dev), torch.empty_like(idx))
    wg = torch.full((T * E * O,), float("nan"), device=dev)
    xg = torch.zeros(B * I, device=dev)
    print(f"[launch] weight gradient T={T} E={E}", flush=True)
    dm.backward_backprop(W, B, g, anchors, idx, md, mi, xg, -1.0, wg, None, overwrite_weights_gradients=True)
    want = torch.zeros(T, E, device=dev)
    for b in range(B):
        rows = idx.view(B, T)[b].long()
        want[torch.arange(T, device=dev), rows] += g[b]
    assert torch.equal(wg.view(T, E), want)
