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


@pytest.mark.parametrize("T", [1, 65])
def test_forward_samples(cuda_device, T):
    """One table (walked) and three blocks of tables (a workgroup a sample)."""
    B, I, O, dgs = (1 << 26) + 77, 2, 1, 32
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(T)
    x = torch.randn(B * I, device=dev, generator=gen)
    W = torch.randn(T * 2, device=dev, generator=gen)
    anchors = anchors_of(T, 1, I, dev, T)
    out = torch.zeros(B, device=dev)
    idx = torch.empty(B * T, dtype=torch.int32, device=dev)
    print(f"[launch] forward B={B} T={T}", flush=True)
    make_dm(I, O, T, 1, bgs=dgs).forward_step(W, B, x, anchors, out, idx)
    a = anchors.view(T, 2).tolist()
    want = torch.zeros(B, device=dev)
    xs = x.view(B, I)
    for t0 in range(0, T, dgs):
        block = torch.zeros(B, dtype=torch.float64, device=dev)
        for t in range(t0, min(t0 + dgs, T)):
            bit = xs[:, a[t][0]] > xs[:, a[t][1]]
            assert torch.equal(idx.view(B, T)[:, t].bool(), bit)
            block += torch.where(bit, W[2 * t + 1], W[2 * t]).double()
        want += block.float()
    assert torch.equal(out, want)


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


def test_input_gradient_items(cuda_device):
    """2^27 items of 32768 outputs, in 16 chunks: the gradients of some samples
    against the same call over these samples alone, which one launch holds."""
    B, I, T, Nc, O = 1 << 15, 2, 1 << 12, 1, 1 << 15
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(9)
    g = torch.randn(B, O, device=dev, generator=gen)
    W = torch.randn(T, 2, O, device=dev, generator=gen)
    x = torch.randn(B * I, device=dev, generator=gen)
    anchors = torch.tensor([0, 1], dtype=torch.int32, device=dev).repeat(T)
    dm = make_dm(I, O, T, Nc)
    idx, mi = (torch.empty(B * T, dtype=torch.int32, device=dev) for _ in range(2))
    md = torch.empty(B * T, device=dev)
    small = make_dm(I, 4, T, Nc)
    small.forward_step(torch.zeros(T * 2 * 4, device=dev), B, x, anchors, torch.zeros(B * 4, device=dev), idx,
                       0.0, None, md, mi)
    some = [0, 1, 7, 8, 4095, B // 2 + 3, B - 1]
    few = torch.tensor(some, device=dev)
    pick = lambda v: v.view(B, T)[few].reshape(-1).contiguous()
    dm.forward_step(W.view(-1), 1, x[:I].contiguous(), anchors, torch.zeros(O, device=dev),
                    torch.empty(T, dtype=torch.int32, device=dev))
    want = torch.zeros(len(some) * I, device=dev)
    dm.backward_backprop(W.view(-1), len(some), g[few].reshape(-1), anchors, pick(idx), pick(md), pick(mi), want,
                         -1.0, None, None)
    xg = torch.zeros(B * I, device=dev)
    print(f"[launch] input gradient B={B} T={T} O={O}", flush=True)
    dm.backward_backprop(W.view(-1), B, g.view(-1), anchors, idx, md, mi, xg, -1.0, None, None)
    got, want = xg.view(B, I)[few].double(), want.view(-1, I).double()
    # fp32 additions of 16 T terms in any order: 16 T 2^-24 of the terms' magnitudes, that is
    # the slope of at most 0.5 times the chunks' dots, which together are about four times
    # the whole dot's
    diff = (W[:, 1] - W[:, 0]).double()
    exact = diff @ g[few].double().T  # [T][samples]
    bound = 2 * 16 * T * 2.0 ** -24 * exact.abs().sum(0) + 1e-6 * want.abs().max(1).values
    assert torch.all((got - want).abs().max(1).values <= bound)
    assert torch.all(want.abs().max(1).values > 0)
