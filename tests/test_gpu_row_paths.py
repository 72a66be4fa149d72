"""GPU parity of the gathered-row kernels of the fully connected path (small
batches, odd output counts, many rows a table) against the CPU oracle, at the
edges of their units: 32-output blocks, 16-byte pieces, samples and tables a
step, and rows that end inside a piece."""
import numpy as np
import pytest
import torch

from test_gpu_fc import make_dm, make_inputs, run_fc, xg_close

pytestmark = pytest.mark.gpu


# B, T, Nc, O: a lone sample; one output; a block and one output more or less;
# sample groups and tables that are not whole; more blocks than lanes (two
# chunks); 512 rows a table; past the direct pushes (many tables on 48 inputs and B * T
# > 2^14), also with rows of two and three chunks, odd and even, and of exactly one
@pytest.mark.parametrize("int_rescaler", [None, 0.5])
@pytest.mark.parametrize("B,T,Nc,O", [(1, 70, 4, 33), (1, 600, 3, 2), (9, 37, 5, 31), (7, 40, 4, 301),
                                      (3, 9, 2, 2049), (2, 5, 2, 4100), (17, 33, 9, 96),
                                      (40, 430, 4, 63), (130, 130, 3, 5), (33, 520, 2, 2049),
                                      (33, 520, 2, 4100), (33, 520, 2, 2048), (17, 1000, 3, 5), (33, 520, 4, 63)])
def test_propagate_rows(oracle, cuda_device, B, T, Nc, O, int_rescaler):
    run_fc(oracle, B, 48, T, Nc, O, seed=B + O, int_rescaler=int_rescaler)


# B, T, Nc, O: wide rows of many samples in chunks (whole, odd, a lone block in the last)
@pytest.mark.parametrize("int_rescaler", [None, 0.5])
@pytest.mark.parametrize("B,T,Nc,O", [(128, 9, 3, 768), (131, 11, 3, 801), (130, 7, 5, 2048), (129, 5, 2, 2081)])
def test_propagate_chunks(oracle, cuda_device, B, T, Nc, O, int_rescaler):
    run_fc(oracle, B, 40, T, Nc, O, seed=B + O, int_rescaler=int_rescaler)


# B, T, Nc, O: as many tables a step as 31-bit offsets reach (all, one); tables of 2 GiB
# and more, whose last row ends inside a piece or not
@pytest.mark.parametrize("int_rescaler", [None, 0.5])
@pytest.mark.parametrize("B,T,Nc,O", [(1, 70, 13, 1024), (1, 3, 19, 257), (5, 2, 15, 8190), (3, 1, 15, 16387),
                                      (2, 1, 20, 516)])
def test_propagate_large_tables(oracle, cuda_device, B, T, Nc, O, int_rescaler):
    """Only the rows that the samples select are the same on both sides; the
    oracle's other rows are never touched."""
    I, E = 64, 1 << Nc
    dev = torch.device("cuda:0")
    x, anchors, _, go = make_inputs(3, B, I, T, Nc, 0)
    go = torch.randn(B * O, generator=torch.Generator().manual_seed(O))
    ridx, rmd, rmi = oracle.check_detectors(x.numpy(), anchors.numpy(), B, I, T, Nc)
    Wd = torch.empty(T * E * O, device=dev).normal_(0.0, 0.01, generator=torch.Generator(device=dev).manual_seed(1))
    W = np.zeros(T * E * O, np.float32)
    for t in range(T):
        for b in range(B):
            row = ridx[b * T + t]
            for r in (row, row ^ (1 << rmi[b * T + t])):
                at = (t * E + r) * O
                W[at:at + O] = Wd[at:at + O].cpu().numpy()
    dm = make_dm(I, O, T, Nc, int_rescaler=int_rescaler)
    idx, md, mi = (torch.from_numpy(v).to(dev) for v in (ridx, rmd, rmi))
    out, xg = torch.zeros(B * O, device=dev), torch.zeros(B * I, device=dev)
    print(f"[rows] large tables B={B} T={T} Nc={Nc} O={O} int={int_rescaler}", flush=True)
    ad, gd = anchors.to(dev), go.to(dev)
    dm.forward_step(Wd, B, x.to(dev), ad, out, idx, 0.0, None, md, mi)
    dm.backward_backprop(Wd, B, gd, ad, idx, md, mi, xg, -1.0, None, None)
    rxg = oracle.propagate_fc(W, go.numpy(), ridx, rmd, rmi, anchors.numpy(), B, I, O, T, Nc, E,
                              int_mode=int_rescaler is not None, int_rescaler=int_rescaler or 1.0)
    if int_rescaler is not None:
        oracle.convert_int_to_float(rxg, int_rescaler)
        assert np.array_equal(xg.cpu().numpy(), rxg)
    else:
        xg_close(xg.cpu().numpy(), rxg, B, I, T, (O + 31) // 32)


def test_input_gradient_in_a_first_capture(cuda_device):
    """An input gradient without a weight gradient is captured by a manager that
    has no scratch yet, and every replay gives the eager (scattered) call's."""
    B, I, T, Nc, O = 64, 512, 2048, 9, 40
    x, anchors, W, go = make_inputs(2, B, I, T, Nc, O)
    dev = torch.device("cuda:0")
    xd, ad, Wd, gd = (v.to(dev) for v in (x, anchors, W, go))
    idx, mi = (torch.empty(B * T, dtype=torch.int32, device=dev) for _ in range(2))
    md, out = torch.empty(B * T, device=dev), torch.zeros(B * O, device=dev)
    first, other = (make_dm(I, O, T, Nc, int_rescaler=0.5) for _ in range(2))
    for dm in (first, other):
        dm.forward_step(Wd, B, xd, ad, out, idx, 0.0, None, md, mi)
    want = torch.zeros(B * I, device=dev)
    other.backward_backprop(Wd, B, gd, ad, idx, md, mi, want, -1.0, None, None)
    xg = torch.zeros(B * I, device=dev)
    torch.cuda.synchronize()
    print("[capture] input gradient", flush=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        xg.zero_()
        first.backward_backprop(Wd, B, gd, ad, idx, md, mi, xg, -1.0, None, None)
    for rep in range(3):
        xg.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        print(f"[capture] replay {rep}", flush=True)
        assert torch.equal(xg, want)


@pytest.mark.parametrize("O", [10, 33, 301])
def test_rows_not_looked_up_are_not_read(oracle, cuda_device, O):
    """Rows that no sample selects hold NaN: a row whose last piece crosses into
    one gives the oracle's gradients, which never touch it."""
    B, I, T, Nc = 6, 40, 25, 6
    E = 1 << Nc
    x, anchors, W, go = make_inputs(5, B, I, T, Nc, O)
    ridx, rmd, rmi = oracle.check_detectors(x.numpy(), anchors.numpy(), B, I, T, Nc)
    used = np.zeros((T, E), bool)
    rows = ridx.reshape(B, T)
    flip = rows ^ (1 << rmi.reshape(B, T))
    for t in range(T):
        used[t, rows[:, t]] = used[t, flip[:, t]] = True
    W = W.view(T, E, O)
    W[torch.from_numpy(~used)] = float("nan")
    W = W.reshape(-1).contiguous()
    dm = make_dm(I, O, T, Nc)
    dev = torch.device("cuda:0")
    xd, ad, Wd, gd = (v.to(dev) for v in (x, anchors, W, go))
    out, xg = torch.zeros(B * O, device=dev), torch.zeros(B * I, device=dev)
    idx = torch.empty(B * T, dtype=torch.int32, device=dev)
    md, mi = torch.empty(B * T, device=dev), torch.empty(B * T, dtype=torch.int32, device=dev)
    wg = torch.empty(T * E * O, device=dev)
    print(f"[rows] O={O}", flush=True)
    dm.forward_step(Wd, B, xd, ad, out, idx, 0.0, None, md, mi)
    dm.backward_backprop(Wd, B, gd, ad, idx, md, mi, xg, -1.0, wg, None, overwrite_weights_gradients=True)
    rxg = oracle.propagate_fc(W.numpy(), go.numpy(), ridx, rmd, rmi, anchors.numpy(), B, I, O, T, Nc, E)
    assert np.array_equal(out.cpu().numpy(), oracle.fill_outputs_fc(W.numpy(), ridx, B, O, T, E))
    assert np.all(np.isfinite(rxg))
    xg_close(xg.cpu().numpy(), rxg, B, I, T, (O + 31) // 32)


def check_forward(oracle, B, T, Nc, O, dgs, ordered):
    """Bit-exact for fp32 and int32 sums and for int8 tables, with or without
    ordered sums."""
    I, E = 32, 1 << Nc
    x, anchors, W, _ = make_inputs(B + T, B, I, T, Nc, O)
    q = torch.randint(-127, 128, (T * E * O,), dtype=torch.int8, generator=torch.Generator().manual_seed(O))
    scales = torch.rand(T, generator=torch.Generator().manual_seed(T)) * 0.01
    Wq = (scales[:, None] * q.view(T, -1).float()).reshape(-1)
    ridx, _, _ = oracle.check_detectors(x.numpy(), anchors.numpy(), B, I, T, Nc)
    dev = torch.device("cuda:0")
    for rescaler in (None, 0.5):
        dm = make_dm(I, O, T, Nc, bgs=dgs, int_rescaler=rescaler)
        dm.set_ordered_sums(ordered)
        for tables, call in ((W, lambda *a: dm.forward_step(W.to(dev), *a)),
                             (Wq, lambda *a: dm.forward_step_i8(q.to(dev), scales.to(dev), *a))):
            out = torch.zeros(B * O, device=dev)
            idx = torch.empty(B * T, dtype=torch.int32, device=dev)
            print(f"[blocks] B={B} T={T} O={O} dgs={dgs} int={rescaler}", flush=True)
            call(B, x.to(dev), anchors.to(dev), out, idx)
            want = oracle.fill_outputs_fc(tables.numpy(), ridx, B, O, T, E, dgs=dgs,
                                          int_mode=rescaler is not None, int_rescaler=rescaler or 1.0)
            if rescaler is not None:
                oracle.convert_int_to_float(want, rescaler)
            assert np.array_equal(idx.cpu().numpy(), ridx)
            assert np.array_equal(out.cpu().numpy(), want)


# B, T, Nc, O, dgs: fewer columns than a quad; a quad that crosses the row's end
# in the first, a middle and the last slice; a lone block; a last block of one
# table; block sizes around the 16 rows in flight; more blocks than a chunk of
# LDS holds (O = 250: 33 blocks of 252 columns); 512 rows a table
@pytest.mark.parametrize("ordered", [False, True])
@pytest.mark.parametrize("B,T,Nc,O,dgs", [(1, 40, 3, 1, 32), (2, 33, 2, 3, 32), (3, 16, 4, 5, 32),
                                          (70, 97, 3, 30, 32), (5, 64, 3, 259, 16), (300, 80, 3, 250, 2),
                                          (9, 35, 9, 67, 17), (1, 300, 2, 1030, 1), (2, 5, 2, 4100, 32), (257, 12, 4, 6, 15)])
def test_forward_blocks(oracle, cuda_device, B, T, Nc, O, dgs, ordered):
    check_forward(oracle, B, T, Nc, O, dgs, ordered)


# B, T, Nc, O, dgs: tables walked in order.  A lone block of one table and of 31, one
# and four columns a lane; a quad over the row's end; one sample a wavefront over several
# blocks (whole, ragged, one table each); four samples, the last wavefront's partly past
# the batch, with one column a lane and with four; a short walk of large tables
@pytest.mark.parametrize("ordered", [False, True])
@pytest.mark.parametrize("B,T,Nc,O,dgs", [(1, 1, 3, 1, 32), (5, 31, 4, 67, 32), (300, 19, 3, 501, 32),
                                          (70000, 5, 2, 2, 32), (400, 40, 3, 1030, 8), (401, 33, 3, 1030, 32),
                                          (400, 13, 3, 999, 1), (2101, 22, 3, 501, 7), (4101, 10, 2, 65, 3),
                                          (1102, 37, 3, 1001, 5), (830, 18, 10, 1301, 9)])
def test_forward_walk(oracle, cuda_device, B, T, Nc, O, dgs, ordered):
    check_forward(oracle, B, T, Nc, O, dgs, ordered)


# B, T, Nc, O: rows of a lane, of a piece and of a slice and one output more or
# less (1, 2 and 4 outputs a lane; 256 a slice); one to many samples a row
@pytest.mark.parametrize("int_rescaler", [None, 0.5])
@pytest.mark.parametrize("B,T,Nc,O", [(1, 3, 1, 1), (5, 7, 2, 65), (9, 11, 5, 127), (300, 6, 3, 129),
                                      (70, 9, 6, 257), (33, 5, 7, 255), (140, 40, 2, 514), (6, 70, 8, 131)])
def test_weight_gradient_rows(oracle, cuda_device, B, T, Nc, O, int_rescaler):
    """Overwritten and accumulated gradients (run_fc checks both, bit for bit)."""
    run_fc(oracle, B, 24, T, Nc, O, seed=B * O, int_rescaler=int_rescaler)


@pytest.mark.parametrize("O", [10, 129, 300])
def test_weight_gradient_accumulates(oracle, cuda_device, O):
    """fp32 accumulation into other values: rows with samples are summed from
    them in ascending order, rows without keep every bit (negative zeros, NaN)."""
    B, I, T, Nc = 20, 30, 13, 7
    E = 1 << Nc
    x, anchors, W, go = make_inputs(9, B, I, T, Nc, O)
    before = torch.randn(T * E * O, generator=torch.Generator().manual_seed(3))
    before[::7] = -0.0
    ridx, _, _ = oracle.check_detectors(x.numpy(), anchors.numpy(), B, I, T, Nc)
    free = np.ones((T, E), bool)
    for t in range(T):
        free[t, ridx.reshape(B, T)[:, t]] = False
    before.view(T, E, O)[..., 1][torch.from_numpy(free)] = float("nan")
    assert torch.isnan(before).any()
    dm = make_dm(I, O, T, Nc)
    dev = torch.device("cuda:0")
    xd, ad, Wd, gd, wg = (v.to(dev) for v in (x, anchors, W, go, before))
    out, xg = torch.zeros(B * O, device=dev), torch.zeros(B * I, device=dev)
    idx = torch.empty(B * T, dtype=torch.int32, device=dev)
    md, mi = torch.empty(B * T, device=dev), torch.empty(B * T, dtype=torch.int32, device=dev)
    print(f"[wgrad] accumulate O={O}", flush=True)
    dm.forward_step(Wd, B, xd, ad, out, idx, 0.0, None, md, mi)
    dm.backward_backprop(Wd, B, gd, ad, idx, md, mi, xg, -1.0, wg, None)
    want = before.numpy().copy()
    oracle.gather_wgrad_fc(go.numpy(), ridx, want, B, O, T, E)
    assert np.array_equal(wg.cpu().numpy().view(np.int32), want.view(np.int32))


# B, S, T, Nc, Npe, O: rows read where they are -- fewer columns than a lane's
# four, several items a wavefront, a quad over the row's end, a whole wavefront,
# two slices; one pair, 64 pairs and one more; totals that are not whole quads
# -- and, from three pairs a row, odd widths and staged slices (whole, partial)
@pytest.mark.parametrize("int_rescaler", [None, 0.5])
@pytest.mark.parametrize("B,S,T,Nc,Npe,O", [(1, 2, 3, 4, 2, 1), (3, 17, 5, 3, 3, 3), (2, 9, 9, 4, 0, 33),
                                            (1, 66, 3, 4, 4, 130), (2, 65, 2, 4, 3, 256),
                                            (1, 33, 2, 4, 2, 261), (5, 40, 11, 2, 1, 35),
                                            (6, 40, 8, 2, 1, 64), (6, 40, 3, 2, 2, 36), (4, 70, 2, 1, 0, 8)])
def test_seq_forward_rows(oracle, cuda_device, B, S, T, Nc, Npe, O, int_rescaler):
    from test_gpu_seq import run_seq
    run_seq(oracle, B, S, 20, T, Nc, Npe, O, seed=S + O, int_rescaler=int_rescaler, int_grad=True)


# B, S, T, Nc, Npe, O: rows where they are (narrow, odd, a row a wavefront), staged slices
@pytest.mark.parametrize("B,S,T,Nc,Npe,O", [(2, 9, 5, 4, 2, 8), (1, 12, 40, 3, 1, 33), (2, 20, 7, 4, 2, 256),
                                            (3, 20, 30, 3, 0, 261), (6, 40, 8, 2, 1, 64)])
def test_seq_forward_first_position(oracle, cuda_device, B, S, T, Nc, Npe, O):
    """Position 0 has no pairs: what its outputs hold stays, bit for bit
    (negative zeros); every other position is added to."""
    from test_gpu_seq import make_seq_dm, seq_inputs
    x, anchors, W, pe, _ = seq_inputs(O, B, S, 20, T, Nc, Npe, O)
    dm = make_seq_dm(20, O, T, Nc, S, Npe)
    dev = torch.device("cuda:0")
    before = torch.randn(B, S, O, generator=torch.Generator().manual_seed(4))
    before[..., ::3] = -0.0
    out = before.reshape(-1).to(dev)
    idx, mi = (torch.empty(B * S * T, dtype=torch.int32, device=dev) for _ in range(2))
    pli, pmi = (torch.empty((S - 1) * T, dtype=torch.int32, device=dev) if Npe else None for _ in range(2))
    md, pmd = torch.empty(B * S * T, device=dev), torch.empty((S - 1) * T, device=dev) if Npe else None
    print(f"[seq] first position S={S} T={T} O={O}", flush=True)
    dm.forward_step_concat(W.to(dev), B, x.to(dev), anchors.to(dev), out, idx, 0.0, pe.to(dev) if Npe else None,
                           pli, md, mi, pmd, pmi)
    got, before = out.cpu().view(B, S, O).numpy(), before.numpy()
    assert np.array_equal(got[:, 0].copy().view(np.int32), before[:, 0].copy().view(np.int32))
    ridx, _, _ = oracle.check_detectors(x.numpy(), anchors.numpy(), B * S, 20, T, Nc)
    rpli = oracle.check_pe(pe.numpy(), S, T, Npe)[0] if Npe else None
    add = oracle.fill_outputs_seq(W.numpy(), ridx, rpli, B, O, T, S, Nc, Npe).reshape(B, S, O)
    # T fp32 additions from another start
    bound = (T + 1) * 2.0 ** -24 * (np.abs(before) + np.abs(add) + T * 0.01 * S)
    assert np.all(np.abs(got.astype(np.float64) - before - add) <= bound)


# tables past the 256 MB cache, whose wavefronts are held back: a row a wavefront,
# and an odd row over two
@pytest.mark.parametrize("S,O", [(40, 256), (33, 261)])
def test_seq_forward_rows_large_tables(oracle, cuda_device, S, O):
    from test_gpu_seq import run_seq
    run_seq(oracle, 1, S, 20, 5, 6, 4, O, seed=S + O, int_grad=True)


# S, Npe, O: the grouped input gradient over rows padded to 64, 128 and 256
# outputs and the weight gradient's unaligned 16-byte pieces: one output, a piece
# and one more, a slice and one more, two slices less one, widths past 128 at few
# and at many pairs a row (even widths change form there)
@pytest.mark.parametrize("B,S,Nc,Npe,O", [(2, 9, 3, 2, 1), (3, 20, 4, 0, 5), (2, 17, 3, 1, 33),
                                          (2, 30, 3, 3, 65), (1, 40, 3, 2, 127), (3, 25, 4, 0, 129),
                                          (2, 12, 4, 1, 132), (6, 33, 2, 1, 252), (2, 30, 3, 4, 255)])
@pytest.mark.parametrize("policy", ["dense", "accumulate", "internal"])
def test_seq_backward_padded_rows(oracle, cuda_device, B, S, Nc, Npe, O, policy):
    from test_gpu_seq import run_seq
    # the accumulating check wants rows that no pair reaches
    accumulate = policy == "accumulate" and Nc > 2
    run_seq(oracle, B, S, 24, 3, Nc, Npe, O, seed=O, internal=policy == "internal", accumulate=accumulate)


@pytest.mark.parametrize("O", [70, 130])
def test_seq_int32_unaligned_rows(oracle, cuda_device, O):
    from test_gpu_seq import run_seq
    run_seq(oracle, 2, 24, 16, 3, 3, 2, O, seed=O, int_rescaler=0.5)


@pytest.mark.parametrize("O", [64, 256])
@pytest.mark.parametrize("overwrite", [True, False])
def test_seq_gradient_target_alignment(oracle, cuda_device, O, overwrite):
    """A weight gradient that starts 4 bytes past a 16-byte boundary gets the
    aligned one's values."""
    from test_gpu_seq import make_seq_dm, seq_inputs
    B, S, I, T, Nc, Npe = 2, 30, 16, 3, 3, 2
    x, anchors, W, pe, go = seq_inputs(6, B, S, I, T, Nc, Npe, O, int_grad=True)
    dm = make_seq_dm(I, O, T, Nc, S, Npe)
    dev = torch.device("cuda:0")
    xd, ad, Wd, ped, gd = (v.to(dev) for v in (x, anchors, W, pe, go))
    out = torch.zeros(B * S * O, device=dev)
    idx, mi = (torch.empty(B * S * T, dtype=torch.int32, device=dev) for _ in range(2))
    pli, pmi = (torch.empty((S - 1) * T, dtype=torch.int32, device=dev) for _ in range(2))
    md, pmd = torch.empty(B * S * T, device=dev), torch.empty((S - 1) * T, device=dev)
    dm.forward_step_concat(Wd, B, xd, ad, out, idx, 0.0, ped, pli, md, mi, pmd, pmi)
    got = []
    for shift in (0, 1):
        wg = torch.ones(Wd.numel() + 1, device=dev)[shift:shift + Wd.numel()]
        xg, peg = torch.zeros(B * S * I, device=dev), torch.zeros((S - 1) * T * Npe, device=dev)
        print(f"[seq] gradient target O={O} shift={shift}", flush=True)
        dm.backward_backprop_concat(Wd, B, gd, ad, idx, md, mi, xg, -1.0, pli, pmd, pmi, peg, wg,
                                    overwrite_weights_gradients=overwrite)
        got.append(wg.cpu().numpy())
    assert np.array_equal(got[0], got[1])


# B, S, T, Nc, Npe, O: enough tables for the rows to be read where they are also at
# widths that have no staged form (see the shapes above)
@pytest.mark.parametrize("int_rescaler", [None, 0.5])
@pytest.mark.parametrize("B,S,T,Nc,Npe,O", [(1, 2, 20, 4, 2, 1), (3, 17, 11, 3, 3, 3), (2, 9, 15, 4, 0, 33),
                                            (1, 33, 8, 4, 2, 261), (6, 5, 2, 3, 2, 35), (1, 66, 5, 4, 4, 131)])
def test_seq_forward_rows_any_width(oracle, cuda_device, B, S, T, Nc, Npe, O, int_rescaler):
    from test_gpu_seq import run_seq
    run_seq(oracle, B, S, 20, T, Nc, Npe, O, seed=S + O, int_rescaler=int_rescaler, int_grad=True)


def test_seq_forward_rows_large_tables_two_slices(oracle, cuda_device):
    from test_gpu_seq import run_seq
    run_seq(oracle, 1, 64, 20, 5, 6, 4, 261, seed=325, int_grad=True)


# B, S, T, Nc, Npe, O: enough pairs for the grouped input gradient over padded rows:
# one output, a piece and one more, a slice less or more one, one output past 128, a
# whole-quad width in each padded size, wide quads
@pytest.mark.parametrize("B,S,T,Nc,Npe,O", [(4, 100, 40, 3, 0, 1), (4, 100, 40, 3, 1, 5), (3, 70, 33, 3, 2, 33),
                                            (3, 60, 20, 4, 1, 65), (2, 66, 24, 3, 2, 127), (2, 50, 24, 3, 1, 129),
                                            (2, 50, 24, 3, 1, 255), (1, 112, 33, 4, 1, 36), (1, 112, 33, 4, 1, 100),
                                            (1, 80, 128, 3, 0, 132), (1, 80, 128, 3, 0, 252)])
def test_seq_backward_grouped_padded_rows(oracle, cuda_device, B, S, T, Nc, Npe, O):
    from test_gpu_seq import run_seq
    run_seq(oracle, B, S, 24, T, Nc, Npe, O, seed=O)
