"""The tiled convolution kernels of the learned preconditioner at the sizes where
their tiles, channel chunks and staged ranges end: channel counts around 16 and
32, volumes smaller than a block's columns (several samples a block) and of odd
size (steps of 16 columns across samples), rows too long for the staging (gather
kernels), and the fused epilogues.  Against PyTorch in FP32 on the same
BF16-rounded operands; FP32 summation order is the only difference, so 1e-5 of
the largest output, as in test_gpu_nn.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
F = torch.nn.functional


def bf(x):
    return x.to(torch.bfloat16).to(torch.float32)


def bits(x):
    return x.to(torch.bfloat16).view(torch.int16).to("cuda:0")


def rel(a, b):
    return float((a.cpu() - b).abs().max() / max(float(b.abs().max()), 1e-30))


CASES = [
    # cin, cout, NB, (D, H, W), slices
    (1, 1, 1, (1, 1, 1), 1), (17, 16, 5, (2, 2, 4), 2), (16, 17, 3, (3, 5, 7), 3), (33, 48, 2, (4, 4, 4), 1),
    (15, 65, 2, (9, 5, 6), 4), (32, 130, 1, (2, 8, 8), 2), (16, 16, 3, (8, 31, 33), 9), (5, 3, 2, (2, 3, 400), 3),
    (16, 32, 2, (16, 32, 33), 20), (64, 64, 1, (6, 16, 40), 5),
]


@pytest.mark.parametrize("cin,cout,nb,dims,ns", CASES)
def test_tiled_convolutions(cin, cout, nb, dims, ns):
    from hirensi_amd import precond as PC
    print(f"tiled conv cin={cin} cout={cout} nb={nb} dims={dims} slices={ns}", flush=True)
    L, s = PC.lib(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(cin * 131 + cout)
    x, dy = torch.randn((nb, cin) + dims, generator=g), torch.randn((nb, cout) + dims, generator=g)
    w, b = torch.randn(cout, cin * 27, generator=g) / np.sqrt(27.0 * cin), torch.randn(cout, generator=g)
    add, gate = torch.randn(dy.shape, generator=g), torch.randn(dy.shape, generator=g)
    ref = F.conv3d(bf(x), bf(w).view(cout, cin, 3, 3, 3), b, padding=1)
    xd, wd, bd, addd, gated, dyd = (v.to("cuda:0") if v.dtype == torch.float32 else v
                                    for v in (x, bits(w), b, add, gate, dy))
    y = torch.empty_like(dyd)

    def conv(a, gt, slope):
        assert L.hr_nn_conv3d_fused(xd.data_ptr(), wd.data_ptr(), bd.data_ptr(), a, gt, slope, y.data_ptr(), cin, cout,
                                    nb, *dims, s) == 0
        return y
    assert rel(conv(None, None, 1.0), ref) < 1e-5
    assert rel(conv(addd.data_ptr(), None, 0.1), F.leaky_relu(ref + add, 0.1)) < 1e-5
    assert rel(conv(None, gated.data_ptr(), 0.1), torch.where(gate > 0, ref, 0.1 * ref)) < 1e-5
    dw, db = torch.empty(cout * cin * 27, device="cuda:0"), torch.empty(cout, device="cuda:0")
    part = torch.empty(ns * dw.numel(), device="cuda:0")
    assert L.hr_nn_conv3d_wgrad(xd.data_ptr(), dyd.data_ptr(), part.data_ptr(), ns, dw.data_ptr(), db.data_ptr(), cin,
                                cout, nb, *dims, s) == 0
    ref_dw = torch.nn.grad.conv3d_weight(bf(x), (cout, cin, 3, 3, 3), bf(dy), padding=1).reshape(-1)
    assert rel(dw, ref_dw) < 1e-5
    assert rel(db, dy.sum(dim=(0, 2, 3, 4))) < 1e-5


def test_infinite_and_nan_inputs_stay_in_their_neighbourhood():
    """Padding columns and K entries past the last channel multiply nothing: a
    non-finite voxel reaches its 27 neighbours and no others."""
    from hirensi_amd import precond as PC
    print("tiled conv with inf and nan voxels", flush=True)
    L, s = PC.lib(), torch.cuda.current_stream().cuda_stream
    cin, cout, nb, dims = 3, 5, 2, (5, 6, 7)
    g = torch.Generator().manual_seed(2)
    x, w = torch.randn((nb, cin) + dims, generator=g), torch.randn(cout, cin * 27, generator=g)
    x[0, 2, 4, 5, 6], x[1, 0, 0, 0, 0] = float("nan"), float("inf")
    ref = F.conv3d(x, w.view(cout, cin, 3, 3, 3), None, padding=1)
    xd, wd = x.to("cuda:0"), bits(w)
    y = torch.empty((nb, cout) + dims, device="cuda:0")
    assert L.hr_nn_conv3d(xd.data_ptr(), wd.data_ptr(), None, y.data_ptr(), cin, cout, nb, *dims, 0, s) == 0
    assert torch.equal(torch.isfinite(y.cpu()), torch.isfinite(ref))


@pytest.mark.parametrize("cin,cout,dims", [(16, 16, (4, 8, 8)), (24, 40, (3, 5, 7)), (40, 70, (2, 4, 4)), (20, 33, (4, 4, 4)),
                                           (128, 64, (2, 4, 8))])
def test_weight_rows_at_every_alignment_give_the_same_bits(cin, cout, dims):
    """Rows at 16 bytes are read 16 bytes a lane and dealt to the lanes, others in smaller
    pieces: the same operands in the same order, so equal bits."""
    from hirensi_amd import precond as PC
    print(f"weight alignment cin={cin} cout={cout} dims={dims}", flush=True)
    L, s = PC.lib(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(cin + cout)
    xd, w = torch.randn((2, cin) + dims, generator=g).to("cuda:0"), bits(torch.randn(cout * cin * 27, generator=g))
    out = []
    for shift in (0, 4, 1):                     # 16, 8 and 2 bytes
        buf = torch.zeros(w.numel() + 8, dtype=torch.int16, device="cuda:0")
        buf[shift:shift + w.numel()] = w
        y = torch.empty((2, cout) + dims, device="cuda:0")
        assert L.hr_nn_conv3d(xd.data_ptr(), buf.data_ptr() + 2 * shift, None, y.data_ptr(), cin, cout, 2, *dims, 0, s) == 0
        out.append(y)
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


# channels on both sides of the rule that leaves a convolution of few of them to the gather kernel
# (K steps against the staged places, for every tile), on narrow and wide rows and small and
# large grids, and rows of weights at 2 and 8 bytes
@pytest.mark.parametrize("cout,nb,dims", [(16, 1, (3, 5, 17)), (16, 4, (8, 33, 100)), (3, 4, (16, 8, 192)), (32, 4, (16, 16, 33)),
                                          (24, 2, (4, 4, 136)), (40, 2, (4, 6, 9)), (40, 2, (8, 33, 24)), (64, 2, (16, 32, 32))])
def test_convolutions_of_few_channels(cout, nb, dims):
    from hirensi_amd import precond as PC
    print(f"few channels cout={cout} nb={nb} dims={dims}", flush=True)
    L, s = PC.lib(), torch.cuda.current_stream().cuda_stream
    for cin in (1, 2, 3, 4, 5, 9, 12, 15, 16, 17, 20):
        g = torch.Generator().manual_seed(cin * 17 + cout)
        x, w = torch.randn((nb, cin) + dims, generator=g), torch.randn(cout, cin * 27, generator=g) / np.sqrt(27.0 * cin)
        b = torch.randn(cout, generator=g)
        xd, wd, bd = x.to("cuda:0"), bits(w), b.to("cuda:0")
        y = torch.empty((nb, cout) + dims, device="cuda:0")
        assert L.hr_nn_conv3d(xd.data_ptr(), wd.data_ptr(), bd.data_ptr(), y.data_ptr(), cin, cout, nb, *dims, 0, s) == 0
        assert rel(y, F.conv3d(bf(x), bf(w).view(cout, cin, 3, 3, 3), b, padding=1)) < 1e-5, cin


@pytest.mark.parametrize("cin,cout,nb,dims,ns", [(24, 64, 8, (1, 3, 16), 1), (1, 64, 8, (3, 2, 16), 12), (3, 40, 5, (1, 1, 16), 2),
                                                 (5, 33, 3, (4, 4, 4), 3), (5, 33, 3, (4, 4, 4), 1)])
def test_weight_gradients_of_small_samples(cin, cout, nb, dims, ns):
    """Samples that cut the staged chunks short, on both sides of the rule that leaves them to the
    gather kernel."""
    from hirensi_amd import precond as PC
    print(f"weight gradient cin={cin} cout={cout} nb={nb} dims={dims} slices={ns}", flush=True)
    L, s = PC.lib(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(cin + 7 * cout)
    x, dy = torch.randn((nb, cin) + dims, generator=g), torch.randn((nb, cout) + dims, generator=g)
    xd, dyd = x.to("cuda:0"), dy.to("cuda:0")
    dw, db = torch.empty(cout * cin * 27, device="cuda:0"), torch.empty(cout, device="cuda:0")
    part = torch.empty(ns * dw.numel(), device="cuda:0")
    assert L.hr_nn_conv3d_wgrad(xd.data_ptr(), dyd.data_ptr(), part.data_ptr(), ns, dw.data_ptr(), db.data_ptr(), cin,
                                cout, nb, *dims, s) == 0
    ref = torch.nn.grad.conv3d_weight(bf(x), (cout, cin, 3, 3, 3), bf(dy), padding=1).reshape(-1)
    assert rel(dw, ref) < 1e-5
    assert rel(db, dy.sum(dim=(0, 2, 3, 4))) < 1e-5


def test_a_batch_of_more_blocks_than_a_tile_can_launch():
    """16 columns a block (rows of 280, more than 32 output channels) pass the launch limit of 2^32
    threads at 2^28 columns, 52 GB here; the gather kernel has four times as
    many columns a block.  Samples of the batch against the same samples alone, whose tiles
    give the same bits."""
    from hirensi_amd import precond as PC
    L, s = PC.lib(), torch.cuda.current_stream().cuda_stream
    cin, cout, nb, dims = 16, 33, 235, (64, 64, 280)
    print(f"conv of {nb} x {dims} voxels, {cin} -> {cout} channels", flush=True)
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 60 GB of device memory")
    assert nb * dims[0] * dims[1] * dims[2] > 1 << 28
    x = torch.empty((nb, cin) + dims, device="cuda:0").uniform_(-1, 1)
    w = bits(torch.randn(cout * cin * 27, generator=torch.Generator().manual_seed(1)))
    y = torch.empty((nb, cout) + dims, device="cuda:0")
    one = torch.empty((1, cout) + dims, device="cuda:0")
    assert L.hr_nn_conv3d(x.data_ptr(), w.data_ptr(), None, y.data_ptr(), cin, cout, nb, *dims, 0, s) == 0
    for q in (0, 117, nb - 1):
        assert L.hr_nn_conv3d(x[q].data_ptr(), w.data_ptr(), None, one.data_ptr(), cin, cout, 1, *dims, 0, s) == 0
        assert torch.equal(y[q], one[0]) and float(one.abs().max()) > 0, q
    del x, y
    torch.cuda.empty_cache()
