"""GPU parity of the runtime-length pass over the lengths whose plans differ: one to five stages, every
radix, direct stages (a prime factor from 17 to 61), chirp convolutions (a larger one), odd and even,
up to the longest lines of one LDS tile, with the axis contiguous or across columns on either side."""
import numpy as np
import pytest

import fftcase as fc

pytestmark = pytest.mark.gpu

LENGTHS = [2, 3, 7, 10, 11, 13, 14, 15, 18, 22, 25, 26, 36, 49, 50, 60, 72, 81, 90, 91, 100, 121, 125, 143, 150, 169, 180,
           225, 240, 250, 320, 343, 384, 400, 625, 768, 1000, 1331, 2187, 2400, 3125, 5000,
           17, 19, 34, 37, 51, 61, 186, 289, 323, 4913, 67, 127, 158, 199, 254, 509, 2003, 4999, 201, 268, 402, 2010, 4489]


@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
@pytest.mark.parametrize("n", LENGTHS)
def test_c2c_lengths(hmi, cuda, oracle, dtype, n):
    import torch
    # lines of n points walked along the axis and across columns, odd column counts (partial tiles)
    for size, inorder, outorder in [((n, 19, 3), (0, 1, 2), (1, 2, 0)), ((7, n, 5), (0, 1, 2), (0, 1, 2)),
                                    ((3, 37, n), (2, 0, 1), (2, 0, 1))]:
        inbox = hmi.box3d([0, 0, 0], [s - 1 for s in size], inorder)
        outbox = hmi.box3d([0, 0, 0], [s - 1 for s in size], outorder)
        plan = hmi.fft3d(hmi.backend.mi355, inbox, outbox)
        x = fc.uniform_complex(2 * int(np.prod(size)), n)
        tx = fc.to_gpu(x, np.complex64 if dtype == "complex64" else np.complex128)
        ty, tz = torch.empty_like(tx), torch.empty_like(tx)
        plan.forward(tx, ty, hmi.scale.none, 2)
        plan.backward(ty, tz, hmi.scale.full, 2)
        bi = oracle.Box.make((0, 0, 0), [s - 1 for s in size], inorder)
        bo = oracle.Box.make((0, 0, 0), [s - 1 for s in size], outorder)
        ref = oracle.fft3d_c2c(bi, bo, x, -1, 1.0, 2)
        assert fc.rel_l2(fc.to_host(ty), ref) <= fc.TOL[dtype], (size, inorder, outorder)
        assert fc.rel_l2(fc.to_host(tz), x) <= fc.TOL[dtype], (size, inorder, outorder)


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("n", [17, 38, 127, 254, 2, 6, 15, 25, 36, 50, 60, 99, 100, 147, 180, 225, 250, 300, 390, 720, 1000])
def test_r2c_and_r2r_lengths(hmi, cuda, oracle, dtype, n):
    import torch
    rdt = np.float32 if dtype == "float32" else np.float64
    rng = np.random.default_rng(n)
    for size, order, axis in [((n, 18, 3), (0, 1, 2), 0), ((5, n, 7), (0, 1, 2), 1), ((9, 5, n), (1, 2, 0), 2)]:
        inbox = hmi.box3d([0, 0, 0], [s - 1 for s in size], order)
        plan = hmi.fft3d_r2c(hmi.backend.mi355, inbox, inbox.r2c(axis), axis)
        x = rng.standard_normal(inbox.count())
        tx = torch.from_numpy(x.astype(rdt)).to(cuda)
        ty = torch.empty(plan.size_outbox(), dtype=torch.complex64 if rdt == np.float32 else torch.complex128, device=cuda)
        tz = torch.empty_like(tx)
        plan.forward(tx, ty)
        plan.backward(ty, tz, hmi.scale.full)
        b = oracle.Box.make((0, 0, 0), [s - 1 for s in size], order)
        half = inbox.r2c(axis)
        ref = oracle.fft3d_r2c(b, oracle.Box.make(half.low, half.high, order), axis, x)
        assert fc.rel_l2(fc.to_host(ty), ref) <= fc.TOL[dtype], (size, order)
        assert fc.rel_l2(fc.to_host(tz), x) <= fc.TOL[dtype], (size, order)
        for kind, fn in [("cos", oracle.r2r_cos), ("sin", oracle.r2r_sin)]:
            rplan = hmi.rtransform(hmi.backend.mi355, inbox, inbox, getattr(hmi.kind, kind))
            tr = torch.empty_like(tx)
            rplan.forward(tx, tr)
            assert fc.rel_l2(fc.to_host(tr), fn(b, b, x, -1)) <= fc.TOL[dtype], (kind, size)
            rplan.backward(tr, tz, hmi.scale.full)
            assert fc.rel_l2(fc.to_host(tz), x) <= fc.TOL[dtype], (kind, size)


@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
@pytest.mark.parametrize("size", [(2, 3, 1), (16, 16, 16), (7, 12, 5), (32, 30, 3), (81, 64, 2), (20, 256, 3), (100, 45, 7),
                                  (3, 4, 900), (64, 1, 9), (98, 102, 4), (256, 19, 6)])
def test_fused_planes(hmi, cuda, oracle, dtype, size):
    """Boxes with one layout on both sides run their two fastest axes in one pass where a plane fits the
    LDS: every order, in and out of place, a batch, both directions and the fused product."""
    import torch
    n = int(np.prod(size))
    x = fc.uniform_complex(2 * n, n % 97)
    for order in [(0, 1, 2), (2, 0, 1), (1, 0, 2)]:
        box = hmi.box3d([0, 0, 0], [s - 1 for s in size], order)
        plan = hmi.fft3d(hmi.backend.mi355, box, box)
        b = oracle.Box.make((0, 0, 0), [s - 1 for s in size], order)
        ref = oracle.fft3d_c2c(b, b, x, -1, 1.0, 2)
        tx = fc.to_gpu(x, np.complex64 if dtype == "complex64" else np.complex128)
        ty = torch.empty_like(tx)
        plan.forward(tx, ty, hmi.scale.none, 2)
        assert fc.rel_l2(fc.to_host(ty), ref) <= fc.TOL[dtype], order
        plan.backward(ty, ty, hmi.scale.full, 2)
        assert fc.rel_l2(fc.to_host(ty), x) <= fc.TOL[dtype], order
        tz = torch.empty_like(tx)
        plan.convolve(tx, ty, tz, None, hmi.scale.full, 2)
        assert fc.rel_l2(fc.to_host(tz), oracle.convolve3d(b, b, x, x, 1.0 / n, 2)) <= 2 * fc.TOL[dtype], order


def passes_of(plan):
    return " ".join(plan.timing())


@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
@pytest.mark.parametrize("size,batch", [((2, 3, 1), 700), ((4, 4, 4), 300), ((5, 7, 3), 401), ((8, 8, 8), 129), ((16, 16, 16), 70),
                                        ((32, 30, 3), 90), ((81, 64, 2), 60), ((20, 256, 3), 20), ((100, 45, 2), 30),
                                        ((98, 100, 4), 30), ((256, 20, 3), 18), ((128, 32, 5), 12)])
def test_fused_planes_of_a_batch(hmi, cuda, oracle, dtype, size, batch):
    """The planes of a whole batch are grouped into blocks, and planes that fill a CU take the fused pass
    only where the batch holds enough of them: both schedules of one plan, one transform and the batch."""
    import torch
    n = int(np.prod(size))
    x = fc.uniform_complex(batch * n, n % 89)
    box = hmi.box3d([0, 0, 0], [s - 1 for s in size])
    plan = hmi.fft3d(hmi.backend.mi355, box, box)
    b = oracle.Box.make((0, 0, 0), [s - 1 for s in size], (0, 1, 2))
    ref = oracle.fft3d_c2c(b, b, x, -1, 1.0, batch)
    tx = fc.to_gpu(x, np.complex64 if dtype == "complex64" else np.complex128)
    ty, tz = torch.empty_like(tx), torch.empty(n, dtype=tx.dtype, device=cuda)
    plan.set_timing(True)
    plan.forward(tx, ty, hmi.scale.none, batch)
    assert "fft_plane" in passes_of(plan)
    assert fc.rel_l2(fc.to_host(ty), ref) <= fc.TOL[dtype]
    plan.set_timing(True)
    plan.forward(tx, tz)
    # one transform: planes of about 64 KiB and more in a CU each would leave the others idle
    wide = (size[0] | 1) * size[1] * tx.element_size() > 64 * 1024
    assert ("fft_plane" in passes_of(plan)) == (not wide)
    plan.set_timing(False)
    assert fc.rel_l2(fc.to_host(tz), ref[:n]) <= fc.TOL[dtype]
    plan.backward(ty, ty, hmi.scale.full, batch)
    assert fc.rel_l2(fc.to_host(ty), x) <= fc.TOL[dtype]


def test_sixteen_million_small_boxes(hmi, cuda, oracle):
    """2^24 boxes of 4 x 4 x 4 in one call, in place (8.6 GB): one plane per block would ask for 2^32
    threads, more than a launch takes."""
    import torch
    few, n = 64, 64
    x = fc.uniform_complex(few * n, 3)
    box = hmi.box3d([0, 0, 0], [3, 3, 3])
    plan = hmi.fft3d(hmi.backend.mi355, box, box)
    b = oracle.Box.make((0, 0, 0), (3, 3, 3), (0, 1, 2))
    ref = oracle.fft3d_c2c(b, b, x, -1, 1.0, few)
    tx = fc.to_gpu(x, np.complex64)
    many = tx.repeat((1 << 24) // few)
    plan.forward(many, many, hmi.scale.none, 1 << 24)
    many = many.view(-1, few * n)
    assert fc.rel_l2(fc.to_host(many[0]), ref) <= fc.TOL["complex64"]
    assert all(torch.equal(rows, many[:1].expand_as(rows)) for rows in many.split(1 << 16))
