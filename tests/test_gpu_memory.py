"""Calls that use memory for speed and accuracy alone, where there is none for
it: the same images without it."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# 2560 is the longest row the FP32 detector takes in FP64 past its columns
@pytest.mark.parametrize("N", [64, 250, 2560, 2592])
def test_detector_captured_without_its_double_columns(pkg, N):
    """A captured FP32 detector of a context that has only run the FP64 one
    cannot allocate the copy of its columns: it works in FP32 throughout, as a
    row too long for that copy does."""
    L, lam, na = 100.0, 4.0, (0.0, 0.5)
    g = torch.Generator(device="cuda").manual_seed(N)
    F = [torch.view_as_complex(torch.randn(N * N, 2, generator=g, device="cuda",
                                           dtype=torch.float64)) for _ in range(2)]
    # the FP64 values of the fields as the FP32 call gets them
    U, Uf = (f.to(torch.complex64) for f in F)
    side = torch.cuda.Stream()
    c = pkg.Context(0, stream=side.cuda_stream)

    def run(prec, u, uf):
        rd = torch.float32 if prec == pkg.FP32_FAST else torch.float64
        out = [torch.zeros(N * N, dtype=rd, device="cuda") for _ in range(3)]
        torch.cuda.synchronize()
        c.detector(u, uf, N, N, 1 / L, 1 / L, *na, lam, 0, N, 1, *out, prec=prec,
                   write_filtered=False)
        torch.cuda.synchronize()
        return out

    want = run(pkg.FP64, U.to(torch.complex128), Uf.to(torch.complex128))
    out = [torch.zeros(N * N, dtype=torch.float32, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        c.detector(U, Uf, N, N, 1 / L, 1 / L, *na, lam, 0, N, 1, *out, prec=pkg.FP32_FAST,
                   write_filtered=False)
    for _ in range(2):
        for o in out:
            o.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        # FP32: about log2(N^2) roundings of 6e-8 each way on a random field
        for o, w in zip(out[:2], want):
            assert (o.double() - w).norm() <= 2e-6 * w.norm()
    eager = run(pkg.FP32_FAST, U, Uf)
    for o, e, w in zip(out[:2], eager, want):
        assert (e.double() - w).norm() <= 2e-6 * w.norm()
        # where there is a wide form, the eager call takes it and is the nearer
        if N <= 2560:
            assert (e.double() - w).norm() < (o.double() - w).norm()
        else:
            assert torch.equal(o, e)
    del graph
    c.close()


def test_batch_without_room_for_its_nodes_and_double_columns(pkg, ctx):
    import bimsim_amd.pipeline as P
    import bimsim_amd.workloads as W
    inst = W.config(2, N=1024, nk=20)
    inst["obj"] = (0.0, 0.9 * inst["lam"] * 512 / inst["L"])   # most columns pass
    insts = [inst] * 64
    waves = [W.mc_waves(inst, pkg.mc_sample_na)] * len(insts)
    arr, spheres, Wv, n = P.batch_tables(insts, waves)
    wd = torch.as_tensor(np.ascontiguousarray(Wv).ravel()).cuda()
    out = [torch.zeros(n, dtype=torch.float32, device="cuda") for _ in range(3)]

    def create():
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        b = ctx.batch(arr, spheres, wd, *out, prec=pkg.FP32_FAST)
        return b, before - torch.cuda.mem_get_info()[0]

    b, _ = create()   # (the tuner's own memory comes and goes in the first)
    b.close()
    b, full = create()
    want = [o.clone() for o in out]
    b.close()
    torch.cuda.empty_cache()
    # room for all but some gigabyte of what it took
    room = 1 << 30
    free = torch.cuda.mem_get_info()[0]
    assert full > 3 * room, full
    hold = torch.empty(free - full + room, dtype=torch.uint8, device="cuda")
    try:
        for o in out:
            o.fill_(5.0)
        b, lean = create()
        assert lean < full - room
        got = [o.clone() for o in out]
        b.launch()
        for o, g in zip(out, got):
            assert torch.equal(o, g)
        b.close()
    finally:
        del hold
        torch.cuda.empty_cache()
    for g, w in zip(got[:2], want):
        assert (g - w).norm() <= 5e-6 * w.norm()
