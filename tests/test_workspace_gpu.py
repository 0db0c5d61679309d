"""Caller-owned workspaces (lz_workspace_create / lz_forward_device_ws):
forwards of different batches on two streams with a workspace each,
enqueued back to back so that they overlap, give exactly the results of
the same forwards run one after the other (fused and layered forms, both
nets)."""
import numpy as np
import pytest

from leela_amd.positions import make_batch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be(weights_a):
    import leela_amd
    b = leela_amd.Backend(0)
    pol, val = weights_a
    b.load_net(leela_amd.NET_POLICY, pol)
    b.load_net(leela_amd.NET_VALUE, val)
    b.finalize()
    yield b
    b.close()


@pytest.mark.parametrize("na,nb", [(300, 257), (16, 40)])
def test_two_streams_two_workspaces(be, na, nb):
    import torch
    import leela_amd
    p = leela_amd.PREC_FP16
    dev = torch.device("cuda", 0)
    print(f"case: n={na},{nb}", flush=True)
    for net, width in ((leela_amd.NET_POLICY, 361), (leela_amd.NET_VALUE, 1)):
        pa = make_batch(na, seed0=101, net=net)
        pb = make_batch(nb, seed0=909, net=net)
        want_a = be.forward(net, p, pa)
        want_b = be.forward(net, p, pb)
        da, db = torch.from_numpy(pa).to(dev), torch.from_numpy(pb).to(dev)
        ra = torch.empty((na, width), device=dev)
        oa = torch.empty_like(ra)
        rb = torch.empty((nb, width), device=dev)
        ob = torch.empty_like(rb)
        s1, s2 = torch.cuda.Stream(dev), torch.cuda.Stream(dev)
        w1, w2 = be.workspace(na), be.workspace(8)  # w2 grows on first use
        try:
            torch.cuda.synchronize()
            for _ in range(3):
                be.forward_device_ws(w1, net, p, na, da.data_ptr(),
                                     ra.data_ptr(), oa.data_ptr(),
                                     s1.cuda_stream)
                be.forward_device_ws(w2, net, p, nb, db.data_ptr(),
                                     rb.data_ptr(), ob.data_ptr(),
                                     s2.cuda_stream)
            torch.cuda.synchronize()
            np.testing.assert_array_equal(ra.cpu().numpy(), want_a[0])
            np.testing.assert_array_equal(oa.cpu().numpy(), want_a[1])
            np.testing.assert_array_equal(rb.cpu().numpy(), want_b[0])
            np.testing.assert_array_equal(ob.cpu().numpy(), want_b[1])
        finally:
            be.free_workspace(w1)
            be.free_workspace(w2)


@pytest.mark.parametrize("own", [False, True])
def test_captured_forwards_outlive_growth(weights_a, own):
    """16-bit forwards captured before the workspace grows (the policy's
    layered tiles: small batches, batches of 65..96 and the rest past a pass
    of 256; the value net's head planes) give the same results when they are
    replayed after it has grown, several times, with eager work between the
    replays."""
    import torch
    import leela_amd
    p = leela_amd.PREC_FP16
    be = leela_amd.Backend(0)
    for net, w in enumerate(weights_a):
        be.load_net(net, w)
    be.finalize()
    ws = be.workspace(8) if own else None

    def forward(net, n, d, raw, out, stream):
        args = (net, p, n, d.data_ptr(), raw.data_ptr(), out.data_ptr(),
                stream.cuda_stream)
        if own:
            be.forward_device_ws(ws, *args)
        else:
            be.forward_device(*args)

    def case(net, n):
        print(f"case: own={own} net={net} n={n}", flush=True)
        d = torch.from_numpy(make_batch(n, seed0=300 + n, net=net)).cuda()
        width = 361 if net == leela_amd.NET_POLICY else 1
        return (net, n, d, torch.empty((n, width), device="cuda"),
                torch.empty((n, width), device="cuda"))

    st = torch.cuda.Stream()
    cases = [case(0, 16), case(0, 80), case(0, 300), case(1, 300)]
    torch.cuda.synchronize()
    for c in cases:
        forward(*c, st)
    st.synchronize()
    want = [(c[3].cpu().numpy(), c[4].cpu().numpy()) for c in cases]
    graphs = []
    for c in cases:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            forward(*c, torch.cuda.current_stream())
        graphs.append(g)
    held = []
    for n in (420, 1500):
        big = [case(0, n), case(1, n)]
        torch.cuda.synchronize()
        for _ in range(2):
            for c in big:
                forward(*c, st)
            # Takes what the growth has given back.
            held += [torch.full((1 << 22,), -1, dtype=torch.int32,
                                device="cuda") for _ in range(8)]
            for c, g, w in zip(cases, graphs, want):
                c[3].fill_(-7.0)
                c[4].fill_(-7.0)
                torch.cuda.synchronize()
                with torch.cuda.stream(st):
                    g.replay()
                st.synchronize()
                np.testing.assert_array_equal(c[3].cpu().numpy(), w[0])
                np.testing.assert_array_equal(c[4].cpu().numpy(), w[1])
        assert all(bool((t == -1).all()) for t in held)
    del graphs
    if own:
        be.free_workspace(ws)
    be.close()


def test_host_forward_beside_device_forwards(weights_a):
    """lz_forward runs on the context's own stream, which a caller cannot
    order against: with device-buffer batches of the same context on the way
    on another stream (layered tiles and head planes in use on both), every
    result is that of the calls made alone."""
    import torch
    import leela_amd
    p = leela_amd.PREC_FP16
    be = leela_amd.Backend(0)
    for net, w in enumerate(weights_a):
        be.load_net(net, w)
    be.finalize()
    try:
        for net, width, na, nb in ((0, 361, 331, 96), (0, 361, 40, 20),
                                   (1, 1, 600, 50)):
            print(f"case: net={net} device n={na} host n={nb}", flush=True)
            pa = make_batch(na, seed0=11, net=net)
            pb = make_batch(nb, seed0=77, net=net)
            want_b = be.forward(net, p, pb)
            da = torch.from_numpy(pa).cuda()
            outs = [torch.empty((2, na, width), device="cuda")
                    for _ in range(21)]
            st = torch.cuda.Stream()
            torch.cuda.synchronize()

            def device(o):
                be.forward_device(net, p, na, da.data_ptr(), o[0].data_ptr(),
                                  o[1].data_ptr(), st.cuda_stream)

            device(outs[20])
            st.synchronize()
            for k in range(5):
                for o in outs[4 * k:4 * k + 4]:
                    device(o)
                got = be.forward(net, p, pb)
                for a, b in zip(got, want_b):
                    np.testing.assert_array_equal(a, b)
            st.synchronize()
            for o in outs[:20]:
                assert torch.equal(o, outs[20])
    finally:
        be.close()


def _dirty_memory():
    """Device memory that the next allocations may get is not zero."""
    import torch
    junk = [torch.full((1 << 25,), -1, dtype=torch.int32, device="cuda")
            for _ in range(6)]
    torch.cuda.synchronize()
    del junk
    torch.cuda.empty_cache()


def test_first_forward_on_fresh_tiles(weights_a):
    """A layered forward on the caller's stream right after its tiles were
    allocated and zeroed (by the forward itself, or by lz_workspace_create):
    the same as the next one. The fill has to be waited for, since the
    caller's stream is not ordered after it."""
    import torch
    import leela_amd
    p = leela_amd.PREC_FP16
    for k in range(4):
        _dirty_memory()
        be = leela_amd.Backend(0)
        for net, w in enumerate(weights_a):
            be.load_net(net, w)
        be.finalize()
        st = torch.cuda.Stream()
        d = torch.from_numpy(make_batch(16, seed0=k)).cuda()
        out = torch.empty((4, 16, 361), device="cuda")
        torch.cuda.synchronize()
        be.forward_device(0, p, 16, d.data_ptr(), None, out[0].data_ptr(),
                          st.cuda_stream)
        be.forward_device(0, p, 16, d.data_ptr(), None, out[1].data_ptr(),
                          st.cuda_stream)
        ws = be.workspace(8)
        for i in (2, 3):
            be.forward_device_ws(ws, 0, p, 16 if i == 3 else 8, d.data_ptr(),
                                 None, out[i].data_ptr(), st.cuda_stream)
        st.synchronize()
        print(f"case: fresh backend {k}", flush=True)
        assert torch.equal(out[0], out[1])
        assert torch.equal(out[2, :8], out[1, :8])
        assert torch.equal(out[3], out[1])
        be.free_workspace(ws)
        be.close()
