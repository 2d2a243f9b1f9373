"""Linear entries enqueued while a stream is captured: the graphs hold the
caller's buffers only, so they are replayed side by side on two streams, beside
eager calls of the same context and after it is destroyed; and eager calls
while another stream is captured."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import assert_close, act_host, dev, empty

pytestmark = pytest.mark.gpu


def _weights(rng, N, K, wfmt, act):
    wf = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    return (O.to_act(wf, act), None) if wfmt == O.W_DENSE else O.quantize(wf, wfmt)


def _ptr(t):
    return None if t is None else t.data_ptr()


class _Linear:
    """lssm_linear of a shape whose K is split (12 tiles, 80 K steps)."""
    M, N, K, act, wfmt = 70, 256, 5120, O.BF16, O.W_Q4_G64

    def __init__(self, rng, w, s):
        self.w, self.s = w, s
        self.x, self.y = dev(O.to_act(rng.standard_normal((self.M, self.K)), self.act)), empty((self.M, self.N), self.act)
        self.outs = [self.y]

    @classmethod
    def weights(cls, rng):
        return [None if a is None else dev(a) for a in _weights(rng, cls.N, cls.K, cls.wfmt, cls.act)]

    def reset(self):
        self.y.zero_()

    def call(self, c):
        c.linear(self.x, self.w, self.s, self.y, self.M, self.N, self.K, self.wfmt, self.act)


class _Rows(_Linear):
    """lssm_norm_linear_decode through the batched GEMV: two row tiles, the last partial."""
    M, N, K, act, wfmt = 24, 4100, 2560, O.BF16, O.W_Q8_G32

    def __init__(self, rng, w, s):
        super().__init__(rng, w, s)
        self.nw = dev(O.to_act(1 + 0.1 * rng.standard_normal(self.K), self.act))

    def call(self, c):
        import lite_ssm_amd as L
        L.check(L.lib.lssm_norm_linear_decode(c.h, _ptr(self.x), _ptr(self.nw), 1e-5, _ptr(self.w), _ptr(self.s),
                                              _ptr(self.y), None, self.M, self.N, self.K, self.wfmt, self.act,
                                              L.EPI_NONE))


class _RowsInt4(_Rows):
    M, N, K, act, wfmt = 33, 1000, 8192, O.F16, O.W_Q4_B32


class _RowsG64(_Rows):
    M, N, K, act, wfmt = 64, 72, 5120, O.BF16, O.W_Q4_G64


class _RowsDense(_Rows):
    """Fewer than four rows, of a dense weight too deep for the VALU GEMV."""
    M, N, K, act, wfmt = 3, 72, 8192, O.BF16, O.W_DENSE


class _Head(_Rows):
    """A dense weight wide enough for the norm launch and the tiled GEMM."""
    M, N, K, act, wfmt = 9, 32780, 2048, O.BF16, O.W_DENSE


class _InProj(_Rows):
    """lssm_inproj_decode: conv state updated in place."""
    D_INNER, G, STATE, H, DCONV = 1024, 2, 64, 16, 4
    XBC = 1024 + 2 * 2 * 64
    M, N, K, act, wfmt = 17, 1024 + XBC + 16, 5120, O.BF16, O.W_Q8_G32

    def __init__(self, rng, w, s):
        super().__init__(rng, w, s)
        a = self.act
        self.cw, self.cb = dev(O.to_act(rng.standard_normal((self.XBC, 4)) * 0.3, a)), dev(O.to_act(rng.standard_normal(self.XBC) * 0.1, a))
        self.cs0 = dev(O.to_act(rng.standard_normal((self.M, self.XBC, 4)), a))
        self.cs = self.cs0.clone()
        self.z, self.xa, self.dt = (empty((self.M, n), a) for n in (self.D_INNER, self.XBC, self.H))
        self.outs = [self.z, self.xa, self.dt, self.cs]

    def reset(self):
        self.cs.copy_(self.cs0)

    def call(self, c):
        import lite_ssm_amd as L
        L.check(L.lib.lssm_inproj_decode(c.h, _ptr(self.x), _ptr(self.nw), _ptr(self.w), _ptr(self.s), _ptr(self.cs),
                                         _ptr(self.cw), _ptr(self.cb), _ptr(self.z), _ptr(self.xa), _ptr(self.dt),
                                         self.M, self.K, self.D_INNER, self.STATE, self.G, self.H, self.DCONV, 1e-5,
                                         self.wfmt, self.act))


def _capture(c, st, call):
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    c.begin_batch()                       # enqueue only
    with torch.cuda.stream(st):
        g.capture_begin()
        call.call(c)
        g.capture_end()
    c.commit_and_wait()
    return g


def _solo(call, run):
    call.reset()
    torch.cuda.synchronize()
    run()
    torch.cuda.synchronize()
    return [t.clone() for t in call.outs]


@pytest.mark.parametrize("kind", [_Linear, _Rows, _RowsInt4, _RowsG64, _RowsDense, _Head, _InProj])
def test_captured_linears_hold_no_context_memory(ctx, rng, kind):
    import lite_ssm_amd as L
    print(f"case: captured {kind.__name__} act {kind.act} fmt {kind.wfmt} {kind.M} x {kind.N} x {kind.K}", flush=True)
    w = kind.weights(rng)
    calls = [kind(rng, *w) for _ in range(3)]
    eager = [_solo(k, lambda: k.call(ctx)) for k in calls]
    st = torch.cuda.Stream()
    c2 = L.Ctx(st.cuda_stream)
    graphs = [_capture(c2, st, k) for k in calls[:2]]
    want = [_solo(k, g.replay) for k, g in zip(calls, graphs)]
    for got, ref in zip(want, eager):
        for a, b in zip(got, ref):
            if kind in (_Linear, _Head):  # another order of sums: one rounding of each output apart
                assert_close(act_host(a, kind.act), act_host(b, kind.act), kind.act, 1.6e-2, "captured against eager")
            else:
                assert torch.equal(a, b)
    # the same call captured after an eager one: the same launches
    again = _solo(calls[2], lambda: calls[2].call(c2))
    assert all(torch.equal(a, b) for a, b in zip(again, eager[2]))
    g0 = _capture(c2, st, calls[0])
    assert all(torch.equal(a, b) for a, b in zip(_solo(calls[0], g0.replay), want[0]))

    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for it in range(10):
        for k in calls:
            k.reset()
        torch.cuda.synchronize()
        for s, g in zip(streams, graphs):
            with torch.cuda.stream(s):
                for _ in range(1 if kind is _InProj else 4):
                    g.replay()
        c2.begin_batch()
        calls[2].call(c2)
        c2.commit_and_wait()
        torch.cuda.synchronize()
        for k, ref in zip(calls, want + [again]):
            assert all(torch.equal(a, b) for a, b in zip(k.outs, ref)), f"replay {it}"
    c2.close()
    for k, g, ref in zip(calls, graphs, want):
        assert all(torch.equal(a, b) for a, b in zip(_solo(k, g.replay), ref))


def test_first_split_call_allocates_nothing(ctx, rng):
    """A context's first lssm_linear that splits K allocates no memory, which a
    capture of another stream (global mode) would refuse and be ended by."""
    import lite_ssm_amd as L
    print("case: first split linear of a context beside a capture", flush=True)
    k = _Linear(rng, *_Linear.weights(rng))
    want = _solo(k, lambda: k.call(ctx))                 # (code loaded)
    st, cap = torch.cuda.Stream(), torch.cuda.Stream()
    c2 = L.Ctx(st.cuda_stream)
    a = torch.zeros(1000, device="cuda")
    k.reset()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    c2.begin_batch()
    with torch.cuda.stream(cap):
        g.capture_begin(capture_error_mode="global")
        a.add_(1)
        k.call(c2)
        g.capture_end()
    c2.commit_and_wait()
    assert torch.equal(k.y, want[0])
    assert free - torch.cuda.mem_get_info()[0] < 16 << 20
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(a, torch.ones_like(a))
    c2.close()
