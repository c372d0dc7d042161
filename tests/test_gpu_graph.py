"""Ops recorded into a HIP graph (stream capture through torch.cuda.graph)
and replayed.  Every replay must equal the eager run of the same iteration
bit for bit; replays are separated by eager work (other fused BatchNorm
launches, which use the eager barrier counters) and synchronizations, as a
training loop would run them."""
import numpy as np
import pytest
import torch

import tensorflow_musa_extension_amd as tfma
from oracle import oracle

pytestmark = pytest.mark.gpu
ops = tfma.raw_ops
EPS = 1.001e-5


def _inputs(dev, shape, seed):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    c = shape[-1]
    return dict(
        x=torch.randn(shape, generator=g, device=dev).half(),
        dz=torch.randn(shape, generator=g, device=dev).half(),
        scale=torch.rand(c, generator=g, device=dev) + 0.5,
        offset=0.1 * torch.randn(c, generator=g, device=dev),
        bias=torch.randn(c, generator=g, device=dev).half(),
        var=0.02 * torch.randn(1 << 20, generator=g, device=dev),
        m=torch.zeros(1 << 20, device=dev),
        v=torch.zeros(1 << 20, device=dev),
        grad=1e-3 * torch.randn(1 << 20, generator=g, device=dev))


def _step(d):
    e = torch.empty(0, device=d["x"].device)
    f = ops.FusedBatchNormV3(d["x"], d["scale"], d["offset"], e, e, epsilon=EPS)
    z = ops.MusaBiasAddRelu(f.y, d["bias"])
    gz = ops.ReluGrad(d["dz"], z)
    db = ops.BiasAddGrad(gz)
    gr = ops.FusedBatchNormGradV3(gz, d["x"], d["scale"], f.reserve_space_1, f.reserve_space_2,
                                  f.reserve_space_3, epsilon=EPS)
    ops.ResourceApplyAdam(d["var"], d["m"], d["v"], 0.9, 0.999, 1e-3, 0.9, 0.999, 1e-7,
                          d["grad"])
    return [f.y, f.batch_mean, f.batch_variance, z, gz, db, gr.x_backprop, gr.scale_backprop,
            gr.offset_backprop]


def _state(d):
    return [d["var"].clone(), d["m"].clone(), d["v"].clone()]


# (16,14,14,256): every row resident, no dynamic chunks.  (128,56,56,256)
# unsliced (override bn_slice_tw 0): the grad hands out phase-3 chunks, so the
# recorded launch zeroes the chunk counters as well as the barrier counters
# at exit; left to the host, the grad runs in 2 slices of 128 channels
# (hand-offs hidden); with slice_tw 8 in 4 slices of 64 channels.
@pytest.mark.parametrize("shape,slice_tw,slices", [((16, 14, 14, 256), None, 1),
                                                   ((128, 56, 56, 256), 0, 1),
                                                   ((128, 56, 56, 256), None, 2),
                                                   ((128, 56, 56, 256), 8, 4)])
def test_recorded_training_step_replays(dev, tune, shape, slice_tw, slices):
    if slice_tw is not None:
        tune("bn_slice_tw", slice_tw)
    d = _inputs(dev, shape, seed=31)
    other = _inputs(dev, (8, 7, 7, 512), seed=32)
    e = torch.empty(0, device=dev)
    start = _state(d)
    eager = []
    for _ in range(3):
        eager.append([t.clone() for t in _step(d)] + _state(d))
        plan = ops.fused_batch_norm_last_plan()
        assert plan["slices"] == slices, plan
        if slice_tw == 0 and shape[1] == 56:
            assert plan["dynamic_rows"] > 0, plan
    other_ref = ops.FusedBatchNormV3(other["x"], other["scale"], other["offset"], e, e,
                                     epsilon=EPS).y.clone()
    torch.cuda.synchronize()
    for t, s in zip((d["var"], d["m"], d["v"]), start):
        t.copy_(s)
    ops.fused_batch_norm_barrier_timed_out(reset=True)

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = _step(d)
    torch.cuda.synchronize()
    for want in eager:
        graph.replay()
        y_other = ops.FusedBatchNormV3(other["x"], other["scale"], other["offset"], e, e,
                                       epsilon=EPS).y
        torch.cuda.synchronize()
        got = [t.clone() for t in outs] + _state(d)
        for k, (w, g) in enumerate(zip(want, got)):
            assert torch.equal(w, g), f"output {k} of a replay differs from the eager run"
        assert torch.equal(y_other, other_ref)
    assert not ops.fused_batch_norm_barrier_timed_out()


# (8,13,13,72): the folded kernel, recorded as it runs, and so are the kernels
# whose workgroups wait for none: units of one row group (33 images of 7x7) and
# shared channels of one part (9 images of 28x28).  The others run kernels whose
# workgroups wait for one another when eager and are recorded as the split
# kernels (a replay may overlap other work).
@pytest.mark.parametrize("shape,fmt,same", [((8, 13, 13, 72), "NHWC", True),
                                            ((8, 13, 13, 99), "NHWC", False),
                                            ((2, 9, 7, 515), "NHWC", False),
                                            ((9, 96, 28, 28), "NCHW", True),
                                            ((17, 96, 28, 28), "NCHW", False),
                                            ((64, 512, 7, 7), "NCHW", False),
                                            ((33, 512, 7, 7), "NCHW", True),
                                            ((9, 230, 28, 28), "NCHW", True)])
def test_recorded_batch_norm_replays(dev, tune, shape, fmt, same):
    """Three replays between eager launches: bit for bit the eager results, or
    one another and within rounding of the eager results."""
    gen_ = torch.Generator(device=dev)
    gen_.manual_seed(33)
    c = shape[-1] if fmt == "NHWC" else shape[1]
    x, dy = (torch.randn(shape, generator=gen_, device=dev).half() for _ in range(2))
    scale = torch.rand(c, generator=gen_, device=dev) + 0.5
    offset = torch.randn(c, generator=gen_, device=dev)
    e = torch.empty(0, device=dev)
    kw = dict(epsilon=EPS, data_format=fmt)
    plans = []
    tune("bn_folded", 1)

    def step():
        f = ops.FusedBatchNormV3(x, scale, offset, e, e, **kw)
        plans.append(ops.fused_batch_norm_last_plan()["fused"])
        return tuple(f) + tuple(ops.FusedBatchNormGradV3(
            dy, x, scale, f.reserve_space_1, f.reserve_space_2, f.reserve_space_3, **kw))

    want = [t.clone() for t in step()]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step()
    assert plans == [1, 1 if same else 0]
    first = None
    for _ in range(3):
        for t in outs:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        if first is None:
            first = [t.clone() for t in outs]
        for got, one, w in zip(outs, first, want):
            assert torch.equal(got, one)
            if same:
                assert torch.equal(got, w)
            elif w.dtype == torch.float16:  # one ulp of the largest value
                assert (got.float() - w.float()).abs().max() <= 2 ** -10 * w.float().abs().max()
            else:  # float32 sums of the same terms in another order
                assert (got - w).abs().max() <= 1e-5 * max(w.abs().max().item(), 1.0)
        assert all(torch.equal(a, b) for a, b in zip(step(), want))
        torch.cuda.synchronize()
    assert not ops.fused_batch_norm_barrier_timed_out()


@pytest.mark.parametrize("gdtype", [torch.float32, torch.bfloat16])
def test_grouped_adam_recorded_replays(dev, gdtype):
    """MusaGroupedResourceApplyAdam recorded into a graph (its tensor table
    travels in the kernel arguments: 100 tensors, two launches) and replayed
    three times, with eager grouped calls on other tensors between the
    replays: every replay applies one Adam step, bit for bit the oracle's."""
    g = torch.Generator(device=dev)
    g.manual_seed(41)
    sizes = [1 + (37 * k) % 5000 for k in range(100)]
    vars_ = [0.02 * torch.randn(n, generator=g, device=dev) for n in sizes]
    ms = [torch.zeros(n, device=dev) for n in sizes]
    vs = [torch.zeros(n, device=dev) for n in sizes]
    grads = [(1e-3 * torch.randn(n, generator=g, device=dev)).to(gdtype) for n in sizes]
    refs = [[t.cpu().numpy().copy() for t in (v, m, w)] for v, m, w in zip(vars_, ms, vs)]
    other = [torch.randn(4096, device=dev) for _ in range(3)]
    om = [torch.zeros(4096, device=dev) for _ in range(3)]
    ov = [torch.zeros(4096, device=dev) for _ in range(3)]
    og = [torch.randn(4096, device=dev) for _ in range(3)]
    b1p, b2p, lr, b1, b2, eps = 0.9, 0.999, 1e-3, 0.9, 0.999, 1e-7
    f32 = lambda x: float(np.float32(x))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.MusaGroupedResourceApplyAdam(vars_, ms, vs, grads, b1p, b2p, lr, b1, b2, eps)
    torch.cuda.synchronize()
    for _ in range(3):
        graph.replay()
        ops.MusaGroupedResourceApplyAdam(other, om, ov, og, b1p, b2p, lr, b1, b2, eps)
        torch.cuda.synchronize()
        for (rv, rm, rw), gt in zip(refs, grads):
            gn = gt.float().cpu().numpy()
            oracle.adam(rv, rm, rw, gn, f32(b1p), f32(b2p), f32(lr), f32(b1), f32(b2), f32(eps))
    for i, (v, m, w) in enumerate(zip(vars_, ms, vs)):
        for name, t, r in (("var", v, refs[i][0]), ("m", m, refs[i][1]), ("v", w, refs[i][2])):
            assert np.array_equal(t.cpu().numpy().view(np.uint32), r.view(np.uint32)), (i, name)


@pytest.mark.parametrize("shape,fmt", [((8, 13, 13, 99), "NHWC"), ((17, 96, 28, 28), "NCHW"),
                                       ((64, 512, 7, 7), "NCHW")])
def test_replays_overlap_eager_odd_shapes(dev, tune, shape, fmt):
    """A replay of a fused batch norm on one stream and eager calls of shapes
    that are not recorded as such (odd channels, shared channels, units) on
    another, in no order: neither touches the other's words, and a workgroup
    that misses what another has no room to run makes up for it."""
    tune("bn_folded", 1)
    g = torch.Generator(device=dev)
    g.manual_seed(35)
    kw = dict(epsilon=EPS)
    e = torch.empty(0, device=dev)

    def op(shape, fmt):
        c = shape[-1] if fmt == "NHWC" else shape[1]
        x, dy = (torch.randn(shape, generator=g, device=dev).half() for _ in range(2))
        scale = torch.rand(c, generator=g, device=dev) + 0.5
        offset = torch.randn(c, generator=g, device=dev)

        def step():
            f = ops.FusedBatchNormV3(x, scale, offset, e, e, data_format=fmt, **kw)
            return tuple(f) + tuple(ops.FusedBatchNormGradV3(
                dy, x, scale, f.reserve_space_1, f.reserve_space_2, f.reserve_space_3,
                data_format=fmt, **kw))
        return step

    fused, odd = op((64, 28, 28, 512), "NHWC"), op(shape, fmt)
    want_fused = [t.clone() for t in fused()]
    want_odd = [t.clone() for t in odd()]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = fused()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(5):
        for t in outs:
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[0]):
            for _ in range(4):
                graph.replay()
        with torch.cuda.stream(streams[1]):
            odds = [odd() for _ in range(12)]
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(outs, want_fused))
        for got in odds:
            for a, b in zip(got, want_odd):
                # Partials that were made up for may differ in the last bit.
                tol = 2 ** -10 if a.dtype == torch.float16 else 1e-6
                assert (a.float() - b.float()).abs().max() <= tol * max(b.abs().max().item(), 1.0)
    assert not ops.fused_batch_norm_barrier_timed_out()
