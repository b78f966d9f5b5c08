"""Several workgroups to a trajectory of a whole sampling run: against one workgroup and against the step-by-step route
with the same variates."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-4, torch.float16: 1e-2, torch.bfloat16: 2e-2}  # as for one workgroup: the same roundings


def _rel(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / b.norm().clamp(min=1e-30))


# Heads per workgroup 1, 2, 4, 8, wavefronts per head 8, 4, 2, 1; trajectories that fill the eight XCDs and that do not; one
# step; contexts that end in, at and past a block, a group of four blocks of every wavefront
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("backend", ["triton_shared_context", "flex_attention"], ids=["shared", "own"])
@pytest.mark.parametrize("D,parts,B,Nc,Nt", [(128, 2, 9, 1, 1), (128, 2, 8, 700, 5), (128, 4, 1, 129, 36), (128, 4, 11, 1031, 4),
                                             (256, 2, 3, 512, 20), (256, 4, 17, 33, 3), (256, 4, 2, 2049, 4), (256, 8, 5, 128, 6),
                                             (256, 8, 1, 1200, 34), (512, 2, 3, 65, 5), (512, 4, 9, 200, 3), (512, 8, 2, 1500, 4)])
def test_parts_equal_one_workgroup_and_step_by_step(device, tuning, dtype, backend, D, parts, B, Nc, Nt):
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    if D == 512 and dtype == torch.float32:
        pytest.skip("no whole-run kernel of this width in float32")
    torch.manual_seed(3)
    model = ARTabPFN(d_model=D, n_heads=D // 32, n_layers=3, d_ff=256, num_features=2, buffer_size=6, num_components=4)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if "norm" in name or name.endswith("bias"):
                p.add_(0.1 * torch.randn_like(p))
        # components that overlap: a draw on the boundary between two of them moves little
        model.head.head[2].weight.mul_(0.02)
        model.head.mean_bias.mul_(0.02)
        model.head.head[2].bias.zero_()
        model.head.std_bias.fill_(math.log(math.expm1(0.5)))
    model = model.eval().to(device, dtype)
    g = torch.Generator().manual_seed(4)
    rows = 1 if backend == "triton_shared_context" else B
    xc = torch.randn(rows, Nc, 2, generator=g).expand(B, -1, -1).to(device, dtype)
    yc = torch.randn(rows, Nc, generator=g).expand(B, -1).to(device, dtype)
    xt = torch.randn(B, Nt, 2, generator=g).to(device, dtype)
    names = ("k_buf_cache", "v_buf_cache") if backend == "triton_shared_context" else ("k_cache", "v_cache")
    results = []
    for n in (parts, 1, 0):  # 0: step by step
        tuning(ARTAB_TRAJECTORY=min(n, 1), ARTAB_TRAJECTORY_PARTS=max(n, 1))
        pred = ARTabPFNPredictor.from_trained_model(model, backend=backend)
        pred.whole_run_decode = n > 0
        for _ in range(2):  # (the second run finds the words of the first)
            torch.manual_seed(5)
            y = pred.sample_sequence(xc, yc, xt)
        assert (pred._trajectory is not None) == (n > 0) and torch.isfinite(y).all()
        results.append([y] + [getattr(l, name).clone() for l in model.backbone.layers for name in names])
    for other in results[1:]:
        for a, b in zip(results[0], other):
            assert _rel(a, b) <= TOL[dtype]


def _run(device, dtype, D, parts, B, Nc, Nt):
    """A call of the whole-run kernel on a model of its own with given variates, and its caches' tensors."""
    from ar_nanotabpfn_amd.glue import TrajectoryDecoder
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    torch.manual_seed(D + B)
    model = ARTabPFN(d_model=D, n_heads=D // 32, n_layers=2, d_ff=256, num_features=2, buffer_size=6, num_components=3).eval().to(device, dtype)
    pred = ARTabPFNPredictor.from_trained_model(model, backend="triton_shared_context")
    pred.init_kv_cache(B, Nt, torch.device(device), dtype)
    pred.prefill_context(torch.randn(1, Nc, 2, device=device, dtype=dtype).expand(B, -1, -1), torch.randn(1, Nc, device=device, dtype=dtype).expand(B, -1))
    run = TrajectoryDecoder(pred.embedder, pred.backbone, pred.head, pred.ar_tokens)
    caches = [(l.k_ctx_cache, l.v_ctx_cache, l.k_buf_cache, l.v_buf_cache) for l in pred.backbone.layers]
    x = torch.randn(B, Nt, device=device, dtype=dtype)
    u, n = torch.rand(Nt, B, device=device), torch.randn(Nt, B, device=device)
    return lambda k=parts: run(caches, Nc, 0, x, u, n, 1, k), [t for c in caches for t in c[2:]]


# (d_model 512: one workgroup to a trajectory is another kernel)
@pytest.mark.parametrize("dtype,D,parts,B,Nc,Nt", [(torch.bfloat16, 128, 4, 11, 70, 5), (torch.float16, 256, 2, 3, 33, 1), (torch.float32, 256, 8, 2, 129, 4),
                                                   (torch.bfloat16, 512, 8, 9, 40, 3)])
def test_trajectories_that_are_given_up(device, tuning, dtype, D, parts, B, Nc, Nt):
    """No second look for another workgroup's word: every trajectory is given up, and is what one workgroup makes of it."""
    call, own = _run(device, dtype, D, parts, B, Nc, Nt)
    want = call(1)
    rows = [t[:, :, : Nt - 1].clone() for t in own]
    for t in own:
        t.zero_()
    tuning(ARTAB_TRAJECTORY_POLLS=0)
    assert torch.equal(call(), want)
    assert all(torch.equal(t[:, :, : Nt - 1], r) for t, r in zip(own, rows))
    tuning(ARTAB_TRAJECTORY_POLLS=None)
    assert torch.isfinite(call()).all() and torch.equal(call(), call())


def test_runs_with_parts_on_two_streams(device):
    calls = [_run(device, torch.bfloat16, 256, parts, B, 300, 12)[0] for parts, B in ((8, 13), (4, 40))]
    want = [call() for call in calls]
    streams = [torch.cuda.Stream(device) for _ in calls]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(4):
        for call, stream, out in zip(calls, streams, got):
            with torch.cuda.stream(stream):
                out.append(call())
    torch.cuda.synchronize()
    for outs, w in zip(got, want):
        assert all(torch.equal(o, w) for o in outs)


def test_runs_with_parts_in_a_recorded_graph(device, tuning):
    """Replays, with other work and a synchronisation between them: the words are cleared by a launch that is recorded too."""
    from ar_nanotabpfn_amd.glue import TrajectoryDecoder
    from ar_nanotabpfn_amd.inference import ARTabPFNPredictor
    from ar_nanotabpfn_amd.model import ARTabPFN

    torch.manual_seed(1)
    model = ARTabPFN(d_model=128, n_heads=4, n_layers=2, d_ff=256, num_features=2, buffer_size=6, num_components=3).eval().to(device, torch.bfloat16)
    pred = ARTabPFNPredictor.from_trained_model(model, backend="triton_shared_context")
    B, Nc, Nt = 9, 70, 5
    pred.init_kv_cache(B, Nt, torch.device(device), torch.bfloat16)
    pred.prefill_context(torch.randn(1, Nc, 2, device=device, dtype=torch.bfloat16).expand(B, -1, -1),
                         torch.randn(1, Nc, device=device, dtype=torch.bfloat16).expand(B, -1))
    run = TrajectoryDecoder(pred.embedder, pred.backbone, pred.head, pred.ar_tokens)
    caches = [(l.k_ctx_cache, l.v_ctx_cache, l.k_buf_cache, l.v_buf_cache) for l in pred.backbone.layers]
    x = torch.randn(B, Nt, device=device, dtype=torch.bfloat16)
    u, n = torch.rand(Nt, B, device=device), torch.randn(Nt, B, device=device)
    call = lambda: run(caches, Nc, 0, x, u, n, 1, 4)  # noqa: E731
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for _ in range(3):
        u.uniform_()
        n.normal_()
        x.normal_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, call())
