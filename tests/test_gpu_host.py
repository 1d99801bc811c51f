"""The native driver of the layers against the layers' own Python code: the same kernels in the same order on the same
operands, so every output and gradient is compared bit for bit."""
import copy
import gc

import pytest
import torch
from torch import nn

from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu


class _Declines:
    """a driver that takes no call: the layers run their Python code"""
    class WeightCache:
        def clear(self):
            pass

    def __getattr__(self, name):
        return lambda *a: None


@pytest.fixture
def python_path(monkeypatch):
    from flash3dtransformer_amd.lib import pshattn

    def run(f):
        with monkeypatch.context() as m:
            m.setattr(pshattn, "_host", _Declines())
            return f()
    return run


def _same(a, b):
    assert type(a) is type(b)
    if isinstance(a, torch.Tensor):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)
    elif isinstance(a, (list, tuple)):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            _same(x, y)
    else:
        assert a == b


def _step(module, call, x, grad_seed=3):
    """output, dx and every parameter's gradient of one step"""
    x = x.detach().clone().requires_grad_()
    module.zero_grad(set_to_none=True)
    y = call(x)
    g = torch.randn(y.shape, generator=torch.Generator(device=DEV).manual_seed(grad_seed), device=DEV).to(y.dtype)
    y.backward(g)
    return [y.detach(), x.grad] + [p.grad for p in module.parameters() if p.requires_grad]


@pytest.mark.parametrize("rows,k,n,bias,norm,residual,form", [
    (1, 32, 8, True, True, False, "2d"), (33, 64, 192, True, True, False, "3d"), (1000, 256, 256, True, False, True, "3d"),
    (257, 512, 1536, False, True, False, "2d"), (515, 40, 24, True, False, False, "2d"), (300, 128, 64, True, False, True, "columns"),
    (96, 96, 32, False, False, False, "frozen weight"),
])
def test_linear_training_step(rows, k, n, bias, norm, residual, form, python_path):
    from flash3dtransformer_amd import layers as L
    torch.manual_seed(rows + k)
    lin = L.Linear(k, n, bias=bias)
    both = nn.ModuleList([lin] + ([L.LayerNorm(k)] if norm else [])).to(DEV)
    if form == "frozen weight":
        lin.weight.requires_grad_(False)
    x = torch.randn(rows, 2 * k if form == "columns" else k, device=DEV).to(torch.bfloat16)
    res = torch.randn(rows, n, device=DEV).to(torch.bfloat16).requires_grad_() if residual else None

    def call(t):
        if form == "3d":
            return lin(t.view(1, rows, k), residual=None if res is None else res.view(1, rows, n), pre_norm=both[1] if norm else None)
        return lin(t[:, k:] if form == "columns" else t, residual=res, pre_norm=both[1] if norm else None)

    def run():
        if res is not None:
            res.grad = None
        return _step(both, call, x) + ([res.grad] if res is not None else [])
    _same(run(), python_path(run))


@pytest.mark.parametrize("rows,k,n", [(1, 32, 96), (33, 64, 8), (257, 128, 384), (515, 256, 768), (70, 512, 64)])
def test_input_that_is_used_twice(rows, k, n, python_path):
    """Linear.forked against the layer and its input used by themselves, their two gradients added by autograd"""
    from flash3dtransformer_amd import layers as L
    torch.manual_seed(rows)
    both = nn.ModuleList([L.Linear(k, n), L.LayerNorm(k)]).to(DEV)
    x = torch.randn(rows, k, device=DEV).to(torch.bfloat16)
    scale = torch.randn(rows, k, device=DEV).to(torch.bfloat16)

    def run(forked):
        def call(t):
            y, again = both[0].forked(t, both[1]) if forked else (both[0](t, pre_norm=both[1]), t)
            return torch.cat([y, again * scale], dim=1)
        return _step(both, call, x)
    _same(run(True), python_path(lambda: run(False)))
    hooked = []
    both[0].register_forward_hook(lambda *a: hooked.append(1))
    run(False)
    assert hooked


@pytest.mark.parametrize("rows,c,hid,own_residual", [(1, 32, 128, True), (333, 64, 256, True), (130, 128, 96, False), (700, 256, 1024, True),
                                                     (65, 512, 2048, None)])
def test_mlp_training_step(rows, c, hid, own_residual, python_path):
    from flash3dtransformer_amd import layers as L
    torch.manual_seed(c)
    mlp = L.LayerNormMLP(c, hid).to(DEV)
    x = torch.randn(rows, c, device=DEV).to(torch.bfloat16)
    other = torch.randn(rows, c, device=DEV).to(torch.bfloat16).requires_grad_()

    def run():
        other.grad = None
        got = _step(mlp, lambda t: mlp(t, None if own_residual is None else t if own_residual else other), x)
        return got + ([other.grad] if own_residual is False else [])
    _same(run(), python_path(run))


@pytest.mark.parametrize("c,heads,scope,rows,whole", [(64, 2, 1, 1536, True), (32, 2, 2, 2048, True), (128, 2, 1, 1024, False),
                                                        (256, 8, 1, 512, True), (512, 16, 1, 512, True)])
def test_block_training_step(c, heads, scope, rows, whole, python_path):
    """whole: a table that covers all rows, as a plan makes it; otherwise a table of the first bucket alone"""
    from flash3dtransformer_amd import layers as L
    from flash3dtransformer_amd.psh.bucket_scope import SwinPlan
    torch.manual_seed(c + scope)
    blk = L.XFMR(c, 4 * c, heads, 512, True, SwinPlan("swin", 512, scope, 0), lambda ch: L.LayerNorm(ch)).to(DEV)
    x = torch.randn(rows, c, device=DEV).to(torch.bfloat16)
    if whole:
        run = lambda: _step(blk, lambda t: blk(None, t, None), x)
    else:
        table = torch.zeros(1, 1, dtype=torch.int32, device=DEV).view(torch.uint32)
        run = lambda: _step(blk, lambda t: blk.bwa(t.view(1, rows, c), table, skip_proj=True)[:, :512], x)
    _same(run(), python_path(run))


@pytest.mark.parametrize("c,heads,rows,scope", [(32, 1, 512, 1), (64, 2, 4096, 8), (128, 4, 1024, 1), (256, 8, 1536, 1), (256, 8, 30208, 1),
                                                (512, 16, 1024, 2)])
def test_block_inference(c, heads, rows, scope, python_path):
    """equal bits; a changed, replaced or refreshed parameter shows; hooks and other classes take the Python code"""
    from flash3dtransformer_amd import layers as L
    from flash3dtransformer_amd.psh.bucket_scope import SwinPlan
    torch.manual_seed(c)
    blk = L.XFMR(c, 4 * c, heads, 512, True, SwinPlan("swin", 512, scope, 0), lambda ch: L.LayerNorm(ch)).to(DEV).eval()
    x = torch.randn(rows, c, device=DEV).to(torch.bfloat16)
    wide = torch.randn(rows, c + 8, device=DEV).to(torch.bfloat16)
    run = lambda t=x: blk(None, t, None)
    with torch.no_grad():
        first = run()
        _same(first, python_path(run))
        _same(run(), first)
        _same(run(wide[:, :c]), python_path(lambda: run(wide[:, :c])))
        blk.mlp.mlp.fc1_weight.mul_(1.5)
        blk.norm.bias.add_(0.25)
        changed = run()
        assert not torch.equal(changed, first)
        _same(changed, python_path(run))
        blk.bwa.proj.bias.data.add_(1.0)      # leaves address and version alone
        L.refresh_weights(blk.bwa)
        refreshed = run()
        assert not torch.equal(refreshed, changed)
        _same(refreshed, python_path(run))
        twin = copy.deepcopy(blk)
        _same(twin(None, x, None), refreshed)
        seen = []
        handle = blk.bwa.register_forward_hook(lambda m, i, o: seen.append(o.shape))
        _same(run(), refreshed)
        assert seen
        handle.remove()
        blk.to(torch.bfloat16)
        _same(run(), python_path(run))
        blk.train()
        _same(run(), python_path(run))


def _fresh_block(c, heads):
    """an inference block whose driver has prepared nothing yet, behind freed memory that reads as NaN"""
    from flash3dtransformer_amd import layers as L
    from flash3dtransformer_amd.psh.bucket_scope import SwinPlan
    torch.manual_seed(c)
    blk = L.XFMR(c, 4 * c, heads, 512, True, SwinPlan("swin", 512, 1, 0), lambda ch: L.LayerNorm(ch)).to(DEV).eval()
    junk = [torch.full((3 * n * c * c + 4 * n * c + 2 * c + 512,), 255, dtype=torch.uint8, device=DEV) for n in (3, 8) for _ in range(2)]
    del junk
    return blk


@pytest.mark.parametrize("c,heads", [(64, 2), (256, 8), (512, 16)])
def test_block_after_a_call_that_was_refused(c, heads, python_path):
    """an input off 16 bytes raises before anything is prepared; the next call prepares"""
    blk = _fresh_block(c, heads)
    x, wide = [torch.randn(1024, w, device=DEV).to(torch.bfloat16) for w in (c, c + 8)]
    with torch.no_grad():
        with pytest.raises(RuntimeError, match="16-byte"):
            blk(None, wide[:, 1:1 + c], None)
        got = blk(None, x, None)
        _same(got, python_path(lambda: blk(None, x, None)))


def test_block_after_a_call_that_ran_out_of_memory(python_path):
    """the hidden activations (268 MB at 65,536 rows), last and largest, do not fit; a smaller call prepares the MLP's weights"""
    blk = _fresh_block(512, 16)
    rows, x = 65536, torch.randn(1024, 512, device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        big = torch.zeros(rows, 512, dtype=torch.bfloat16, device=DEV)
        torch.cuda.synchronize()
        gc.collect()
        torch.cuda.empty_cache()
        room = rows * (3 * 512 * 2 + 3 * 512 * 2 + 16 * 4) + (64 << 20)      # qkv; o, mid, y; lse; weight copies
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_allocated() + room) / total)      # the call needs 200 MB more
        try:
            with pytest.raises(torch.cuda.OutOfMemoryError):
                blk(None, big, None)
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert blk._host._native is not None
        got = blk(None, x, None)
        _same(got, python_path(lambda: blk(None, x, None)))


@pytest.mark.parametrize("c,heads,rows", [(32, 1, 1024), (256, 8, 1536), (512, 16, 512)])
def test_block_in_inference_mode(c, heads, rows, monkeypatch):
    """the driver takes the block there as under no_grad, cold and warm, with equal bits; copies made there serve later calls"""
    from flash3dtransformer_amd.lib import pshattn
    taken = []

    class Spy:
        def __getattr__(self, name):
            f = getattr(native, name)
            return f if name == "WeightCache" else lambda *a: (lambda r: (taken.append((name, r is not None)), r)[1])(f(*a))
    native = pshattn.host()
    monkeypatch.setattr(pshattn, "_host", Spy())
    blk, twin = _fresh_block(c, heads), _fresh_block(c, heads)
    x = torch.randn(rows, c, device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        want = twin(None, x, None)
    with torch.inference_mode():
        for t in (x, x.clone(), x.clone()):
            _same(blk(None, t, None).clone(), want)
    with torch.no_grad():
        _same(blk(None, x, None), want)
        blk.mlp.mlp.fc2_bias.add_(1.0)
        twin.mlp.mlp.fc2_bias.add_(1.0)
        _same(blk(None, x, None), twin(None, x, None))
    assert taken and all(t == ("block_infer", True) for t in taken)


def test_attention_outside_the_kernels_is_told_apart():
    from flash3dtransformer_amd.layers.buck_swin import BucketSwinAttentionModule
    m = BucketSwinAttentionModule(48, 2, 512).to(DEV)      # 24-wide heads
    table = torch.zeros(1, 1, dtype=torch.int32, device=DEV).view(torch.uint32)
    with pytest.raises(RuntimeError, match="head_dim"):
        m(torch.zeros(1, 512, 48, dtype=torch.bfloat16, device=DEV), table)


@pytest.mark.parametrize("rows,k,n,residual", [(1, 64, 8, False), (2049, 32, 64, True), (300, 136, 72, False)])
def test_linear_inference(rows, k, n, residual, python_path):
    from flash3dtransformer_amd import layers as L
    torch.manual_seed(rows)
    lin = L.Linear(k, n).to(DEV).eval()
    x = torch.randn(rows, k, device=DEV).to(torch.bfloat16)
    res = torch.randn(rows, n, device=DEV).to(torch.bfloat16) if residual else None
    with torch.no_grad():
        run = lambda: [lin(x, residual=res), lin(x.view(1, rows, k)), lin(x.float())]
        _same(run(), python_path(run))


@pytest.mark.parametrize("training", [False, True])
def test_linear_inference_copies_its_parameters_once(training, monkeypatch):
    """also for an input that the driver declines"""
    from flash3dtransformer_amd import layers as L
    from flash3dtransformer_amd.layers import nn_ops
    asked, get = [], nn_ops._Bf16Cache.get
    monkeypatch.setattr(nn_ops._Bf16Cache, "get", lambda self, p, t=False: (asked.append(p), get(self, p, t))[1])
    lin = L.Linear(64, 32).to(DEV).train(training)
    x = torch.randn(40, 64, device=DEV)
    with torch.no_grad():
        want = lin(x.to(torch.bfloat16))
        asked.clear()
        assert torch.equal(lin(x), want)
    assert len(asked) == 2


@pytest.mark.parametrize("layout", ["one row for all", "columns of 67", "columns at 3"])
@pytest.mark.parametrize("kind", ["linear", "norm_linear", "residual_linear", "mlp", "norm", "block", "no dx", "embedding"])
def test_gradients_in_any_layout(kind, layout, python_path):
    """what autograd hands to a layer's backward behind a sum over the rows or a concatenation of columns: an expanded row, rows at
    an odd stride, rows off 16 bytes.  The gradients of the same values in a tensor of their own, by either path"""
    from flash3dtransformer_amd import layers as L
    from flash3dtransformer_amd.psh.bucket_scope import SwinPlan
    torch.manual_seed(7)
    C, rows = 64, 512
    lin, norm, mlp = L.Linear(C, C).to(DEV), L.LayerNorm(C).to(DEV), L.LayerNormMLP(C, 2 * C).to(DEV)
    blk = L.XFMR(C, 4 * C, 2, 512, True, SwinPlan("swin", 512, 1, 0), lambda ch: L.LayerNorm(ch)).to(DEV)
    emb, seps = L.PSH3DCoordEmbedding(C, 16, rows).to(DEV), torch.tensor([rows], dtype=torch.int32, device=DEV).view(torch.uint32)
    coords = torch.rand(rows, 3, device=DEV).half()
    module, call = {"embedding": (emb, lambda t: emb(coords, seps, 1)), "linear": (lin, lin), "norm_linear": (nn.ModuleList([lin, norm]), lambda t: lin(t, pre_norm=norm)),
                    "residual_linear": (lin, lambda t: lin(t, residual=t)), "mlp": (mlp, lambda t: mlp(t, residual=t)), "norm": (norm, norm),
                    "block": (blk, lambda t: blk(None, t, None)), "no dx": (lin, lambda t: lin(t.detach()))}[kind]
    x = torch.randn(rows, C, device=DEV).to(torch.bfloat16)
    wide = torch.randn(rows, C + 3, device=DEV).to(torch.bfloat16)
    g = {"one row for all": wide[0, :C].expand(rows, C), "columns of 67": wide[:, :C], "columns at 3": wide[:, 3:]}[layout]

    def step(grad):
        t = x.clone().requires_grad_()
        module.zero_grad(set_to_none=True)
        call(t).backward(grad)
        return ([] if kind in ("no dx", "embedding") else [t.grad]) + [p.grad for p in module.parameters()]
    want = step(g.contiguous())
    _same(step(g), want)
    _same(python_path(lambda: step(g)), python_path(lambda: step(g.contiguous())))


def test_layers_without_columns_raise():
    """no output columns, or no input columns, beside a residual: an error, in training and in inference"""
    from flash3dtransformer_amd import layers as L
    from flash3dtransformer_amd.lib import pshattn
    lin = L.Linear(64, 0).to(DEV)
    x, res = torch.zeros(5, 64, dtype=torch.bfloat16, device=DEV), torch.zeros(5, 0, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError):
        lin(x.requires_grad_(), residual=res)
    with torch.no_grad(), pytest.raises(RuntimeError):
        lin(x, residual=res)
    nothing = torch.zeros(5, 0, dtype=torch.bfloat16, device=DEV, requires_grad=True)
    assert pshattn.host().linear_train(nothing, torch.zeros(8, 0, device=DEV), None, torch.zeros(5, 8, dtype=torch.bfloat16, device=DEV), None,
                                       None, 0.0) is None


def test_saved_tensor_hooks_and_in_place_changes_are_seen():
    """the native nodes save through autograd: pack hooks run, and a weight changed between forward and backward is refused"""
    from flash3dtransformer_amd import layers as L
    lin = L.Linear(64, 64).to(DEV)
    mlp = L.LayerNormMLP(64, 128).to(DEV)
    x = torch.randn(40, 64, device=DEV).to(torch.bfloat16).requires_grad_()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t)[1], lambda t: t):
        y = mlp(lin(x))
    assert len(packed) >= 10
    y.float().sum().backward()
    y = mlp(lin(x))
    with torch.no_grad():
        mlp.fc2_weight.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.float().sum().backward()
