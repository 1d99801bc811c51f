"""Host-side logic of the layer modules that needs no GPU: when the bf16 weight copies the kernels read are made anew,
and loading a checkpoint that carries TransformerEngine's per-module `_extra_state` entries."""
import pytest
import torch

from flash3dtransformer_amd import layers as L
from flash3dtransformer_amd.layers import nn_ops


def test_bf16_weight_copy_follows_the_parameter():
    lin = L.Linear(8, 4)
    w0 = lin._w.get(lin.weight, lin.training)
    # training mode or enabled gradients: every call casts again, so an edit through .data is seen at once
    lin.weight.data.mul_(0)
    assert lin._w.get(lin.weight, lin.training).abs().max().item() == 0 and w0.abs().max().item() > 0
    lin.weight.data.normal_()
    lin.eval()
    with torch.no_grad():
        a = lin._w.get(lin.weight, lin.training)
        assert lin._w.get(lin.weight, lin.training) is a                 # kept between eval-mode forwards
        lin.weight.mul_(2.0)                                             # ordinary in-place edit: version moves
        b = lin._w.get(lin.weight, lin.training)
        assert b is not a and torch.equal(b, lin.weight.to(torch.bfloat16))
        lin.weight.data.zero_()                                          # through .data: invisible ...
        assert lin._w.get(lin.weight, lin.training) is b
        L.refresh_weights(lin)                                           # ... until the copies are dropped
        assert lin._w.get(lin.weight, lin.training).abs().max().item() == 0
        lin.weight.data.fill_(1.0)
        lin.eval()                                                       # a mode call drops them too
        assert lin._w.get(lin.weight, lin.training).min().item() == 1.0
    # a bf16 parameter is handed over itself
    lin16 = L.Linear(8, 4).to(torch.bfloat16).eval()
    with torch.no_grad():
        assert lin16._w.get(lin16.weight, False).data_ptr() == lin16.weight.data_ptr()


def test_load_state_dict_drops_copies_and_accepts_extra_state():
    mlp = L.LayerNormMLP(32, 64).eval()
    with torch.no_grad():
        old = mlp._c[2].get(mlp.fc1_weight, False)
        sd = {k: torch.zeros_like(v) for k, v in mlp.state_dict().items()}
        sd["_extra_state"] = None           # what te.LayerNormMLP stores beside its parameters
        mlp.load_state_dict(sd, strict=True)
        new = mlp._c[2].get(mlp.fc1_weight, False)
    assert new.abs().max().item() == 0 and old.abs().max().item() > 0
    # nested: the reference's MLP wrapper holds te.LayerNormMLP as `.mlp`, te.Linear as the leaf `.proj`
    blk = L.MLP(32, 64)
    sd = dict(blk.state_dict())
    sd["mlp._extra_state"] = torch.zeros(1)
    blk.load_state_dict(sd, strict=True)
    lin = L.Linear(8, 4)
    sd = dict(lin.state_dict())
    sd["_extra_state"] = None
    lin.load_state_dict(sd, strict=True)
    assert isinstance(lin, nn_ops._CachedParamModule)


def test_planner_tables_cover_every_bucket_and_say_so():
    """every plan of bucket_scope.py puts each bucket of the buffer into exactly one scope (reference:
    flash3dxfmr/psh/bucket_scope.py:58-82); the cached table carries that fact for ops that write only covered rows"""
    from flash3dtransformer_amd.psh.bucket_scope import SwinPlan
    for plan, total, bs, sc in (("swin", 8192, 512, 1), ("swin", 16384, 512, 8), ("swin", 5 * 512, 512, 2),
                                ("stride", 12 * 256, 256, 2)):
        import warnings
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")
            t = SwinPlan(plan, bs, sc, 0 if plan == "swin" else 1).gen_scopes_from_plan(total, torch.device("cpu"))
        assert getattr(t, "covers_all_rows", False)
        ids = t.view(torch.int32).flatten().tolist()
        assert sorted(ids) == list(range(total // bs))


def test_layernorm_qkv_of_a_rank4_embedding_folds_to_four_numbers_per_feature():
    """The identity behind the first block's attention kernel that forms Q, K, V from coordinates (float64, no GPU):
    for x = E c with c = (x, y, z, 1),  W (gamma * (x - mean x) / sqrt(var x + eps) + beta) + b
    = rstd (M c) + b'  with  M = W diag(gamma) E',  b' = W beta + b,  rstd = 1 / sqrt(|L c|^2 + eps),
    E' = E minus its column means and L the upper Cholesky factor of E'^T E' / C -- checked against LayerNorm and the
    two linear layers evaluated as the reference's module sequence writes them (psh_ops.py:64-68, stage.py:94-96)."""
    import torch
    g = torch.Generator().manual_seed(3)
    C, N, eps = 96, 500, 1e-5
    rnd = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64)
    ew, eb, gamma, beta, w, b = rnd(C, 3), rnd(C), 1 + 0.2 * rnd(C), 0.3 * rnd(C), rnd(3 * C, C) / C ** 0.5, rnd(3 * C)
    c3 = rnd(N, 3) * torch.tensor([40.0, 40.0, 3.0], dtype=torch.float64)
    x = torch.nn.functional.linear(c3, ew, eb)
    want = torch.nn.functional.linear(torch.nn.functional.layer_norm(x, (C,), gamma, beta, eps), w, b)
    E = torch.cat([ew, eb[:, None]], 1)
    Ep = E - E.mean(0, keepdim=True)
    L = torch.linalg.cholesky(Ep.T @ Ep / C).T
    M, bp = (w * gamma[None, :]) @ Ep, w @ beta + b
    c = torch.cat([c3, torch.ones(N, 1, dtype=torch.float64)], 1)
    rstd = 1.0 / torch.sqrt((c @ L.T).pow(2).sum(1, keepdim=True) + eps)
    got = rstd * (c @ M.T) + bp
    assert (got - want).abs().max().item() <= 1e-9 * max(1.0, want.abs().max().item())
    # a dropped mean, a missing gamma or the uncentred Gram matrix are not the same function
    assert ((rstd * (c @ ((w * gamma[None, :]) @ E).T) + bp) - want).abs().max().item() > 1e-3
    assert ((rstd * (c @ (w @ Ep).T) + bp) - want).abs().max().item() > 1e-3


def test_layers_keep_one_buffer_of_prepared_weights():
    """only the kernel with the LayerNorm inside prepares weights: one buffer a layer, the second linear of an MLP has none"""
    for layer in (L.Linear(512, 512), L.LayerNormMLP(512, 2048), L.LayerNormMLP(128, 512, activation="gelu")):
        assert sum(isinstance(c, nn_ops._StagedWeights) for c in layer._bf16_caches()) == 1


def _pool_buffers(n, tail=0):
    from flash3dtransformer_amd.psh import subbuck
    seps = torch.tensor([3, n], dtype=torch.int32)
    coords, feat = torch.zeros(n + tail, 3, dtype=torch.float16), torch.zeros(n + tail, 8, dtype=torch.bfloat16)
    return seps, lambda **kw: subbuck.SubbuckBuffers.create_subbuck_buff(coords, feat, seps, 2, out_alignment=16, **kw)


def test_pooling_buffers_cover_rows_only_once_built():
    """a map nobody has filled has no slot for any row: gradients start from zero, and so do the point ids"""
    from flash3dtransformer_amd.psh import subbuck
    for _ in range(3):      # memory that is handed out again holds something
        seps, make = _pool_buffers(4001)
        junk = [torch.full((4001, 8), 7.0).to(torch.bfloat16), torch.full((4001,), 7, dtype=torch.int32)]
        del junk
        sb = make()
        assert not sb.covers(4001) and not sb.subbuck_id.view(torch.int32).any()
        grads = subbuck.UnpoolGradients.create_unpool_grad(torch.ones(4001, 8, dtype=torch.bfloat16), sb, 2016)
        assert not grads.grad_res.any() and not grads.grad_down[sb.unpool_ind.shape[0]:].any()
    sb.mark_built(seps, 4001)
    assert sb.covers(4001) and not sb.covers(4000)
    sb.unpool_ind.view(torch.int32).add_(1)             # changed since
    assert not sb.covers(4001)
    seps, make = _pool_buffers(4001, tail=5)            # rows behind the last cloud
    sb = make(build_follows=True)
    sb.mark_built(seps, 4006)
    assert not sb.covers(4006) and not sb.subbuck_id.view(torch.int32).any()


def test_pooling_buffers_are_prefilled_unless_the_builder_fills_them():
    """a caller who runs the builder without `fill` finds the marker of an empty slot in the whole map, and the box set"""
    for how in ({}, dict(build_follows=True)):
        for _ in range(3):      # memory that is handed out again holds something
            junk = [torch.full((2002, 2), 7, dtype=torch.int32), torch.zeros(3, dtype=torch.float16), torch.zeros(3, dtype=torch.float16)]
            del junk
            sb = _pool_buffers(4001)[1](**how)
            assert (sb.unpool_ind.view(torch.int32) == 4004).all() and sb.unpool_ind.shape == (2001, 2)
            assert sb.bbox_min.tolist() == [-65504.0] * 3 and sb.bbox_max.tolist() == [65504.0] * 3


def test_pooling_buffers_in_inference_mode():
    """tensors made there keep no version counter; separators seen before stay usable"""
    from flash3dtransformer_amd.psh import batching
    seps, make = _pool_buffers(40)
    make()
    batching.host_sizes(seps)
    with torch.inference_mode():
        for how in ({}, dict(build_follows=True)):
            sb = make(**how)
            sb.mark_built(seps, 40)
            assert not sb.covers(40) and sb.unpool_ind.shape == (21, 2)


@pytest.mark.parametrize("made_in_inference_mode", [False, True])
def test_separators_in_inference_mode(made_in_inference_mode):
    """sizes, padded separators and pooled ones of a first call there; what is derived from them has a version and is remembered"""
    from flash3dtransformer_amd.psh import batching, subbuck
    with torch.inference_mode(made_in_inference_mode):
        seps = torch.tensor([3, 40], dtype=torch.int32)
    with torch.inference_mode():
        assert batching.host_sizes(seps) == [3, 37] and batching.max_inslen_from_seps(seps) == 37
        padded = batching.with_last_separator(seps, 48)
        assert padded.tolist() == [3, 48] and batching.host_sizes(padded) == [3, 45]
        rows, sizes, cum = subbuck.calc_red_sep_sizes(padded, 2)
        assert rows == 25 and sizes.tolist() == [2, 23] and cum.tolist() == [2, 25]
        assert subbuck.calc_red_sep_sizes(padded, 2)[2] is cum and batching.host_facts(cum)["sizes"] == [2, 23]
        assert (batching.with_last_separator(seps, 48) is padded) == (not made_in_inference_mode)
        if made_in_inference_mode:      # a change leaves no trace, so sizes are read again
            seps[1] = 44
            assert batching.host_sizes(seps) == [3, 41]
    seps2 = torch.tensor([5], dtype=torch.int32)
    assert batching.host_facts(seps2) is batching.host_facts(seps2)


def test_weight_copies_made_in_inference_mode_have_a_version():
    cache, p = nn_ops._Bf16Cache(), torch.nn.Parameter(torch.ones(4))
    with torch.inference_mode():
        copy = cache.get(p)
    with torch.no_grad():
        assert copy._version == 0 and cache.get(p) is copy
        p.add_(1.0)
        assert cache.get(p).tolist() == [2.0] * 4


def test_block_pickled_without_the_drivers_cache(monkeypatch):
    """the state of a block from before there was one; its first inference call makes it"""
    import pickle
    from flash3dtransformer_amd.lib import pshattn
    from flash3dtransformer_amd.psh.bucket_scope import SwinPlan

    class Driver:
        class WeightCache:
            pass

        def block_infer(self, cache, x, *rest):
            return (type(cache).__name__, x)
    monkeypatch.setattr(pshattn, "_host", Driver())
    plan = SwinPlan("swin", 512, 1, 0)
    blk = L.XFMR(64, 256, 2, 512, True, plan, L.LayerNorm).eval()
    del blk.__dict__["_host"]
    old = pickle.loads(pickle.dumps(blk))
    assert "_host" not in old.__dict__
    x = torch.zeros(512, 64, dtype=torch.bfloat16)
    for _ in range(2):
        assert old._whole_block(x, plan.gen_scopes_from_plan(512, "cpu"))[0] == "WeightCache"


def test_extra_state_of_a_subclass_is_loaded():
    """layers drop the entry TransformerEngine's modules store, but not that of a subclass that has one of its own"""
    from flash3dtransformer_amd.psh.bucket_scope import SwinPlan

    class Counting(L.XFMR):
        steps = 0

        def get_extra_state(self):
            return {"steps": self.steps}

        def set_extra_state(self, state):
            self.steps = state["steps"]
    make = lambda: Counting(32, 64, 1, 512, True, SwinPlan("swin", 512, 1, 0), L.LayerNorm)
    a, b = make(), make()
    a.steps = 5
    b.load_state_dict(a.state_dict())
    assert b.steps == 5
