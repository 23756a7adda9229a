"""Residual add + LayerNorm in one launch against the two-operator definition (add in the activation dtype, then
LayerNorm with fp32 statistics): the pair ``hidden_states = residual + hidden_states`` / ``nn.LayerNorm`` of
additional_designs/model_executor/models/aptserve_opt.py:186-211.  The sum must be bit-exact (one rounding of an
exact fp32 sum); the normalised rows may differ from the fp32 oracle by the final rounding."""
import pytest
import torch
import torch.nn.functional as F

from aptserve_hip import ops
from util import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,width", [(1, 8), (5, 768), (7, 5120), (256, 5120), (3, 16384), (2, 1000),
                                        # on both sides of where a thread takes one vector more
                                        (3, 2048), (3, 2056), (3, 4096), (3, 4104), (3, 6144), (3, 6152), (3, 8192), (3, 8200)])
def test_add_layer_norm_matches_the_two_operator_definition(dev, dtype, rows, width):
    x, r = randn((rows, width), 1, dtype), (randn((rows, width), 2) * 3).to(dtype)
    w, b = (1 + 0.1 * randn((width,), 3)).to(dtype), (0.1 * randn((width,), 4)).to(dtype)
    s_ref = (x.float() + r.float()).to(dtype)
    n_ref = F.layer_norm(s_ref.float(), (width,), w.float(), b.float(), 1e-5)
    normed, s = ops.add_layer_norm(x.to(dev), r.to(dev), w.to(dev), b.to(dev))
    assert torch.equal(s.cpu().view(torch.int16), s_ref.view(torch.int16))
    ulp = 2 ** -10 if dtype == torch.float16 else 2 ** -7
    d = (normed.float().cpu() - n_ref).abs()
    assert (d <= ulp * n_ref.abs() + 1e-3).all(), d.max().item()
    # without a residual: the norm of x, and x itself comes back as the sum
    n2, s2 = ops.add_layer_norm(x.to(dev), None, w.to(dev), None)
    assert s2.data_ptr() == s2.data_ptr() and torch.equal(s2.cpu(), x)
    d2 = (n2.float().cpu() - F.layer_norm(x.float(), (width,), w.float(), None, 1e-5)).abs()
    assert d2.max().item() <= 4 * ulp + 1e-3


def test_add_layer_norm_strided_rows_and_errors(dev):
    wide = randn((6, 2 * 768), 5).to(dev)
    x, r = wide[:, :768], wide[:, 768:]                     # column slices: row stride twice the width
    w, b = torch.ones(768, dtype=torch.float16, device=dev), torch.zeros(768, dtype=torch.float16, device=dev)
    normed, s = ops.add_layer_norm(x, r, w, b)
    s_ref = (x.float() + r.float()).half()
    assert torch.equal(s, s_ref)
    assert torch.allclose(normed.float(), F.layer_norm(s_ref.float(), (768,)), atol=2e-3, rtol=2e-3)
    with pytest.raises(RuntimeError):
        ops.add_layer_norm(randn((2, 12), 1).to(dev), None, torch.ones(12, dtype=torch.float16, device=dev), None)
    with pytest.raises(ValueError):
        ops.add_layer_norm(x, r.float(), w, b)
    assert ops.add_layer_norm(x[:0], r[:0], w, b)[0].shape == (0, 768)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(1, 768, 768), (5, 5120, 20480), (12, 768, 3072), (48, 2560, 2048), (49, 768, 20480),
                                   (65, 5120, 5120), (361, 5120, 5120), (130, 7168, 4096), (700, 1024, 4096), (5, 2048, 2048),
                                   (5, 2304, 2304), (12, 4096, 4096), (12, 6144, 6144), (12, 8192, 8192), (12, 8448, 8448)])
def test_product_with_the_norm_behind_it_equals_the_two_calls(dev, m, n, k, dtype):
    """Products of one part, of few (the norm adds them) and of more than the norm adds; the same bits as linear_nt, then
    add_layer_norm.  With and without biases, and with a bias that no vector load takes."""
    x, w = randn((m, k), 1, dtype).to(dev), (randn((n, k), 2, dtype) * 0.02).to(dev)
    r, g = randn((m, 2 * n), 3, dtype).to(dev)[:, n:], (1 + 0.1 * randn((n,), 4)).to(dtype).to(dev)
    odd = randn((n + 1,), 5, dtype).to(dev)
    for bias, beta in ((odd[:n].clone(), odd[1:].clone()), (None, None), (odd[1:], None)):
        normed, total = ops.linear_add_layer_norm(x, w, bias, r, g, beta)
        ref_n, ref_t = ops.add_layer_norm(ops.linear_nt(x, w, bias), r, g, beta)
        assert torch.equal(total.view(torch.int16), ref_t.view(torch.int16))
        assert torch.equal(normed.view(torch.int16), ref_n.view(torch.int16))


@pytest.mark.parametrize("m,n,k,parts_left", [(1, 768, 768, False), (5, 5120, 20480, True), (12, 768, 3072, True),
                                              (48, 2560, 2560, True), (361, 5120, 5120, True), (130, 7168, 4096, True),
                                              (49, 768, 20480, False), (48, 2560, 10240, False), (4096, 768, 768, False)])
def test_which_products_leave_their_parts_to_the_norm(dev, m, n, k, parts_left):
    """A product whose parts the norm adds is never stored: its scratch keeps what was in it.  One of one part, of more than
    eight, or with a bias that no vector load takes is stored."""
    from aptserve_hip import _lib
    lib = _lib.load()
    x, w, r, g = randn((m, k), 1).to(dev), (randn((n, k), 2) * 0.02).to(dev), randn((m, n), 3).to(dev), randn((n,), 4).to(dev)
    odd = randn((n + 1,), 5).to(dev)
    need = lib.aps_linear_nt_workspace_bytes(m, n, k)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=dev)
    for bias in (None, odd[:n], odd[1:]):
        normed, total, product = (torch.full((m, n), float("nan"), dtype=torch.float16, device=dev) for _ in range(3))
        st = lib.aps_linear_add_layer_norm(
            normed.data_ptr(), total.data_ptr(), product.data_ptr(), x.data_ptr(), w.data_ptr(),
            None if bias is None else bias.data_ptr(), r.data_ptr(), g.data_ptr(), None, m, n, k, k, k, n, 1e-5, 0,
            ws.data_ptr(), need, ops._tile_counters(dev).data_ptr(), torch.cuda.current_stream(dev).cuda_stream)
        assert st == 0 and not normed.isnan().any() and not total.isnan().any()
        stored = not product.isnan().any().item()
        assert stored or product.isnan().all()
        assert stored == (not parts_left or bias is not None and bias.data_ptr() % 16 != 0)


def test_product_with_the_norm_behind_it_errors(dev):
    x, w = randn((3, 768), 1).to(dev), randn((768, 768), 2).to(dev)
    r, g = randn((3, 768), 3).to(dev), randn((768,), 4).to(dev)
    for bad in (dict(residual=r[:2]), dict(residual=r.float()), dict(ln_weight=None), dict(ln_weight=g[:5]), dict(x=x[:, :64])):
        with pytest.raises(ValueError):
            ops.linear_add_layer_norm(**{**dict(x=x, weight=w, bias=None, residual=r, ln_weight=g, ln_bias=None), **bad})
    assert ops.linear_add_layer_norm(x[:0], w, None, r[:0], g, None)[0].shape == (0, 768)


def test_decoder_with_fused_norms_equals_plain_ops(dev):
    """Two decoder layers with the (add, LayerNorm) pairs fused against the same model on plain element-wise ops:
    same kernels everywhere else, so the hidden states agree to the norms' last-bit differences."""
    from aptserve_hip import backend, metadata, opt_model, workloads
    cfg = opt_model.OPTConfig(hidden_size=768, num_attention_heads=12, num_hidden_layers=2, ffn_dim=1024,
                              vocab_size=500, max_position_embeddings=2048)
    w = opt_model.random_weights(cfg, 0, dev)
    N, BS = 96, 16
    batch = workloads.small_decode_batch(5, 9, 100, 0.5, N)
    md = metadata.build_from_batch(batch, dev)
    ids = torch.arange(len(batch.seq_lens), device=dev) % 500
    outs = []
    for fused in (True, False):
        kv, shared = backend.allocate_caches(2, N, BS, 12, 64, torch.float16, dev)
        for c in kv:
            c.copy_(randn(tuple(c.shape), 9).to(dev))
        model = opt_model.HybridOPTModel(cfg, w, fused_norm=fused)
        outs.append(model(ids, md.input_positions, kv, shared, md).float())
    assert (outs[0] - outs[1]).abs().max().item() < 2e-2


@pytest.mark.parametrize("place", ["attention", "attention of a subclass", "mlp of a layer", "mlp of a subclass"])
def test_decoder_with_fused_norms_calls_what_stands_in_for_its_parts(dev, monkeypatch, place):
    """An object that can only be called in place of a layer's attention, or another MLP, is called in every layer; one that
    calls what it replaces gives the same bits."""
    from aptserve_hip import backend, metadata, opt_model, workloads
    cfg = opt_model.OPTConfig(hidden_size=768, num_attention_heads=12, num_hidden_layers=2, ffn_dim=1024,
                              vocab_size=500, max_position_embeddings=2048)
    w = opt_model.random_weights(cfg, 0, dev)
    N, BS = 96, 16
    batch = workloads.small_decode_batch(5, 9, 100, 0.5, N)
    md = metadata.build_from_batch(batch, dev)
    ids = torch.arange(len(batch.seq_lens), device=dev) % 500
    calls, outs = [], []

    def counted(f):
        return lambda *args: calls.append(1) or f(*args)

    class Callable:
        def __init__(self, f):
            self.f = counted(f)

        def __call__(self, *args):
            return self.f(*args)

    class Attention(backend.HybridOPTAttention):
        def __call__(self, *args):
            return counted(self.forward)(*args)

    class Layer(opt_model.HybridOPTDecoderLayer):
        def _mlp(self, x):
            return counted(super()._mlp)(x)
    for replaced in (False, True):
        kv, shared = backend.allocate_caches(2, N, BS, 12, 64, torch.float16, dev)
        for c in kv:
            c.copy_(randn(tuple(c.shape), 9).to(dev))
        model = opt_model.HybridOPTModel(cfg, w)
        for layer in model.layers if replaced else ():
            if place == "attention":
                layer.self_attn = Callable(layer.self_attn)
            elif place == "attention of a subclass":
                layer.self_attn.__class__ = Attention
            elif place == "mlp of a layer":
                monkeypatch.setattr(layer, "_mlp", counted(layer._mlp))
            else:
                layer.__class__ = Layer
        outs.append(model(ids, md.input_positions, kv, shared, md))
    assert len(calls) == 2 and torch.equal(outs[0], outs[1])
