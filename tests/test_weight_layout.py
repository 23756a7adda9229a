"""Weights at the row pitch the products read fastest: what the layout changes (strides only), and every flow of a layer
on such weights against the same flow on contiguous ones."""
import pytest
import torch

from aptserve_hip import backend, metadata, opt_model, workloads
from util import randn


def plain(cfg, seed, device, dtype=torch.float16):
    """Weights as a checkpoint holds them: every matrix contiguous, in memory of its own."""
    return {k: v.contiguous().clone() for k, v in opt_model.random_weights(cfg, seed, device, dtype=dtype).items()}


def test_lay_out_weights_changes_strides_and_nothing_else():
    cfg = opt_model.OPTConfig(1536, 24, 2, 3072, 64, 32)      # rows of 3 KiB (not a multiple of 2) and 6 KiB
    w = plain(cfg, 1, "cpu")
    before = dict(w)
    assert opt_model.lay_out_weights(w) is w
    for k, v in w.items():
        assert torch.equal(v, before[k]) and v.shape == before[k].shape and v.stride(-1) == 1
        if k.endswith("fc2_w"):
            assert v.stride(0) * 2 == 6 * 1024 + 128
        else:
            assert v is before[k]
    again = dict(w)
    opt_model.lay_out_weights(w)
    assert all(w[k] is again[k] for k in w)
    for k, v in opt_model.random_weights(cfg, 1, "cpu").items():   # the generator lays its matrices out the same way
        assert v.stride() == w[k].stride() and torch.equal(v, w[k])


@pytest.mark.parametrize("k,dtype,pitch", [(768, torch.float16, 768), (1024, torch.float16, 1024), (2048, torch.bfloat16, 2048),
                                           (8192, torch.float16, 8192), (3072, torch.float16, 3136), (5120, torch.bfloat16, 5184),
                                           (20480, torch.float16, 20544), (1536, torch.float32, 1568)])
def test_row_pitch(k, dtype, pitch):
    """128 bytes more for rows of a multiple of 2 KiB, unless that is a power of two (those are as fast as they are)."""
    m = opt_model.row_pitched(3, k, dtype, "cpu")
    assert m.shape == (3, k) and m.stride() == (pitch, 1) and m.dtype == dtype


@pytest.mark.gpu
@pytest.mark.parametrize("absorbed", [False, True])
@pytest.mark.parametrize("prompt,seqs,longest", [(False, 5, 90), (False, 60, 60), (True, 3, 12), (True, 8, 90)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_layer_flows_on_laid_out_weights(dev, absorbed, prompt, seqs, longest, dtype):
    """Projections of few and many rows, the gathered re-projection, the absorbed queries and the head-wise value
    projection on rows 128 bytes further apart (6 and 12 KiB) than on contiguous ones: the same sums in another order,
    so the tolerance of a layer between two such orders."""
    cfg = opt_model.OPTConfig(3072, 24, 1, 6144, 100, 256)
    N = 512
    make = workloads.small_prefill_batch if prompt else workloads.small_decode_batch
    batch = make(seqs, seqs, longest, 0.5, N)
    md = metadata.build_from_batch(batch, dev)
    rows = sum(batch.seq_lens) if prompt else seqs
    ids = torch.arange(rows, device=dev) % 100
    w = plain(cfg, 2, dev, dtype)
    laid = opt_model.lay_out_weights(dict(w))
    assert all(laid["layers.0." + k].stride(0) == w["layers.0." + k].stride(0) + 64 for k in ("qkv_w", "out_w", "fc1_w", "fc2_w"))
    outs = []
    for weights in (w, laid):
        kv, shared = backend.allocate_caches(1, N, 16, 24, 128, dtype, dev)
        kv[0].copy_(randn(tuple(kv[0].shape), 9, dtype).to(dev))
        model = opt_model.HybridOPTModel(cfg, weights, absorbed=absorbed)
        outs.append((model(ids, md.input_positions, kv, shared, md).float(), kv[0].float()))
    tol = 2.7e-3 if dtype == torch.float16 else 2.2e-2
    for a, b in zip(*outs):
        assert torch.isfinite(a).all() and ((a - b).norm() / a.norm()).item() <= tol
