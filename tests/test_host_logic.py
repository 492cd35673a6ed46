"""CPU checks of host-side logic of the package (no GPU): RoPE tables and
weight-layout conversions that run before any kernel."""
import pytest
import torch


def test_gpt_oss_yarn_matches_hf(mk):
    """YaRN frequencies and attention scaling == transformers' "yarn" rope init for
    the GPT-OSS config (truncate=False)."""
    from transformers import GptOssConfig
    from transformers.modeling_rope_utils import ROPE_INIT_FUNCTIONS
    from nki_moe_megakernel_amd import gpt_oss_with_megakernel as G
    inv, sc = G.yarn_inv_freq(G.GptOssMKConfig())
    inv_hf, sc_hf = ROPE_INIT_FUNCTIONS["yarn"](GptOssConfig(head_dim=64), "cpu")
    torch.testing.assert_close(inv, inv_hf.float(), rtol=1e-6, atol=0)
    assert sc == pytest.approx(sc_hf, rel=1e-12)


def test_gpt_oss_converter_deinterleaves_and_folds_up_bias(mk):
    """HF gate_up [E, H, 2I] interleaved -> gate rows then up rows; up bias + 1;
    H zero-padded (gpt_oss_with_megakernel.py:554-560)."""
    from nki_moe_megakernel_amd import gpt_oss_with_megakernel as G
    cfg = G.GptOssMKConfig(hidden_size=96, hidden_pad=512, num_attention_heads=4, num_key_value_heads=2,
                           head_dim=16, num_experts=3, intermediate_size=8)
    hf = G.random_layer_hf(cfg, 0, 1, "cpu")
    c = G.convert_layer(hf, cfg)
    gu = hf["experts.gate_up_proj"]
    I = 8
    assert torch.equal(c["gate_up"][:, :I, :96], gu[:, :, 0::2].transpose(1, 2))
    assert torch.equal(c["gate_up"][:, I:, :96], gu[:, :, 1::2].transpose(1, 2))
    assert not c["gate_up"][:, :, 96:].any()
    b = hf["experts.gate_up_proj_bias"].float()
    assert torch.equal(c["gate_up_bias"][:, 0].float(), b[:, 0::2].bfloat16().float())
    assert torch.equal(c["gate_up_bias"][:, 1].float(), (b[:, 1::2] + 1).bfloat16().float())
    assert torch.equal(c["down"][:, :96], hf["experts.down_proj"].transpose(1, 2))
    assert not c["w_qkv"][:, 96:].any() and not c["ln_in"][96:].any()


def test_prefill_rejects_bad_requests_before_any_gpu_call(mk):
    """model.prefill's host checks: the sequence slot must exist and the prompt must
    fit the caches; a model without embedding / lm_head cannot prefill."""
    from types import SimpleNamespace
    from nki_moe_megakernel_amd.qwen_with_megakernel import _prefill
    cfg = SimpleNamespace(max_seq=16, vocab_size=32)
    m = SimpleNamespace(embed_tokens=torch.zeros(1), lm_head_packed=torch.zeros(1), batch=2, cfg=cfg,
                        device=torch.device("cpu"))
    ids = torch.arange(4, dtype=torch.int32)
    with pytest.raises(ValueError, match="sequence 2"):
        _prefill(m, ids, 0, 2, 128, 8, 8, 2, lambda p: (None, None))
    with pytest.raises(ValueError, match="does not fit"):
        _prefill(m, ids, 13, 0, 128, 8, 8, 2, lambda p: (None, None))
    with pytest.raises(ValueError, match="does not fit"):
        _prefill(m, ids[:0], 0, 0, 128, 8, 8, 2, lambda p: (None, None))
    with pytest.raises(ValueError, match="embedding"):
        _prefill(SimpleNamespace(**{**m.__dict__, "lm_head_packed": None}), ids, 0, 0, 128, 8, 8, 2,
                 lambda p: (None, None))


def _attention_call(mk, **kw):
    """attention_block_tkg on CPU tensors: B 4, H 128, four query heads and one kv head of 64, 31
    cached positions in a cache of 32; `kw` replaces arguments."""
    B, d, nq, none = 4, 64, 4, mk.QuantizationType.NONE
    a = dict(cos=torch.ones(d // 2, B, 1), sin=torch.zeros(d // 2, B, 1),
             kv_cache_update_idx=torch.zeros(B, 1, dtype=torch.int32))
    a.update(kw)
    zeros = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)
    return mk.attention_block_tkg(
        zeros(B, 1, 128), None, False, 1e-6, None, zeros(128, d * (nq + 2)), None, none, None, None, False, 1e-6,
        None, None, a["cos"], a["sin"], True, False, 1e-6, None, None, False, None, zeros(B, 32, d),
        zeros(B, 32, d), torch.ones(32, B, nq, 1, dtype=torch.uint8), None, True, a["kv_cache_update_idx"], None,
        None, none, None, None, False, False)


@pytest.mark.parametrize("shape", [(32, 1, 1), (16, 4, 1), (32, 4, 2), (32, 8, 1), (32, 4), (128,)])
def test_attention_refuses_rope_tables_of_another_shape(mk, monkeypatch, shape):
    """Both tables are indexed over [d/2, B, S_tkg] by their strides, so either of another
    shape is refused before any kernel (a shorter one would be read past its end)."""
    from nki_moe_megakernel_amd import _lib as L
    monkeypatch.setattr(L, "require_gpu", lambda *t: None)
    for name in ("cos", "sin"):
        with pytest.raises(ValueError, match=f"{name} shape mismatch"):
            _attention_call(mk, **{name: torch.zeros(shape)})


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_attention_refuses_too_few_write_positions(mk, monkeypatch, dtype):
    """One write position per sequence is read; fewer are refused before any kernel."""
    from nki_moe_megakernel_amd import _lib as L
    monkeypatch.setattr(L, "require_gpu", lambda *t: None)
    for shape in ((3, 1), (1,), (0, 1)):
        with pytest.raises(ValueError, match="kv_cache_update_idx must be"):
            _attention_call(mk, kv_cache_update_idx=torch.zeros(shape, dtype=dtype))


def test_disjoint_knows_shared_memory(mk):
    from nki_moe_megakernel_amd.moe import _disjoint
    a, b = torch.zeros(8, 4), torch.zeros(8, 4)
    assert _disjoint([a, b]) and _disjoint([a[:4], a[4:], b]) and _disjoint([a[4:], a[:4]])
    assert not _disjoint([a, a]) and not _disjoint([a[:5], a[4:]]) and not _disjoint([a[:, :2], a[:, 2:]])
    assert not _disjoint([b, a.t(), a[7:]]) and _disjoint([a[:0], a, b])
