"""Host logic on the CPU: GPT-2 plumbing model, engine loops, LR schedule, VLM generic path,
and the gradient arena bookkeeping (on CPU tensors, no kernels)."""

import pytest
import torch

from conftest import sub_dict
from oracle.gen_golden import TINY_GPT


def test_gpt2_plumbing_matches_reference(golden):
    from llm_quest_amd.gpt.gpt_model import GPTModel

    t = golden("gpt2_tiny")
    m = GPTModel(dict(TINY_GPT)).eval()
    sd = sub_dict(t, "sd.")
    missing, unexpected = m.load_state_dict(sd, strict=False)
    assert all(k.endswith(".mask") for k in missing) and not unexpected
    with torch.no_grad():
        assert torch.allclose(m(t["in.ids"]), t["out.logits"], atol=1e-5)
        assert torch.allclose(m(t["in.ids"], attn_mask=t["in.key_mask"].bool()), t["out.logits_masked"], atol=1e-5)
        emb = m.emb_dict(t["in.ids"]) + m.pos_emb_dict(torch.arange(16))
        assert torch.allclose(m(emb, input_embedded=True), t["out.logits"], atol=1e-5)
        last = m(t["in.ids"], attn_mask=t["in.key_mask"].bool(), last_token_only=True)
        assert last.shape == (4, 256)


def test_config1_shape_gpt2_small_cpu_forward():
    """GPT-2-small forward on CPU, batch 4 x seq 128, random tokens (plumbing)."""
    from llm_quest_amd.config import gpt2_config_creator
    from llm_quest_amd.gpt.gpt_model import GPTModel

    torch.manual_seed(123)
    cfg = gpt2_config_creator("gpt_s")
    cfg["n_layers"] = 2  # keep the CPU suite fast; width/heads/vocab are the real ones
    m = GPTModel(cfg).eval()
    x = torch.randint(0, 50257, (4, 128))
    with torch.no_grad():
        y = m(x)
    assert y.shape == (4, 128, 50257) and torch.isfinite(y).all()


def test_lr_scheduler_matches_reference_trace(golden):
    from llm_quest_amd.engine import LearningRateScheduler

    t = golden("per_op")
    opt = torch.optim.SGD([torch.nn.Parameter(torch.zeros(1))], lr=1.0)
    sch = LearningRateScheduler(opt, total_steps=10, init_lr=1e-5, peak_lr=1e-3, warmup_steps=3, min_lr=1e-4, decay="cosine")
    trace = []
    for s in range(10):
        sch.step(s)
        trace.append(sch.current_lr)
        assert opt.param_groups[0]["lr"] == sch.current_lr
    assert torch.allclose(torch.tensor(trace, dtype=torch.float64), t["lr.trace"], rtol=1e-12, atol=0)
    with pytest.raises(ValueError):
        LearningRateScheduler(opt, 10, init_lr=1e-3, peak_lr=1e-3, warmup_steps=2)
    with pytest.raises(ValueError):
        LearningRateScheduler(opt, 10, init_lr=1e-5, peak_lr=1e-3, min_lr=1e-4)


def _tiny_gpt():
    from llm_quest_amd.gpt.gpt_model import GPTModel

    torch.manual_seed(0)
    return GPTModel(dict(TINY_GPT))


def test_training_eval_loop_cpu_semantics():
    """accumulation with a ragged last window, eval at step 1 and every eval_freq, returns two lists."""
    from llm_quest_amd.engine import LearningRateScheduler, global_loss, training_eval_loop

    m = _tiny_gpt()
    g = torch.Generator().manual_seed(1)
    data = [(torch.randint(0, 256, (2, 16), generator=g), torch.randint(0, 256, (2, 16), generator=g)) for _ in range(5)]
    opt = torch.optim.AdamW(m.parameters(), lr=1e-3)
    sch = LearningRateScheduler(opt, total_steps=10, init_lr=1e-5, peak_lr=1e-3, warmup_steps=2)
    tr, va = training_eval_loop(data, data[:2], m, opt, 1, sch, eval_freq=2, eval_iter=1, device=torch.device("cpu"), accumulation_steps=2, use_amp=False)
    assert len(tr) == 2 and len(va) == 2  # 3 optimizer steps: evals at step 1 and 2
    with pytest.raises(AttributeError):
        global_loss(torch.zeros(1, 2, 3), torch.zeros(1, 2, dtype=torch.long), model=None)  # upstream quirk: model required


def test_vlm_generic_path_on_cpu():
    """The reference's own wiring (ViT-ish encoder -> adapter -> GPT-2 with input_embedded) through our engine."""
    from llm_quest_amd.multimodal.vlm_engine import get_embeddings, vlm_loss, vlm_step_loss

    class FakeViT(torch.nn.Module):
        def forward(self, x, output_hidden_states=False):
            return x.flatten(2).transpose(1, 2)[:, :5, :8].contiguous()

    llm = _tiny_gpt()
    adapter = torch.nn.Linear(8, 64, bias=False)
    img = torch.randn(2, 8, 3, 3)
    ids = torch.randint(0, 256, (2, 7))
    tm = torch.ones(2, 7, dtype=torch.bool)
    tm[0, 5:] = False
    loss = vlm_step_loss(FakeViT(), llm, adapter, img, ids, tm, hf_vit_model=False)
    # same thing written out as the reference does
    ve = adapter(FakeViT()(img))
    x = torch.cat([ve, get_embeddings(ids, llm)], dim=1)
    cm = torch.cat([torch.ones(2, 5, dtype=torch.bool), tm], dim=1)
    ref = vlm_loss(llm(x, attn_mask=cm, input_embedded=True), ids, tm, 5)
    assert torch.allclose(loss, ref)
    loss.backward()
    assert adapter.weight.grad is not None


def test_param_arena_views_and_grad_targets():
    from llm_quest_amd.arena import ParamArena

    lin_a, lin_b, lin_c = torch.nn.Linear(8, 16, bias=False), torch.nn.Linear(8, 8, bias=False), torch.nn.Linear(8, 8, bias=False)
    named = [("a", lin_a.weight), ("b", lin_b.weight), ("c", lin_c.weight)]
    before = [p.detach().clone() for _, p in named]
    ar = ParamArena(named)
    assert ar.ensure() is True and ar.ensure() is False
    for (_, p), b in zip(named, before):
        assert torch.equal(p, b)
    fused = ar.fused(lin_a.weight, lin_c.weight)
    assert fused.shape == (32, 8) and fused.data_ptr() == lin_a.weight.data_ptr()
    assert torch.equal(fused[16:24], lin_b.weight)
    view, acc = ar.grad_target(lin_a.weight, lin_c.weight)
    assert view.shape == (32, 8) and acc is False and lin_b.weight.grad.data_ptr() == view[16:24].data_ptr()
    view2, acc2 = ar.grad_target(lin_b.weight)
    assert acc2 is True
    for p in (lin_a.weight, lin_b.weight, lin_c.weight):
        p.grad = None  # zero_grad(set_to_none=True)
    _, acc3 = ar.grad_target(lin_b.weight)
    assert acc3 is False
    # .to()/rebinding is detected and the arena is rebuilt around the new storage
    lin_b.weight.data = lin_b.weight.data.clone()
    assert ar.ensure() is True and ar.fused(lin_a.weight, lin_c.weight).shape == (32, 8)


def test_hf_qwen3_checkpoint_import_round_trip(tmp_path, capsys):
    """HF parameter names -> this package's: a synthetic HF-named checkpoint built from one model loads
    into a second model bit for bit, through a dict and through a .safetensors file; bad shapes / unknown names are reported."""
    from safetensors.torch import save_file

    from llm_quest_amd.qwen.qwen3.qwen3_model import Qwen3Model
    from llm_quest_amd.qwen.qwen3.qwen3_weight_loading import get_remapping_rules, load_qwen3_weights

    cfg = dict(vocab_size=96, emb_dim=32, n_layers=2, n_heads=4, num_kv_groups=2, head_dim=8, hidden_dim=64, context_length=16,
               rope_base=10_000, dtype=torch.bfloat16, tie_embeddings=True, model_type="dense")
    torch.manual_seed(0)
    src, dst = Qwen3Model(cfg), Qwen3Model(cfg)
    inverse = [(ours, hf) for hf, ours in get_remapping_rules(cfg)]
    hf = {}
    for name, w in src.state_dict().items():
        if name in ("mask", "cos", "sin", "out_head.weight"):
            continue
        hf_name = name
        for ours, theirs in inverse:
            hf_name = hf_name.replace(ours, theirs)
        hf[hf_name] = w.detach().clone()
    assert "model.layers.1.self_attn.q_proj.weight" in hf and "model.layers.0.mlp.up_proj.weight" in hf
    hf["model.layers.0.self_attn.rotary_emb.inv_freq"] = torch.zeros(4)  # unknown upstream tensor: reported, not loaded
    load_qwen3_weights(dst, cfg, source=hf)
    out = capsys.readouterr().out
    assert "No match for HF weight 'model.layers.0.self_attn.rotary_emb.inv_freq'" in out
    for (n1, p1), (n2, p2) in zip(src.named_parameters(), dst.named_parameters()):
        assert n1 == n2 and torch.equal(p1, p2), n1
    assert dst.out_head.weight is dst.emb_dict.weight
    # through a file, into a third model
    path = tmp_path / "model.safetensors"
    hf.pop("model.layers.0.self_attn.rotary_emb.inv_freq")
    save_file({k: v.contiguous() for k, v in hf.items()}, str(path))
    third = load_qwen3_weights(Qwen3Model(cfg), cfg, source=str(path), verbose=False)
    assert all(torch.equal(a, b) for a, b in zip(src.parameters(), third.parameters()))
    with pytest.raises(ValueError):
        load_qwen3_weights(Qwen3Model(cfg), cfg)


def _to_hf_names(state_dict, rules, skip=()):
    """Inverse of the loader's rename: our names -> HF names, last rule first so that nested substrings unwind correctly."""
    out = {}
    for name, w in state_dict.items():
        if name in skip:
            continue
        hf_name = name
        for hf, ours in reversed(rules):
            if ours in hf_name and (ours.startswith(".") or hf_name.startswith(ours)):
                hf_name = hf_name.replace(ours, hf, 1)
        out[hf_name] = w.detach().clone()
    return out


def test_hf_qwen3_5_checkpoint_import_round_trip(tmp_path, capsys):
    """Row f2 for BASELINE config 5: an HF-named Qwen3.5 checkpoint (text stack + vision tower + an ``mtp.`` head that must be
    ignored) loads bit for bit into the text-only model and into the VLM; fp32 stragglers keep their dtype."""
    from safetensors.torch import save_file

    from llm_quest_amd.qwen.qwen3_5.qwen3_5_text_model import Qwen3_5TextModel
    from llm_quest_amd.qwen.qwen3_5.qwen3_5_vlm_model import Qwen3_5VLM
    from llm_quest_amd.qwen.qwen3_5.qwen3_5_weight_loading import (
        get_remapping_rules,
        get_vision_remapping_rules,
        load_qwen3_5_text_weights,
        load_qwen3_5_vlm_weights,
    )

    cfg = dict(
        vocab_size=256, emb_dim=128, hidden_dim=128, n_layers=4, linear_sdpa_ratio=2, n_heads=2, num_kv_groups=1, head_dim=32,
        rope_base=10_000_000, partial_rope_factor=0.5, context_length=64, linear_num_qk_heads=2, linear_num_value_heads=4,
        linear_qk_head_dim=16, linear_value_head_dim=16, linear_conv_kernel_size=4, tie_embeddings=True, p_dropout=0.0,
        training=False, mrope_section=[3, 3, 2], dtype=torch.bfloat16,
        vision_n_layers=2, vision_emb_dim=128, vision_hidden_dim=256, vision_num_heads=2, llm_d_in=128, in_channels=3, patch_size=8,
        spatial_merge_size=2, temporal_patch_size=2, num_position_embeddings=64, img_width=32, img_height=32,
        vision_rope_base=10_000, image_token_id=250,
    )
    torch.manual_seed(1)
    src = Qwen3_5VLM(cfg)
    with torch.no_grad():  # the zero / one initialised tensors would make the comparison vacuous
        for p in src.parameters():
            if p.dim() == 1:
                p.copy_(torch.randn(p.shape))
    hf = _to_hf_names(src.language_model.state_dict(), get_remapping_rules(),
                      skip=("out_head.weight", "mask", "cos", "sin"))  # tied head; buffers are rebuilt locally
    hf.update(_to_hf_names(src.vision_model.state_dict(), get_vision_remapping_rules()))
    assert {"model.language_model.embed_tokens.weight", "model.language_model.norm.weight",
            "model.language_model.layers.0.linear_attn.A_log", "model.language_model.layers.0.linear_attn.in_proj_qkv.weight",
            "model.language_model.layers.1.self_attn.q_proj.weight", "model.language_model.layers.3.self_attn.k_norm.weight",
            "model.language_model.layers.2.linear_attn.norm.weight", "model.language_model.layers.2.mlp.down_proj.weight",
            "model.visual.patch_embed.proj.bias", "model.visual.pos_embed.weight", "model.visual.blocks.1.attn.qkv.weight",
            "model.visual.blocks.0.mlp.linear_fc2.bias", "model.visual.blocks.0.norm2.weight",
            "model.visual.merger.linear_fc1.weight", "model.visual.merger.norm.bias"} <= set(hf)
    assert not [k for k in hf if not k.startswith(("model.language_model.", "model.visual."))]
    hf["mtp.fc.weight"] = torch.zeros(4, 4)

    # text-only model: vision + mtp tensors are skipped silently, everything else lands
    text = load_qwen3_5_text_weights(Qwen3_5TextModel(cfg), cfg, source=hf)
    out = capsys.readouterr().out
    assert "WARNING" not in out and f"Skipped {1 + len(src.vision_model.state_dict())} weights" in out
    for (n1, p1), (n2, p2) in zip(src.language_model.named_parameters(), text.named_parameters()):
        assert n1 == n2 and p1.dtype == p2.dtype and torch.equal(p1, p2), n1
    assert text.out_head.weight is text.emb_dict.weight
    assert text.trf_blocks[0].att.log_A.dtype == torch.float32

    # VLM, through a file
    path = tmp_path / "model.safetensors"
    save_file({k: v.contiguous() for k, v in hf.items()}, str(path))
    dst = load_qwen3_5_vlm_weights(Qwen3_5VLM(cfg), cfg, source=str(path))
    out = capsys.readouterr().out
    assert "WARNING" not in out and "Unexpected" not in out
    assert f"Loaded {len(hf) - 1}/{len(dst.state_dict())} weights" in out  # everything in the file but the mtp head
    for (n1, p1), (n2, p2) in zip(src.named_parameters(), dst.named_parameters()):
        assert n1 == n2 and torch.equal(p1, p2), n1
    assert dst.language_model.out_head.weight is dst.language_model.emb_dict.weight

    # a mis-shaped tensor is reported and left alone; no source is an error, not a download
    bad = dict(hf)
    bad["model.language_model.layers.0.linear_attn.dt_bias"] = torch.zeros(7)
    keep = Qwen3_5TextModel(cfg)
    before = keep.trf_blocks[0].att.dt_bias.detach().clone()
    load_qwen3_5_text_weights(keep, cfg, source=bad, verbose=False)
    assert "Shape mismatch: trf_blocks.0.att.dt_bias" in capsys.readouterr().out
    assert torch.equal(keep.trf_blocks[0].att.dt_bias, before)
    with pytest.raises(ValueError):
        load_qwen3_5_vlm_weights(Qwen3_5VLM(cfg), cfg)


def test_hf_checkpoint_key_maps_match_the_reference_converter(capsys):
    """Row f2 pinned to the reference: ``tests/golden/weight_maps.json`` holds synthetic Hugging-Face-named checkpoints ((name, shape)
    lists written from the published HF layouts) and what the REFERENCE's ``convert_weights`` + rule tables made of them
    (``oracle/gen_golden.py::gen_weight_maps``).  The same checkpoints through this package's converter, against this package's models,
    must reach exactly the same parameter names, report as many problems and skip as many tensors."""
    import json
    import os

    from llm_quest_amd.qwen.qwen3 import qwen3_weight_loading as W3
    from llm_quest_amd.qwen.qwen3.qwen3_model import Qwen3Model
    from llm_quest_amd.qwen.qwen3_5 import qwen3_5_weight_loading as W35
    from llm_quest_amd.qwen.qwen3_5.qwen3_5_vlm_model import Qwen3_5VLM
    from llm_quest_amd.utils import convert_weights

    with open(os.path.join(os.path.dirname(__file__), "golden", "weight_maps.json")) as f:
        fx = json.load(f)

    def run(tensors, state, rules, ignored=None):
        hf = {n: torch.zeros(tuple(s)) for n, s in tensors}
        capsys.readouterr()
        conv = convert_weights(hf, state, rules, ignored_prefixes=ignored)
        out = capsys.readouterr().out
        skipped = [int(line.split()[1]) for line in out.splitlines() if line.startswith("Skipped ")]
        return {"loaded": sorted(conv), "warnings": sum(1 for line in out.splitlines() if line.startswith("WARNING")), "skipped": skipped[0] if skipped else 0}

    for case in ("qwen3_tie1", "qwen3_tie0"):
        cfg = dict(fx[case]["cfg"], dtype=torch.bfloat16)
        got = run(fx[case]["tensors"], Qwen3Model(cfg).state_dict(), W3.get_remapping_rules(cfg))
        assert got == fx[case]["result"], case
    cfg = dict(fx["qwen35"]["cfg"], dtype=torch.bfloat16)
    vlm = Qwen3_5VLM(cfg)
    assert run(fx["qwen35"]["tensors"], vlm.language_model.state_dict(), W35.get_remapping_rules(), ("model.visual.", "mtp.")) == fx["qwen35"]["text"]
    assert run(fx["qwen35"]["tensors"], vlm.vision_model.state_dict(), W35.get_vision_remapping_rules(), ("model.language_model.", "mtp.")) == fx["qwen35"]["vision"]
    # every parameter of either model that a checkpoint can fill was filled (the rule tables cover the whole state dict)
    loaded = set(fx["qwen35"]["text"]["loaded"])
    missing = [k for k in vlm.language_model.state_dict() if k not in loaded and k not in ("mask", "cos", "sin", "out_head.weight")]
    assert not missing, missing
