"""Headline benchmark: img+tokens/sec of the early-fusion VLM forward+backward step.

    python bench.py --gpus N --steps K --warmup W

N > 1 runs one rank per GPU over RCCL.  Under ``torch.distributed.run`` (WORLD_SIZE set) this process IS a rank; started
plainly with ``--gpus N`` it starts the N ranks itself -- a child ``python -m torch.distributed.run --nproc-per-node N bench.py ...``
spawned before this process has touched the GPU -- and relays rank 0's JSON line and the child's exit status.

A step = vision tower (frozen ViT-B/16, eval) -> ffn adapter -> early-fusion concat -> Qwen3-0.6B decoder on the fused
709-token sequence -> tied LM head + cross entropy on the 512 text positions -> full backward (adapter + LLM), plus the
RCCL gradient all-reduce when N > 1.  The optimizer step is NOT part of the metric; gradients are
dropped between steps (zero_grad(set_to_none=True)).  Synthetic seeded inputs, random-init weights, inputs resident in
HBM before the timed region.  One JSON line on rank 0.
"""

import argparse
import json
import os
import sys
import time

import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

N_VISION, N_TEXT, VOCAB = 197, 512, 151_936
UNITS_PER_SAMPLE = 1 + N_TEXT  # 1 image + 512 text tokens
ALGO_FLOP_PER_SAMPLE = 2.566e12  # 35.13 G (frozen ViT fwd) + 3 x (2.17 G adapter + 841.5 G LLM)
PEAK_BF16_TFLOPS = 2500.0  # MI355X dense bf16 MFMA peak (MI355X_MICROARCH.md)
CPU_SAMPLES = 8  # size of the bounded CPU-baseline sample (~10-15 s on the box's 16-core quota)


def build_models(device, seed=123):
    from llm_quest_amd.config import VIT_BASE_CONFIG, qwen3_config_creator
    from llm_quest_amd.multimodal.vision_transformer.vit_engine import ViTAdapter
    from llm_quest_amd.multimodal.vision_transformer.vit_model import ViTModel
    from llm_quest_amd.qwen.qwen3.qwen3_model import Qwen3Model

    torch.manual_seed(seed)
    vit_cfg = dict(VIT_BASE_CONFIG, drop_rate=0.0)
    llm_cfg = dict(qwen3_config_creator("0.6B"), context_length=1024)
    with torch.device(device):
        vit = ViTModel(vit_cfg)
        llm = Qwen3Model(llm_cfg)
        ad = ViTAdapter(768, 1024, adapter_type="ffn", dtype=torch.bfloat16)
    vit.eval()
    for p in vit.parameters():
        p.requires_grad = False
    llm.train()
    ad.train()
    return vit, vit_cfg, ad, llm, llm_cfg


def synthetic_batch(batch, device, seed, ragged=False):
    """The headline's inputs: randn images, uniform token ids, all-ones text mask; ``ragged``: real lengths ~ U[256, 512], right-padded."""
    g = torch.Generator().manual_seed(seed)
    img = torch.randn(batch, 3, 224, 224, generator=g)
    ids = torch.randint(0, VOCAB, (batch, N_TEXT), generator=g)
    mask = torch.ones(batch, N_TEXT, dtype=torch.bool)
    if ragged:
        lengths = torch.randint(256, N_TEXT + 1, (batch,), generator=g)
        mask = torch.arange(N_TEXT).unsqueeze(0) < lengths.unsqueeze(1)
    return img.to(device), ids.to(device), mask.to(device)


def usable_cores():
    """CPU threads this process may really use: affinity mask capped by the cgroup CPU quota (GPU boxes share a host)."""
    n = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    try:
        quota, period = open("/sys/fs/cgroup/cpu.max").read().split()
        if quota != "max":
            n = min(n, max(1, int(int(quota) / int(period))))
    except (OSError, ValueError):
        pass
    return max(1, n)


def _cpu_baseline_worker(state_path, seed, threads, q):
    """Child process: the CPU oracle (oracle/models.py) on one full-size sample, forward + backward."""
    torch.set_num_threads(threads)
    from llm_quest_amd.config import VIT_BASE_CONFIG, qwen3_config_creator
    from oracle import models

    st = torch.load(state_path)
    vit_cfg = dict(VIT_BASE_CONFIG, drop_rate=0.0)
    llm_cfg = dict(qwen3_config_creator("0.6B"), context_length=1024)
    ad_sd = {k: v.requires_grad_(True) for k, v in st["ad"].items()}
    llm_sd = {k: v.requires_grad_(True) for k, v in st["llm"].items()}
    llm_sd["out_head.weight"] = llm_sd["emb_dict.weight"]
    img, ids, mask = synthetic_batch(CPU_SAMPLES, "cpu", seed)

    def step(i, t, m):
        loss, _, _ = models.vlm_forward_loss(st["vit"], vit_cfg, ad_sd, llm_sd, llm_cfg, i, t, m)
        loss.backward()
        return float(loss.detach())

    step(img[:1], ids[:1, :16], mask[:1, :16])  # warm the thread pool / allocator on a short sequence
    t0 = time.perf_counter()
    loss = step(img, ids, mask)
    q.put((time.perf_counter() - t0, loss))


def cpu_baseline(vit, ad, llm, seed, budget_s=240):
    """The CPU oracle (proved equal to the reference on fixtures) timed on this host's cores on a BOUNDED sample: one
    full-size sample (1 image + 512 tokens, S=709), forward+backward, same weights.  Runs in a child process with a hard
    time budget so the default bench always finishes in minutes; reported, never the optimisation target."""
    import tempfile

    import torch.multiprocessing as mp

    cores = min(usable_cores(), 32)
    state = {
        "vit": {k: v.detach().cpu() for k, v in vit.state_dict().items()},
        "ad": {k: v.detach().cpu().clone() for k, v in ad.state_dict().items()},
        "llm": {k: v.detach().cpu().clone() for k, v in llm.state_dict().items() if k not in ("mask", "cos", "sin", "out_head.weight")},
    }
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "state.pt")
        torch.save(state, path)
        del state
        ctx = mp.get_context("spawn")
        q = ctx.Queue()
        proc = ctx.Process(target=_cpu_baseline_worker, args=(path, seed, cores, q))
        proc.start()
        proc.join(budget_s)
        if proc.is_alive():
            proc.kill()
            proc.join()
            return {"value": None, "unit": "img+tok/s", "cores": cores, "kind": "port",
                    "sample": f"{CPU_SAMPLES} full-size samples fwd+bwd did not finish within the {budget_s} s budget on {cores} threads"}
        dt, loss = q.get(timeout=10)
    return {
        "value": round(CPU_SAMPLES * UNITS_PER_SAMPLE / dt, 3), "unit": "img+tok/s", "cores": cores, "kind": "port",
        "sample": f"{CPU_SAMPLES} samples (each 1 img + 512 tok, S=709) full-size fwd+bwd in {dt:.1f} s on {cores} threads, torch {torch.__version__} CPU, oracle loss {loss:.4f}",
    }


def _profile_json(name):
    """A committed counter file from profiles/ -- only if it was measured on the kernel sources this process runs
    (llm_quest_amd/fingerprint.py); a stale file yields None, never a number."""
    from llm_quest_amd.fingerprint import kernel_sources_sha

    path = os.path.join(ROOT, "profiles", name)
    try:
        with open(path) as f:
            d = json.load(f)
    except (OSError, ValueError):
        return None, f"{name} not found"
    if d.get("kernel_sources_sha") != kernel_sources_sha():
        return None, f"{name} was measured on other kernel sources (its fingerprint {d.get('kernel_sources_sha')} != {kernel_sources_sha()}): re-collect it"
    return d, None


def pmc_traffic():
    """TCC counters of the dominant kernel, collected with rocprofv3 --pmc in separate passes and committed (PMC cannot be read
    from inside the timed process)."""
    from llm_quest_amd.fingerprint import EVIDENCE_ROUND

    d, why = _profile_json(f"{EVIDENCE_ROUND}_pmc_tcc_gemm.json")
    return (d["kernels"] if d else None), why


def pmc_step_traffic():
    """Whole-step TCC counters (profiles/<round>_pmc_tcc_step.json), collected with rocprofv3 --pmc over this script."""
    from llm_quest_amd.fingerprint import EVIDENCE_ROUND

    return _profile_json(f"{EVIDENCE_ROUND}_pmc_tcc_step.json")


def dominant_kernel_rate(batch, device):
    """HIP-event timing of the step's dominant kernel class (gemm_quad_kernel for the NT forms, gemm_quad_grouped_kernel for TN) on its largest shapes, on the stream the
    kernels are launched on (torch's current stream)."""
    from llm_quest_amd import _lib as L
    from llm_quest_amd import kernels as K

    M = batch * (N_VISION + N_TEXT)
    x = torch.randn(M, 1024, device=device).to(torch.bfloat16)
    w = torch.randn(6144, 1024, device=device).to(torch.bfloat16)
    dy = torch.randn(M, 6144, device=device).to(torch.bfloat16)
    shapes = [(4096, 1024), (1024, 2048), (6144, 1024), (1024, 3072)]  # [out, in] of the block's four weight matrices
    group = [(torch.randn(M, o, device=device).to(torch.bfloat16), torch.randn(M, i, device=device).to(torch.bfloat16), torch.zeros(o, i, device=device, dtype=torch.bfloat16), None)
             for o, i in shapes]
    out = {}
    for name, fn, flops in (
        ("NT gate-up fwd", lambda: K.gemm(L.GEMM_NT, x, w), 2.0 * M * 6144 * 1024),
        ("NN gate-up dgrad (the step's form: the weight as it lies)", lambda: K.dgrad(dy, w), 2.0 * M * 6144 * 1024),
        ("NT gate-up dgrad on a transposed copy of the weight (not used by the step)", lambda: K.gemm(L.GEMM_NT, dy, K.transpose(w)), 2.0 * M * 6144 * 1024),
        ("TN block weight gradients, grouped (the step's launch: QKV, out_proj, gate-up, down = 240 tiles)", lambda: K.gemm_grouped(L.GEMM_TN, group), 2.0 * M * sum(o * i for o, i in shapes)),
    ):
        for _ in range(3):
            fn()
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        for _ in range(10):
            fn()
        e.record()
        torch.cuda.synchronize()
        ms = s.elapsed_time(e) / 10
        out[name] = {"ms": round(ms, 4), "tflops": round(flops / ms / 1e9, 1)}
    return out


class BoardPower:
    """Board power and shader clock over the timed steps, from the amdgpu hwmon files (power1_input uW, freq1_input Hz: readable without privileges, sampled every 10 ms
    by a thread that touches nothing else).  A box shows the hwmon directories of cards that are not this job's: the card is the one whose power follows the warm-up
    steps.  Reported beside the roofline because the step runs AT the board's cap (profiles/r05_power.json): what the matrix pipe sustains there, not at 2.4 GHz, is
    what the step is up against."""

    def __init__(self):
        import glob
        import threading

        self.dirs = [os.path.dirname(p) for p in glob.glob("/sys/class/drm/card*/device/hwmon/hwmon*/power1_input")]
        self.idle = {d: self._read(d)[0] for d in self.dirs}
        self.peak = dict(self.idle)
        self.chosen, self.samples, self._stop = None, [], threading.Event()
        self._thread = threading.Thread(target=self._run, daemon=True)
        if self.dirs:
            self._thread.start()

    @staticmethod
    def _read(d):
        try:
            return int(open(d + "/power1_input").read()) / 1e6, int(open(d + "/freq1_input").read()) / 1e6
        except (OSError, ValueError):
            return 0.0, 0.0

    def _run(self):
        while not self._stop.is_set():
            if self.chosen is None:
                for d in self.dirs:
                    self.peak[d] = max(self.peak[d], self._read(d)[0])
            else:
                self.samples.append(self._read(self.chosen))
            time.sleep(0.01)

    def choose(self):  # after the warm-up steps, before the timed region
        rise = {d: self.peak[d] - self.idle[d] for d in self.dirs}
        best = max(rise, key=rise.get) if rise else None
        if best is not None and rise[best] >= 150.0:
            self.samples = []
            self.chosen = best

    def mark(self):  # the timed region starts here
        self.samples = []

    def result(self):
        self._stop.set()
        if self.chosen is None:
            return {"mean_W": None, "note": "no visible amdgpu hwmon followed the warm-up steps (telemetry of this card not exposed)"}
        s = [x for x in self.samples if x[0] > 0]
        if not s:
            return {"mean_W": None, "note": "no samples"}
        try:
            cap = int(open(self.chosen + "/power1_cap").read()) / 1e6
        except (OSError, ValueError):
            cap = None
        return {"mean_W": round(sum(x[0] for x in s) / len(s), 1), "cap_W": cap, "sclk_mean_MHz": round(sum(x[1] for x in s) / len(s)), "samples": len(s),
                "source": "amdgpu hwmon power1_input / freq1_input every 10 ms over the timed steps; the dense peak in `roofline` assumes 2 400 MHz"}


def launch_ranks(n):
    """``python bench.py --gpus N`` without a torchrun environment: run the N ranks as a child ``torch.distributed.run`` job (a fresh
    process tree; nothing in THIS process has initialised the GPU yet) and pass its output and exit status through."""
    import socket
    import subprocess

    with socket.socket() as sk:
        sk.bind(("127.0.0.1", 0))
        port = sk.getsockname()[1]
    cmd = [sys.executable, "-m", "torch.distributed.run", "--nnodes=1", f"--nproc-per-node={n}", "--master-addr", "127.0.0.1",
           "--master-port", str(port), os.path.abspath(__file__)] + sys.argv[1:]
    env = dict(os.environ, HSA_ENABLE_IPC_MODE_LEGACY=os.environ.get("HSA_ENABLE_IPC_MODE_LEGACY", "0"))
    return subprocess.run(cmd, env=env).returncode


# ------------------------------------------------------------------------------------------------ the other BASELINE configurations
# ``--config 2 | 3 | 5`` print the same JSON schema for the three other workloads (inputs, units,
# algorithmic FLOP per sample).  They are parity-test configurations of the same kernels, not the headline: the default (``--config 4``) is
# untouched by them.  No counter files are kept for them, so ``roofline.traffic`` is null.
OTHER_CONFIGS = {
    # batch 332: 65 404 tokens = 255.5 row tiles of 256, so the N = 768 outputs are 768 tiles = three whole rounds of the chip (at 256 images: 591 tiles = 2.3 rounds; 21.9 -> 23.1 %, same box)
    2: dict(metric="img/sec fwd+bwd, ViT-Base/16 224x224, bf16 MFMA operands", unit="img/s", flop=105.4e9, batch=332, units_per_sample=1, max_gpus=1,
            workload="BASELINE configs[1]: ViT-Base/16 (VIT_BASE_CONFIG, num_classes 100), 224x224, forward + cross entropy + backward of every parameter, "
                     "fp32 master weights / fp32 residual stream / bf16 MFMA operands, no optimizer step"),
    3: dict(metric="tokens/sec fwd+bwd, Qwen3-0.6B dense text-only, seq 1024, bf16", unit="tok/s", flop=4.023e12, batch=64, units_per_sample=1024, max_gpus=1,
            workload="BASELINE configs[2]: Qwen3-0.6B (context_length 1024), 1024 random tokens per sequence, forward + global_loss + backward, no optimizer step"),
    5: dict(metric="frames+tokens/sec fwd+bwd, Qwen3.5-style VLM (Qwen3-ViT 3-D patches 8x224x224 + hybrid GDN / gated-attention 0.8B text stack, MRoPE-I), bf16",
            unit="frames+tok/s", flop=3.492e12, batch=32, units_per_sample=8 + 512, max_gpus=8,
            workload="BASELINE configs[4]: Qwen3_5VLM(QWEN3_5_08B_CONFIG, 224x224), 8 frames -> 196 merged vision rows at the placeholders + 512 text tokens "
                     "(S = 708), targets = shifted ids, forward + loss + backward of both towers, no optimizer step"),
}


def _other_config_step(cfg_id, batch, device, rank):
    """Builds the model and the synthetic batch of configs 2 / 3 / 5 (seeded) and returns (step_fn, sync, state_for_cpu)."""
    from llm_quest_amd import ddp

    torch.manual_seed(123)
    if cfg_id == 2:
        from llm_quest_amd.config import VIT_BASE_CONFIG
        from llm_quest_amd.engine import _cross_entropy
        from llm_quest_amd.multimodal.vision_transformer.vit_model import ViTModel

        cfg = dict(VIT_BASE_CONFIG, drop_rate=0.0)  # the parity setting; drop_rate 0.1 (as configured upstream) costs 12-13 %
        with torch.device(device):
            model = ViTModel(cfg).train()
        g = torch.Generator().manual_seed(123 + rank)
        img = torch.randn(batch, 3, 224, 224, generator=g).to(device)
        y = torch.randint(0, cfg["num_classes"], (batch,), generator=g).to(device)

        def step():
            model.zero_grad(set_to_none=True)
            loss = _cross_entropy(model(img), y)
            loss.backward()
            return loss

        return step, None, ("vit", cfg, model, (img, y))
    if cfg_id == 3:
        from llm_quest_amd.config import qwen3_config_creator
        from llm_quest_amd.qwen.qwen3.qwen3_model import Qwen3Model

        cfg = dict(qwen3_config_creator("0.6B"), context_length=1024)
        with torch.device(device):
            model = Qwen3Model(cfg).train()
        g = torch.Generator().manual_seed(123 + rank)
        x = torch.randint(0, VOCAB, (batch, 1024), generator=g).to(device)
        y = torch.randint(0, VOCAB, (batch, 1024), generator=g).to(device)

        def step():
            model.zero_grad(set_to_none=True)
            h = model.forward_hidden(x)  # == global_loss(model(x), y): the head + CE on every position (all 1024 feed the loss), logits written once
            loss = model.lm_loss(h.reshape(-1, h.shape[-1]), y.reshape(-1))
            loss.backward()
            return loss

        return step, None, ("qwen3", cfg, model, (x, y))
    from llm_quest_amd.config import QWEN3_5_08B_CONFIG
    from llm_quest_amd.qwen.qwen3_5.qwen3_5_vlm_model import Qwen3_5VLM, fuse_vision_embeddings

    cfg = dict(QWEN3_5_08B_CONFIG, img_width=224, img_height=224, context_length=1024)
    with torch.device(device):
        vlm = Qwen3_5VLM(cfg).train()
    sync = ddp.sync_for_qwen35(vlm)
    sync.broadcast_parameters([vlm])
    g = torch.Generator().manual_seed(123 + rank)
    n_img = (8 // cfg["temporal_patch_size"]) * (14 // cfg["spatial_merge_size"]) ** 2  # 196 merged rows
    ids = torch.randint(0, 248_000, (batch, 512 + n_img), generator=g)
    ids[:, 100 : 100 + n_img] = cfg["image_token_id"]
    pix = torch.randn(batch, 3, 8, 224, 224, generator=g).to(device)
    ids = ids.to(device)
    tgt = torch.roll(ids, -1, 1)
    lm = vlm.language_model

    def step():
        vlm.zero_grad(set_to_none=True)
        emb = lm.emb_dict(ids)
        mask = ids == cfg["image_token_id"]
        emb = fuse_vision_embeddings(emb, mask, vlm.vision_model(pix))
        pos = vlm.compute_3d_position_ids(ids, vlm.get_feeds_3d_shape(pix), image_mask=mask)
        h = lm.forward_hidden(inputs_embs=emb, position_ids=pos)  # Qwen3_5VLM.forward with the head + CE fused behind it (logits written once)
        loss = lm.lm_loss(h.reshape(-1, h.shape[-1]), tgt.reshape(-1))
        sync.begin_step()
        loss.backward()
        sync.finish_step()
        return loss

    return step, sync, ("qwen35", cfg, vlm, (ids, pix, tgt))


def _other_cpu_worker(kind, cfg, state_path, threads, q):
    """Child process: the CPU oracle of configs 2 / 3 / 5 on a bounded sample of the same workload, forward + backward."""
    torch.set_num_threads(threads)
    import torch.nn.functional as F

    from oracle import models, ops
    from oracle import qwen3_5 as q35

    st = torch.load(state_path)
    sd = {k: (v.requires_grad_(True) if v.is_floating_point() and not k.endswith(("cos", "sin")) else v) for k, v in st["sd"].items()}
    t0 = time.perf_counter()
    if kind == "vit":
        img, y = st["batch"]
        loss = F.cross_entropy(models.vit_forward(sd, cfg, img).float(), y)
        units = img.shape[0]
    elif kind == "qwen3":
        x, y = st["batch"]
        sd["out_head.weight"] = sd["emb_dict.weight"]
        loss = ops.lm_loss(models.qwen3_forward(sd, cfg, x), y)
        units = x.numel()
    else:
        ids, pix, tgt = st["batch"]
        logits, _ = q35.vlm35_forward(sd, cfg, ids, pix)
        loss = ops.lm_loss(logits, tgt)
        units = ids.shape[0] * (8 + 512)
    loss.backward()
    q.put((time.perf_counter() - t0, float(loss.detach()), units))


def _other_cpu_baseline(state, n_samples, unit, budget_s=300):
    import tempfile

    import torch.multiprocessing as mp

    kind, cfg, model, batch = state
    cores = min(usable_cores(), 32)
    sd = {k: v.detach().cpu().clone() for k, v in model.state_dict().items() if k not in ("mask", "out_head.weight") and not k.endswith("language_model.out_head.weight")}
    for k in list(sd):
        if k.endswith("mask"):
            sd[k] = sd[k].bool()
    small = tuple(t[:n_samples].detach().cpu() for t in batch)
    cfg = {k: v for k, v in cfg.items()}
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "state.pt")
        torch.save({"sd": sd, "batch": small}, path)
        ctx = mp.get_context("spawn")
        q = ctx.Queue()
        proc = ctx.Process(target=_other_cpu_worker, args=(kind, cfg, path, cores, q))
        proc.start()
        proc.join(budget_s)
        if proc.is_alive():
            proc.kill()
            proc.join()
            return {"value": None, "unit": unit, "cores": cores, "kind": "port", "sample": f"{n_samples} full-size sample(s) fwd+bwd did not finish within the {budget_s} s budget on {cores} threads"}
        dt, loss, units = q.get(timeout=10)
    return {"value": round(units / dt, 3), "unit": unit, "cores": cores, "kind": "port",
            "sample": f"{n_samples} full-size sample(s) forward + backward through the CPU oracle in {dt:.1f} s on {cores} threads, torch {torch.__version__} CPU, oracle loss {loss:.4f}"}


def _config_traffic(config, batch):
    """``traffic`` of `bench.py --config N`: memory-side bytes per step from the committed counter passes (profiles/<round>_pmc_tcc_step_config<N>.json), shown only when
    they were taken on the library sources this run uses (fingerprint over every kernel source) and at this batch."""
    from llm_quest_amd import fingerprint as F

    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles", f"{F.EVIDENCE_ROUND}_pmc_tcc_step_config{config}.json")
    try:
        with open(path) as f:
            d = json.load(f)
    except (OSError, ValueError):
        return {"traffic": None, "traffic_note": f"no counter passes are committed for this configuration ({os.path.basename(path)})"}
    if d.get("all_sources_sha") != F.all_sources_sha():
        return {"traffic": None, "traffic_note": "traffic withheld: the committed counter passes were taken on other kernel sources (re-collect: tools/collect_evidence.sh)"}
    if d.get("per_gpu_batch") != batch:
        return {"traffic": None, "traffic_note": f"the committed counter passes were taken at per-GPU batch {d.get('per_gpu_batch')}"}
    return {"traffic": d["per_step"]["total_bytes"],
            "traffic_note": "memory-side bytes PER STEP: 2 x FETCH_SIZE (gfx950 correction) + WRITE_SIZE over every kernel of one step, separate rocprofv3 --pmc passes over "
                            f"`bench.py --config {config}` ({os.path.basename(path)}, per-kernel table inside; fingerprint of all kernel sources checked)"}


def run_other_config(args):
    from llm_quest_amd import _lib, ddp

    spec = OTHER_CONFIGS[args.config]
    if args.gpus > spec["max_gpus"]:
        raise SystemExit(f"--config {args.config} is specified on {spec['max_gpus']} MI355X (BASELINE.json): --gpus {args.gpus} is not a configuration of it")
    if args.gpus > 1 and "WORLD_SIZE" not in os.environ:
        if torch.cuda.device_count() < args.gpus:
            raise SystemExit(f"--gpus {args.gpus} but only {torch.cuda.device_count()} GPU(s) are visible")
        raise SystemExit(launch_ranks(args.gpus))
    if int(os.environ.get("WORLD_SIZE", "1")) != args.gpus:
        raise SystemExit(f"--gpus {args.gpus} but WORLD_SIZE={os.environ.get('WORLD_SIZE', '1')}")
    rank, world, local = ddp.init_from_env()
    if not torch.cuda.is_available():
        raise SystemExit("bench.py needs an MI355X: the HIP path has no CPU fallback")
    torch.cuda.set_device(local)
    device = torch.device("cuda", local)
    _lib.load()
    batch = args.batch if args.batch_given else spec["batch"]
    power = BoardPower() if rank == 0 else None
    step, sync, state = _other_config_step(args.config, batch, device, rank)

    def fence():
        if world > 1:
            torch.distributed.barrier()
        torch.cuda.synchronize()

    for _ in range(args.warmup):
        loss = step()
    fence()
    if power is not None:
        power.choose()
        power.mark()
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    ev0.record()
    for _ in range(args.steps):
        loss = step()
    ev1.record()
    fence()
    elapsed = time.perf_counter() - t0
    board_power = power.result() if power is not None else None
    dev_ms = ev0.elapsed_time(ev1)
    if world > 1:
        t = torch.tensor([elapsed], dtype=torch.float64, device=device)
        torch.distributed.all_reduce(t, op=torch.distributed.ReduceOp.MAX)
        elapsed = float(t)
    if rank == 0:
        achieved = spec["flop"] * batch / (elapsed / args.steps) / 1e12
        line = {
            "metric": spec["metric"], "value": round(world * batch * spec["units_per_sample"] * args.steps / elapsed, 1), "unit": spec["unit"], "n_gpus": world,
            "rccl_ranks": world if world > 1 else 0, "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(elapsed / args.steps * 1e3, 3), "higher_is_better": True,
            "scaling": "weak", "vs_baseline": None, "dtype": "bf16", "data": "synthetic",
            "config": {"workload": spec["workload"], "per_gpu_batch": batch, "global_batch": batch * world, "parallelism": f"dp{world}", "units_per_sample": spec["units_per_sample"]},
            "roofline": {"bound": "mfma", "achieved": round(achieved, 1), "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s", "frac": round(achieved / PEAK_BF16_TFLOPS, 4), **_config_traffic(args.config, batch),
                         "basis": f"algorithmic {spec['flop'] / 1e9:.1f} GFLOP/sample (SURVEY 8d) x per-GPU batch / step time; device-side (HIP events) {dev_ms / args.steps:.3f} ms/step"},
            "board_power": board_power,
            "loss": round(float(loss.detach()), 5), "peak_memory_gib": round(torch.cuda.max_memory_allocated(device) / 2**30, 1),
        }
        if world == 1 and args.cpu_baseline == "auto":
            try:
                line["cpu_baseline"] = _other_cpu_baseline(state, {2: 8, 3: 2, 5: 1}[args.config], spec["unit"])
            except Exception as exc:  # the baseline is a reported number, never the measured path
                line["cpu_baseline"] = {"value": None, "unit": spec["unit"], "cores": os.cpu_count(), "kind": "port", "sample": f"failed: {exc!r}"}
        print(json.dumps(line), flush=True)
    if world > 1:
        torch.distributed.barrier()
        torch.distributed.destroy_process_group()


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--config", type=int, choices=[2, 3, 4, 5], default=4, help="which workload: 4 = the headline VLM early-fusion step "
                    "(default; everything below describes it), 2 = ViT-B/16, 3 = Qwen3-0.6B text-only at S = 1024, 5 = Qwen3.5-style VLM -- the same JSON schema for each")
    ap.add_argument("--batch", type=int, default=None, help="per-GPU micro-batch (samples); default 160 for the headline (--config 2 / 3 / 5: 332 / 64 / 32).  Headline: 160 x 709 tokens keep 165 GiB of the 288 GB of HBM live; same-box pairs: 64 -> 34.2 / 34.1 %%, "
                    "128 -> +1.4 %%, 160 -> 35.0 / 34.9 %%, 192 -> level with 160 (202 GiB).  More rounds of tiles per launch amortise every launch's fill and tail.  (92 -- every "
                    "launch a whole number of rounds at batch ~64 -- measured the same as 64: the tail tiles of a partial round run faster, the chip is power-limited)")
    ap.add_argument("--cpu-baseline", choices=["auto", "off"], default="auto")
    ap.add_argument("--ragged", action="store_true", help="text lengths ~ U[256, 512] (padding mask active in attention and loss) instead of all-ones masks")
    ap.add_argument("--optimizer", choices=["on", "off"], default="on", help="also time the same steps with clip + AdamW (reported beside the fwd+bwd metric)")
    ap.add_argument("--vision-ahead", choices=["on", "off"], default="on", help="frozen ViT of the next step's batch on a second stream (vlm_engine.VisionAhead), as the training loop runs it")
    ap.add_argument("--pipe-probe", choices=["on", "off"], default="on", help="N = 1: also time the matrix pipe alone on random operands for 2 s (kernels.mfma_pipe_rate) -- the rate this board's "
                    "power cap allows, printed beside the dense peak the roofline is priced against")
    ap.add_argument("--tower", choices=["default", "fp32", "bf16"], default="default", help="arithmetic of the frozen vision tower (vit_model.tower_precision): fp32 = the reference's "
                    "(vlm_engine.py:99-104 runs the ViT outside autocast; split-bf16 GEMMs + exact-fp32 attention), bf16 = bf16 MFMA operands on an fp32 residual stream; default = the package's default")
    ap.add_argument("--fp32-tower-leg", choices=["on", "off"], default="on", help="N = 1: also time the same steps with the frozen tower at the reference's fp32 precision (`with_fp32_tower`)")
    ap.add_argument("--other-configs", choices=["on", "off"], default="on", help="N = 1, default batch: append BASELINE configs 2 / 3 / 5 (5 steps each, child processes) as `other_configs`")
    ap.add_argument("--serve", default=None, metavar="MODEL", help="instead of the training step: serving throughput (prompts and one-token steps, random weights) of a registry "
                    "model -- `gemepel` or `mepatar` beside the Qwen3.5 hybrid text stack, `mopalorn` beside a Mepatar stack of attention layers, `gepilix` beside the Mepatar hybrid, `foderax` beside Gemepel, `pavisun` beside a Mepatar stack of attention layers with routed experts -- at equal width and depth (llm_quest_amd/serve_bench.py); --steps / --warmup count one-token steps")
    ap.add_argument("--serve-sizes", default="1024x8,2048x16", help="--serve: width x attention heads, comma separated")
    ap.add_argument("--serve-only", action="store_true", help="--serve: skip the reference model's rows")
    args = ap.parse_args()
    if args.serve:
        from llm_quest_amd import serve_bench

        sizes = tuple(tuple(int(v) for v in s.split("x")) for s in args.serve_sizes.split(","))
        serve_bench.run(args.serve, steps=max(args.steps, 8), warmup=args.warmup, sizes=sizes, batch=args.batch or 8, with_reference=not args.serve_only)
        return
    args.batch_given = args.batch is not None
    if args.batch is None:
        args.batch = 160

    if args.gpus < 1:
        raise SystemExit("--gpus must be >= 1")
    if args.config != 4:
        return run_other_config(args)
    # MI355_DDP_REHEARSAL=1 (one-GPU boxes only): the N ranks share the visible GPUs round-robin and exchange over gloo -- every line of the N > 1 path
    # (rank start-up, broadcast, bucketed exchange on the communication stream, split tied-weight bucket, barriers, max-over-ranks timing, the one
    # JSON line) runs except RCCL itself.  The line it prints carries "rehearsal": true and is no measurement.
    rehearsal = os.environ.get("MI355_DDP_REHEARSAL") == "1"
    if rehearsal and args.gpus > torch.cuda.device_count() and args.batch * args.gpus > 192 * max(torch.cuda.device_count(), 1):
        raise SystemExit("rehearsal: the ranks share the visible GPU(s) -- pass a small --batch (e.g. 8), the default would not fit")
    if args.gpus > 1 and "WORLD_SIZE" not in os.environ:
        n_dev = torch.cuda.device_count()  # counts devices without creating a HIP context
        if n_dev < args.gpus and not rehearsal:
            raise SystemExit(f"--gpus {args.gpus} but only {n_dev} GPU(s) are visible")
        raise SystemExit(launch_ranks(args.gpus))

    from llm_quest_amd import _lib, ddp
    from llm_quest_amd.multimodal.vlm_engine import VisionAhead, vlm_step_loss

    if int(os.environ.get("WORLD_SIZE", "1")) != args.gpus:  # before any rendezvous: a mismatched launch must fail at once, not wait for peers
        raise SystemExit(f"--gpus {args.gpus} but WORLD_SIZE={os.environ.get('WORLD_SIZE', '1')}: start one rank per GPU (python bench.py --gpus N does it itself)")
    rank, world, local = ddp.init_from_env("gloo" if rehearsal else None)
    if not torch.cuda.is_available():
        raise SystemExit("bench.py needs an MI355X: the HIP path has no CPU fallback")
    if rehearsal:
        local = local % torch.cuda.device_count()
    torch.cuda.set_device(local)
    device = torch.device("cuda", local)
    _lib.load()
    power = BoardPower() if rank == 0 else None

    vit, vit_cfg, ad, llm, llm_cfg = build_models(device)
    if args.tower != "default":
        vit.tower_precision = args.tower
    from llm_quest_amd.multimodal.vision_transformer.vit_model import tower_precision

    tower = tower_precision(vit)
    sync = ddp.sync_for_vlm(llm, ad)
    sync.broadcast_parameters([llm, ad, vit])
    img, ids, mask = synthetic_batch(args.batch, device, seed=123 + rank, ragged=args.ragged)

    n_targets = mask.sum()  # this rank's target tokens: ragged shards weight their mean loss by it (ddp.GradSync.loss_weight)
    # The frozen tower runs one batch ahead on a second stream, exactly as vlm_training_loop_simple runs it: every step takes the hidden
    # states submitted during the previous step and submits the next batch's (here the same synthetic images) -- one ViT forward per
    # step, inside the timed region, concurrent with the decoder instead of in front of it.
    ahead = VisionAhead(vit) if args.vision_ahead == "on" else None
    if ahead is not None:
        ahead.submit(img)

    tower_at = os.environ.get("MI355_BENCH_TOWER_AT", "start")  # A/B: where in the step the next batch's tower forward is submitted to the side stream

    cached_hidden = []

    def vision():
        if ahead is None:
            return None
        if tower_at == "never":  # TIMING ABLATION ONLY: the tower's forward runs once, outside the timed steps -- what the tower costs the step is the difference
            if not cached_hidden:
                cached_hidden.append(ahead.take(img))
            return cached_hidden[0]
        h = ahead.take(img)
        if tower_at == "start":
            ahead.submit(img)
        return h

    def step():
        loss = vlm_step_loss(vit, llm, ad, img, ids, mask, hf_vit_model=False, vit_hidden=vision())
        if ahead is not None and tower_at == "backward":
            ahead.submit(img)
        sync.begin_step(embedding_tokens=ids.numel())  # the tied head / embedding bucket: dense or in two parts, by bytes (ddp.GradSync.split_pays)
        (loss * sync.loss_weight(n_targets) if (args.ragged and world > 1) else loss).backward()
        sync.finish_step()
        llm.zero_grad(set_to_none=True)
        ad.zero_grad(set_to_none=True)
        return loss

    def fence():
        if world > 1:
            torch.distributed.barrier()
        torch.cuda.synchronize()

    for _ in range(args.warmup):
        loss = step()
    fence()
    if power is not None:
        power.choose()
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    if power is not None:
        power.mark()
    t0 = time.perf_counter()
    ev0.record()
    for _ in range(args.steps):
        loss = step()
    ev1.record()
    fence()
    elapsed = time.perf_counter() - t0
    board_power = power.result() if power is not None else None
    dev_ms = ev0.elapsed_time(ev1)
    if world > 1:
        t = torch.tensor([elapsed], dtype=torch.float64, device=device)
        torch.distributed.all_reduce(t, op=torch.distributed.ReduceOp.MAX)
        elapsed = float(t)
    loss_gpu = float(loss.detach())

    # The metric is forward + backward, the optimizer step excluded.  So that nothing of a real
    # training step is left unmeasured, the same K steps are timed again WITH the optimizer: global-norm clip 1.0 + AdamW on the
    # parameter arenas (llm_quest_amd/optim.py::ArenaAdamW), reported beside `value`, never instead of it.
    train_step = None
    if args.optimizer == "on":
        from llm_quest_amd.optim import ArenaAdamW

        opt = ArenaAdamW(list(llm.parameters()) + list(ad.parameters()), lr=1e-5, weight_decay=0.01, max_grad_norm=1.0)
        opt.attach(llm, ad)

        def full_step():
            loss_ = vlm_step_loss(vit, llm, ad, img, ids, mask, hf_vit_model=False, vit_hidden=vision())
            sync.begin_step(embedding_tokens=ids.numel())
            (loss_ * sync.loss_weight(n_targets) if (args.ragged and world > 1) else loss_).backward()
            sync.finish_step()
            opt.step()
            opt.zero_grad(set_to_none=True)
            return loss_

        for _ in range(max(args.warmup, 1)):
            full_step()
        fence()
        t1 = time.perf_counter()
        for _ in range(args.steps):
            full_step()
        fence()
        el2 = time.perf_counter() - t1
        if world > 1:
            t = torch.tensor([el2], dtype=torch.float64, device=device)
            torch.distributed.all_reduce(t, op=torch.distributed.ReduceOp.MAX)
            el2 = float(t)
        train_step = {"what": "the same steps including the optimizer: global-norm clip 1.0 + AdamW (ArenaAdamW, one fused launch per parameter arena)",
                      "ms_per_step": round(el2 / args.steps * 1e3, 3), "value": round(world * args.batch * UNITS_PER_SAMPLE * args.steps / el2, 1), "unit": "img+tok/s"}

    # The reference's VLM loop runs the frozen tower in fp32 (vlm_engine.py:99-104, outside autocast); the package's default tower multiplies bf16
    # operands.  So that the line also carries the step at the reference's precision, the same K steps are timed once more with
    # vit.tower_precision = "fp32" (split-bf16 GEMMs + exact-fp32 attention: hidden states within 1e-4 of the oracle's), reported beside `value`.
    fp32_tower = None
    if world == 1 and tower != "fp32" and args.fp32_tower_leg == "on":
        vit.tower_precision = "fp32"
        for _ in range(max(args.warmup, 2)):  # (the first step still takes hidden states submitted by the bf16 tower)
            step()
        fence()
        t2 = time.perf_counter()
        for _ in range(args.steps):
            loss32 = step()
        fence()
        el3 = time.perf_counter() - t2
        fp32_tower = {"what": "the same steps with the frozen tower at the reference's fp32 precision (vit.tower_precision = 'fp32'; bench.py --tower fp32 makes it the headline)",
                      "ms_per_step": round(el3 / args.steps * 1e3, 3), "value": round(args.batch * UNITS_PER_SAMPLE * args.steps / el3, 1), "unit": "img+tok/s",
                      "frac": round(ALGO_FLOP_PER_SAMPLE * args.batch / (el3 / args.steps) / 1e12 / PEAK_BF16_TFLOPS, 4), "loss": round(float(loss32.detach()), 5)}
        vit.tower_precision = tower
        step()  # (drains the fp32 hidden states in flight, so that the legs below run the default tower again)

    if rank == 0:
        ms_per_step = elapsed / args.steps * 1e3
        value = world * args.batch * UNITS_PER_SAMPLE * args.steps / elapsed
        achieved = ALGO_FLOP_PER_SAMPLE * args.batch / (elapsed / args.steps) / 1e12  # per GPU
        line = {
            "metric": "img+tokens/sec fwd+bwd, ViT-B+Qwen3-0.6B VLM, 224px+512tok",
            "value": round(value, 1), "unit": "img+tok/s", "n_gpus": world, "rccl_ranks": world if (world > 1 and not rehearsal) else 0, "steps": args.steps, "warmup": args.warmup,
            **({"rehearsal": True, "rehearsal_note": "ranks share the visible GPU(s) and exchange over gloo: a run of the N > 1 code path, not a measurement"} if rehearsal else {}),
            "ms_per_step": round(ms_per_step, 3), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "bf16", "data": "synthetic",
            "config": {
                "workload": "BASELINE configs[3]: VLM early fusion, ViT-B/16 (frozen, fwd) + ffn adapter 768->3072->1024 + Qwen3-0.6B, "
                            "224x224 image + 512 text tokens (S=709), fwd+loss+bwd, no optimizer step",
                "per_gpu_batch": args.batch, "global_batch": args.batch * world, "parallelism": f"dp{world}", "text_mask": "ragged U[256,512]" if args.ragged else "all ones",
                "units_per_sample": UNITS_PER_SAMPLE,
                "vision_tower": "frozen ViT forward of the NEXT step's batch on a second HIP stream, one per timed step (vlm_engine.VisionAhead)" if ahead is not None else "in front of the decoder, same stream",
                "vision_tower_precision": tower + (" (the reference's: fp32-grade split-bf16 GEMMs + exact-fp32 attention)" if tower == "fp32" else " MFMA operands, fp32 residual stream"),
                **({"ABLATION": f"MI355_BENCH_TOWER_AT={tower_at}: not the workload (the tower's forward is submitted elsewhere or left out of the timed steps)"} if tower_at != "start" else {}),
            },
            "roofline": {
                "bound": "mfma", "achieved": round(achieved, 1), "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s",
                "frac": round(achieved / PEAK_BF16_TFLOPS, 4), "traffic": None,
                "traffic_note": "not collected",
                "basis": "algorithmic 2.566 TFLOP/sample (SURVEY 8d) x per-GPU batch / step time; device-side (HIP events) "
                         f"{dev_ms / args.steps:.3f} ms/step",
            },
            "board_power": board_power,
            "loss": round(loss_gpu, 5), "peak_memory_gib": round(torch.cuda.max_memory_allocated(device) / 2**30, 1),
        }
        if world > 1:  # how the N > 1 step's large NT GEMMs were launched: on the persistent kernel, or on the per-tile kernel inside a window behind a bucket group (ddp.GradSync)
            from llm_quest_amd import kernels as K_

            line["gemm_windows"] = dict(K_._WINDOW.stats, bucket_blocks=sync.bucket_blocks, window_launches=sync.window_launches, window_sized_from_measurements=sync.window_auto)
        if train_step is not None:
            line["with_optimizer_step"] = train_step
        if fp32_tower is not None:
            line["with_fp32_tower"] = fp32_tower
        if world == 1 and args.pipe_probe == "on":
            from llm_quest_amd import kernels as K_

            pipe = K_.mfma_pipe_rate(2.0)
            pipe16 = K_.mfma_pipe_rate(2.0, shape="16x16x32")
            line["roofline"]["power_capped_pipe"] = {
                "rate": round(pipe, 1), "unit": "TFLOP/s", "achieved_over_rate": round(achieved / pipe, 4),
                "rate_16x16x32": round(pipe16, 1), "achieved_over_rate_16x16x32": round(achieved / pipe16, 4),
                "what_16x16x32": "the same on v_mfma_f32_16x16x32_bf16, the shape the GEMMs issue (32 products on a 128 x 64 wave tile's twelve fragments per repetition)",
                "what": "v_mfma_f32_32x32x16_bf16 on every SIMD, random bf16 operands in registers, no memory traffic, measured on this board right after the timed steps: on random data the "
                        "board's power cap holds the pipe itself below the 2 500 TFLOP/s of `peak` (DESIGN.md section 5)"}
        if world == 1:
            line["roofline"]["dominant_kernel"] = {"name": "gemm_quad_kernel / gemm_quad_grouped_kernel (256x256 tiles by four waves of 128x128: NT projections, a persistent workgroup per CU; the block's weight gradients as one grouped launch)", "hip_event_timing": dominant_kernel_rate(args.batch, device)}
            pmc, why_gemm = pmc_traffic()
            step_pmc, why_step = pmc_step_traffic()
            pmc_batch = step_pmc.get("per_gpu_batch") if step_pmc else None
            if step_pmc is not None and pmc_batch != args.batch:  # the PMC passes were taken at another batch's shapes
                line["roofline"]["traffic_note"] = f"the committed counter passes were taken at per-GPU batch {pmc_batch}"
            elif step_pmc is None:
                line["roofline"]["traffic_note"] = "traffic withheld: " + why_step
            else:
                line["roofline"]["traffic"] = step_pmc["per_step"]["total_bytes"]
                line["roofline"]["traffic_note"] = (
                    "memory-side bytes PER STEP (like `achieved`): 2 x FETCH_SIZE (gfx950 correction) + WRITE_SIZE summed over every kernel of one step, separate "
                    "rocprofv3 --pmc passes over this bench (profiles/<round>_pmc_tcc_step.json, per-kernel table inside; fingerprint of the kernel sources checked); "
                    "Infinity-Cache hits are counted in FETCH_SIZE")
            if pmc is not None and pmc_batch == args.batch:
                line["roofline"]["dominant_kernel"]["pmc_bytes_per_launch"] = {f: pmc[f]["hbm_bytes"] for f in pmc}
                line["roofline"]["dominant_kernel"]["over_algorithmic"] = {f: pmc[f]["over_algorithmic"] for f in pmc}
            elif pmc is None:
                line["roofline"]["dominant_kernel"]["pmc_note"] = "withheld: " + why_gemm
        if world == 1 and args.cpu_baseline == "auto":
            try:
                line["cpu_baseline"] = cpu_baseline(vit, ad, llm, seed=123)
            except Exception as exc:  # the baseline is a reported number, never the measured path
                line["cpu_baseline"] = {"value": None, "unit": "img+tok/s", "cores": os.cpu_count(), "kind": "port", "sample": f"failed: {exc!r}"}
        if world == 1 and args.other_configs == "on" and not args.batch_given and not args.ragged:
            # the other workloads beside the headline (a few steps each, own processes: this one first gives its memory back), so that one record
            # carries them too; `python bench.py --config N` prints each one's full line
            vit = ad = llm = img = ids = mask = ahead = sync = loss = None  # (the closures above see the same cells)
            if args.optimizer == "on":
                opt = None
            import gc

            gc.collect()
            torch.cuda.empty_cache()
            line["other_configs"] = other_configs_block()
        print(json.dumps(line), flush=True)
    if world > 1:
        torch.distributed.barrier()
        torch.distributed.destroy_process_group()


def other_configs_block(steps=5, warmup=2, budget_s=150):
    import subprocess

    out = {}
    for cfg in (2, 3, 5):
        cmd = [sys.executable, os.path.abspath(__file__), "--config", str(cfg), "--steps", str(steps), "--warmup", str(warmup), "--cpu-baseline", "off"]
        try:
            r = subprocess.run(cmd, capture_output=True, text=True, timeout=budget_s)
            d = json.loads(r.stdout.strip().splitlines()[-1])
            out[str(cfg)] = {"workload": d["config"]["workload"], "value": d["value"], "unit": d["unit"], "ms_per_step": d["ms_per_step"], "frac": d["roofline"]["frac"],
                             "per_gpu_batch": d["config"]["per_gpu_batch"], "steps": steps, "board_power_w": (d.get("board_power") or {}).get("mean_W")}
        except Exception as exc:  # reported beside the headline, never instead of it
            out[str(cfg)] = {"value": None, "error": repr(exc)[:200]}
    return out


if __name__ == "__main__":
    main()
