"""One-row LM head of a Whisper / Llama model through the streaming GEMM at several persistent grid
caps (workgroups; 4-wave workgroups at K < 2048): more co-resident workgroups = more waves per CU
streaming the 133 MB (Whisper-large-v3) head.  The Infinity Cache is flushed between launches
(a 512 MB copy) so the head streams from HBM as it does after a decode step.

    python tools/lm_head_probe.py [--asr whisper-large-v3] [--caps 256,512,768,1024] [--iters 50]
"""
import argparse
import dataclasses
import json
import os
import statistics
import sys

import torch

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
from voice_enabled_browser_automation_amd import ops  # noqa: E402
from voice_enabled_browser_automation_amd.models.config import get_config  # noqa: E402
from voice_enabled_browser_automation_amd.models.whisper import WhisperModel  # noqa: E402


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--asr", default="whisper-large-v3")
    ap.add_argument("--caps", default="256,512,768,1024")
    ap.add_argument("--iters", type=int, default=50)
    a = ap.parse_args()
    E = ops.ext()
    cfg = dataclasses.replace(get_config(a.asr), n_enc_layers=1, n_dec_layers=2)
    m = WhisperModel(cfg, device="cuda", seed=0, tile_decoder=True)
    w, b, c = m.f_lm
    torch.manual_seed(0)
    x = torch.randn(1, cfg.d_model, device="cuda").to(torch.bfloat16)
    out = torch.empty(1, w.shape[0], dtype=torch.float32, device="cuda")
    flush_a = torch.empty(256 << 20, dtype=torch.int16, device="cuda")
    flush_b = torch.empty_like(flush_a)
    ref = None
    res = {}
    for cap in [int(v) for v in a.caps.split(",")]:
        E.set_skinny_mode(1, cap, 0)
        ts = []
        for i in range(a.iters + 3):
            flush_b.copy_(flush_a)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            ops.linear(x, w, b, out=out, eps=cfg.ln_eps, ln_c=c)
            e1.record()
            e1.synchronize()
            if i >= 3:
                ts.append(e0.elapsed_time(e1) * 1e3)
        if ref is None:
            ref = out.clone()
        same = bool(torch.equal(out, ref))
        res[cap] = dict(us=round(statistics.median(ts), 2), same_bits=same)
        print(json.dumps(dict(tool="lm_head_probe", asr=a.asr, grid_cap=cap, us=res[cap]["us"],
                              tb_s=round(w.numel() * 2 / (statistics.median(ts) * 1e-6) / 1e12, 2),
                              same_bits=same)), flush=True)
    E.set_skinny_mode(1, 256, 0)


if __name__ == "__main__":
    main()
