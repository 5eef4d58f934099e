"""GPU checks of the latent block's GEMMs for more than 64 tokens (k_lgemm; run with -m gpu).

Against the CPU restatement at shapes whose plans take the k-split sums and tiles
of several sizes (ragged token counts, one token past a tile, a row block past
the weights' end), and, at a Kimi K3 TP8 rank's widths, against the kernels for
up to 64 tokens run on 64 rows at a time: the same products summed in fp32 in
another order, so equal but for roundings (near_oracle's bar). Repeated launches
agree bit for bit.
"""

import pytest
import torch

import k3moe
from k3moe import synthetic
from k3moe.configs import MoEConfig
from oracle import latent_ref
from test_gpu_latent import block_weights, near_oracle
from test_gpu_moe import run_and_check

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize('B,h,lh,S', [(65, 1024, 512, 256), (81, 128, 128, 128), (97, 3072, 1536, 512),
                                      (200, 3072, 1536, 512), (333, 3072, 1536, 512), (409, 3072, 1536, 512),
                                      (500, 1024, 1536, 384), (1500, 1024, 512, 256)])
def test_latent_gemms_match_oracle(gpu, B, h, lh, S):
    say(f'case: latent GEMMs B={B} h={h} lh={lh} S={S} seed=5')
    w = block_weights(B, h, lh, S, 5)
    g = {k: v.to(gpu) for k, v in w.items()}
    lat, sh = k3moe.latent_in(g['x'], g['latent_down'], g['shared_gate'], g['shared_up'])
    want_lat, want_sh = latent_ref.latent_in(w['x'], w['latent_down'], w['shared_gate'], w['shared_up'])
    near_oracle(lat, want_lat)
    near_oracle(sh, want_sh, steps=2)
    out = k3moe.latent_out(g['expert_sum'], g['latent_norm'], g['latent_up'], want_sh.to(gpu), g['shared_down'])
    want = latent_ref.latent_out(w['expert_sum'], w['latent_norm'], w['latent_up'], want_sh, w['shared_down'])
    near_oracle(out, want, steps=2, floor=2e-2)


@pytest.mark.parametrize('B', [65, 129, 333, 777, 1025])
def test_latent_gemms_match_64_row_launches(gpu, B):
    h, lh, S = 7168, 3584, 768
    say(f'case: latent GEMMs B={B} h={h} lh={lh} S={S} seed=2 against launches of 64 rows')
    g = {k: v.to(gpu) for k, v in block_weights(B, h, lh, S, 2).items()}
    win = (g['latent_down'], g['shared_gate'], g['shared_up'])
    lat, sh = k3moe.latent_in(g['x'], *win)
    wout = (g['latent_norm'], g['latent_up'])
    out = k3moe.latent_out(g['expert_sum'], *wout, sh, g['shared_down'])
    again = k3moe.latent_in(g['x'], *win), k3moe.latent_out(g['expert_sum'], *wout, sh, g['shared_down'])
    assert torch.equal(again[0][0], lat) and torch.equal(again[0][1], sh) and torch.equal(again[1], out)
    for b0 in range(0, B, 64):
        rows = slice(b0, min(B, b0 + 64))
        plat, psh = k3moe.latent_in(g['x'][rows].contiguous(), *win)
        near_oracle(lat[rows], plat.cpu())
        near_oracle(sh[rows], psh.cpu(), steps=2)
        pout = k3moe.latent_out(g['expert_sum'][rows].contiguous(), *wout, sh[rows].contiguous(), g['shared_down'])
        near_oracle(out[rows], pout.cpu(), steps=2, floor=2e-2)


@pytest.mark.parametrize('E,k,B', [(3, 2, 5), (7, 3, 70), (9, 2, 2), (12, 6, 33), (20, 4, 129), (61, 8, 3)])
def test_router_rows_of_no_whole_blocks(gpu, E, k, B):
    """The router's rows end inside a loader's block of 8 (or before its first ends)."""
    say(f'case: router E={E} k={k} B={B} seed=0')
    cfg = MoEConfig(f'e{E}', E, k, 384, 256, B)
    run_and_check(cfg, synthetic.moe_layer_inputs(cfg, 0, scale_mode='kimi'), gpu, path='general')
