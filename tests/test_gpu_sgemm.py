"""GPU checks of the streaming grouped GEMMs in their bf16 forms (k_sgemm; run with -m gpu).

Batches past the decode kernel's run them on the general path: with 32 pairs per
unit below 16 tokens per expert, with 64 from there on where the widths do not fit
the FP4 form (test_gpu_fgemm.py). Checked against the per-16-token streams on the
same routing (the same products, summed in fp32 in another order, so the bf16
roundings of gate, up, h and y flip now and then: the bar of the grouped GEMMs'
comparison) at the edges of the units: 1 to 33, 48 and 49, 64 and 65 and 129 tokens
of an expert (partly filled 16-token tiles, one to five groups), reductions of 1 to
28 k-steps, odd counts, scale rows that are not whole 16-byte words, a partial row
block, and no expert active twice in a row.
"""

import pytest
import torch

import k3moe
from k3moe import synthetic
from k3moe.configs import MoEConfig
from oracle import moe_ref

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def both(cfg, seed, dev, routes=None):
    g = {k: (v.to(dev) if isinstance(v, torch.Tensor) else v) for k, v in
         synthetic.moe_layer_inputs(cfg, seed, scale_mode='kimi').items()}
    kw = dict(topk=cfg.topk, gating=cfg.gating, activation=cfg.activation, routes=routes, latent=g.get('latent'))
    outs = {p: k3moe.moe_step(*synthetic.step_args(g), path=p, **kw) for p in ('general', 'streamed')}
    torch.cuda.synchronize(dev)
    return outs['general'], outs['streamed']


def check(a, b):
    assert torch.equal(a['expert_ids'], b['expert_ids'])
    assert torch.equal(a['route_weights'], b['route_weights'])
    assert bool(torch.isfinite(a['expert_sum']).all())
    assert moe_ref.rel_l2(a['expert_sum'].cpu(), b['expert_sum'].cpu()) < 2e-3


@pytest.mark.parametrize('cfg', [
    MoEConfig('sgemm-i128', 24, 4, 512, 128, 70),                               # 4 and 1 k-steps
    MoEConfig('sgemm-k640-i384', 32, 4, 640, 384, 100, activation='silu'),      # narrow scales, a partial row block
    MoEConfig('sgemm-i512', 16, 2, 1024, 512, 90, gating='softmax'),            # whole scale words in both
    MoEConfig('sgemm-k3584-i384', 48, 16, 512, 384, 66, latent=3584),           # 64 pairs per unit, four scale chunks
    MoEConfig('sgemm-b800', 896, 16, 256, 128, 800, latent=512),                # many groups
], ids=lambda c: c.name)
def test_streaming_gemms_match_the_streams(gpu, cfg):
    say(f'case: {cfg.name} seed=6 general (k_sgemm) vs streamed')
    check(*both(cfg, 6, gpu))


@pytest.mark.parametrize('counts', [(1, 16, 17, 32, 33), (64, 65, 2, 1), (15, 31, 48)])
def test_streaming_gemms_token_counts(gpu, counts):
    """Forced routes that give experts exactly these token counts; every token's second expert spreads over the rest."""
    B, E = sum(counts), 64
    cfg = MoEConfig('sgemm-counts', E, 2, 768, 256, max(B, 65))
    first = [e for e, n in enumerate(counts) for _ in range(n)] + [len(counts)]*(cfg.tokens - B)
    lo = len(counts) + 1
    routes = torch.tensor([[e, lo + t % (E - lo)] for t, e in enumerate(first)], dtype=torch.int64, device=gpu)
    say(f'case: {cfg.name} tokens per expert {counts} seed=1')
    check(*both(cfg, 1, gpu, routes))


@pytest.mark.parametrize('K,I', [(640, 384), (640, 1536), (3584, 640)])
@pytest.mark.parametrize('counts', [(33, 48, 49, 64, 65, 129), (1, 16, 17, 130, 31, 193)])
def test_units_of_64_pairs_token_counts(gpu, counts, K, I):
    """As above for the units of 64 pairs (at least 16 pairs per expert on average, widths that the FP4 form does not
    take): scale rows of whole words and not in both GEMMs, a partial row block in each."""
    B, E = sum(counts), 20
    cfg = MoEConfig('sgemm64-counts', E, 2, K, I, B)
    assert 2*B >= 16*E and (K % 512 or I % 256)
    first = [e for e, n in enumerate(counts) for _ in range(n)]
    lo = len(counts) + 1
    routes = torch.tensor([[e, lo + t % (E - lo)] for t, e in enumerate(first)], dtype=torch.int64, device=gpu)
    say(f'case: {cfg.name} K={K} I={I} tokens per expert {counts} seed=1')
    check(*both(cfg, 1, gpu, routes))


def moved(t, off, dev):
    """t's copy on dev that starts off bytes past a 256-byte boundary."""
    raw = torch.empty(t.numel()*t.element_size() + off, dtype=torch.uint8, device=dev)
    view = raw[off:].view(t.dtype).view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize('name,off', [('gate_scales', 1), ('up_scales', 3), ('down_scales', 5), ('gate_blocks', 4),
                                      ('down_blocks', 8), ('latent', 4), ('router', 4)])
@pytest.mark.parametrize('cfg', [MoEConfig('sgemm-i128', 24, 4, 512, 128, 70, latent=512),
                                 MoEConfig('sgemm-fp4', 16, 4, 512, 512, 96, gating='softmax', latent=1024)],
                         ids=lambda c: c.name)
def test_tensors_inside_a_word(gpu, cfg, name, off):
    """A tensor that starts inside a 16-byte word (scales: at any byte) takes the kernels with ordinary loads."""
    say(f'case: {cfg.name} {name} at byte {off}')
    inputs = synthetic.moe_layer_inputs(cfg, 3, scale_mode='kimi')
    g = {k: (v.to(gpu) if isinstance(v, torch.Tensor) else v) for k, v in inputs.items()}
    kw = dict(topk=cfg.topk, gating=cfg.gating, activation=cfg.activation)
    want = k3moe.moe_step(*synthetic.step_args(g), latent=g['latent'], path='streamed', **kw)
    g[name] = moved(g[name], off, gpu)
    got = k3moe.moe_step(*synthetic.step_args(g), latent=g['latent'], **kw)
    if name == 'router':
        # the logits' h = 512 products are summed by another kernel, in another order: two fp32 sums differ by at most
        # 2 x 512 x 2^-24 of the products' magnitudes' sum (512 x E|x| x E|w| = 6.5; 9 covers its largest), 5.5e-4, and
        # a weight by no more than its logits
        assert float((got['route_weights'] - want['route_weights']).abs().max()) <= 5.5e-4
        got = {**got, 'route_weights': want['route_weights']}
    check(got, want)


@pytest.mark.parametrize('name', ['latent_down', 'shared_up', 'latent_up', 'shared_down'])
def test_latent_weights_inside_a_word(gpu, name):
    """The latent block's projections past 64 tokens with such a weight: launches of 64 rows, on shapes whose 64-row
    kernels read the weights by ordinary loads."""
    from test_gpu_latent import block_weights, near_oracle
    B, h, lh, S = 100, 512, 256, 128
    say(f'case: latent B={B} h={h} lh={lh} S={S} {name} at byte 4')
    g = {k: v.to(gpu) for k, v in block_weights(B, h, lh, S, 4).items()}

    def both():
        lat, sh = k3moe.latent_in(g['x'], g['latent_down'], g['shared_gate'], g['shared_up'])
        return lat, sh, k3moe.latent_out(g['expert_sum'], g['latent_norm'], g['latent_up'], g['shared_h'],
                                         g['shared_down'])
    g['shared_h'] = k3moe.latent_in(g['x'], g['latent_down'], g['shared_gate'], g['shared_up'])[1]
    want = [t.cpu() for t in both()]
    g[name] = moved(g[name], 4, gpu)
    for t, w, steps in zip(both(), want, (1, 2, 2)):
        near_oracle(t, w, steps=steps, floor=2e-2)
