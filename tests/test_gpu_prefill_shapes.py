"""Prefill kernels at the edges of their tiles: prompt lengths around the chunk
and the time steps a thread takes, two groups, and a prompt with enough rows
for the long-column form of the conv, against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import MAXREL, max_rel

pytestmark = pytest.mark.gpu


def _check(ctx, act, wfmt, B, Lq, name="mamba2-130m", **over):
    from lite_ssm_amd.model import DeviceModel, Engine, shape
    print(f"case: prefill {name} {over} act {act} fmt {wfmt} {B} x {Lq}", flush=True)
    sh = shape(name, vocab_size=512, **over)
    m = DeviceModel(sh, act=act, wfmt=wfmt, seed=3)
    om = O.Model(m.to_host(), vars(sh), act, wfmt)
    eng = Engine(ctx, m, max_batch=B, max_seq=Lq)
    g = torch.Generator().manual_seed(Lq)
    ids = torch.randint(0, sh.vocab_size, (B, Lq), generator=g, dtype=torch.int32)
    nxt = torch.zeros(B, dtype=torch.int32, device="cuda")
    eng.prefill(ids.cuda(), nxt)
    conv, ssd = om.new_state(B)
    ref = O.from_act(om.prefill(conv, ssd, ids.numpy()), act)
    assert max_rel(eng.logits(B).float().cpu().numpy(), ref) <= MAXREL[act]
    gconv, gssd = eng.state()
    assert max_rel(gssd.cpu().numpy(), ssd) < MAXREL[act]
    assert max_rel(gconv.float().cpu().numpy().reshape(-1), O.from_act(conv, act).reshape(-1)) < MAXREL[act]
    eng.close()


# lengths below the conv's width, around 4 and 8 time steps a thread, and around
# one and two chunks of 64
@pytest.mark.parametrize("act,wfmt", [(O.F16, O.W_Q8_G32), (O.BF16, O.W_Q4_G64)])
@pytest.mark.parametrize("Lq", [2, 3, 4, 5, 17, 36, 63, 64, 65, 127, 129])
def test_prefill_lengths_vs_oracle(ctx, act, wfmt, Lq):
    _check(ctx, act, wfmt, 2, Lq, n_layer=2)


@pytest.mark.parametrize("act,wfmt", [(O.F16, O.W_DENSE), (O.BF16, O.W_Q4_G64)])
def test_prefill_two_groups_vs_oracle(ctx, act, wfmt):
    _check(ctx, act, wfmt, 2, 70, n_layer=2, n_groups=2)


def test_prefill_long_columns_vs_oracle(ctx):
    """16 time steps a thread (enough blocks for two per CU in one stream)."""
    _check(ctx, O.BF16, O.W_Q4_G64, 1, 3290, name="mamba2-2.7b", n_layer=1)
