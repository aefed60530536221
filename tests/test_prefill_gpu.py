"""Attention of prompt passes in its other forms: 64 query rows a workgroup
(taken once those workgroups cover the chip; smaller prompts take 32), at each
head size and with a last tile that is not full, and prompts of one stream
longer than a pass, whose later rows attend to cached keys.  Against the
oracle's token-by-token logits (the bars of parity_util)."""
import numpy as np
import pytest

from parity_util import compare_logits
from test_decoder_gpu import build, prompts
from test_wide_gpu import prompt_cfg

pytestmark = pytest.mark.gpu

PASS_ROWS = 2048  # tokens x streams of a pass


def blocks64(cfg, batch, tokens):
    """Workgroups of 64 query rows of a pass; from 256 on it takes that form."""
    g = cfg.n_heads // cfg.n_kv_heads
    return -(-tokens * g // 64) * cfg.n_kv_heads * batch


def check(xe, gpu, cfg, batch, n, label):
    dec, om = build(xe, gpu, cfg, seed=53, batch=batch)
    assert dec.prompt_pass(batch, n - 1) == min(n - 1, PASS_ROWS // batch)
    pr = prompts(cfg, batch, n, seed=batch + n)
    dec.feed(pr[:, :-1])
    got, _ = dec.step(pr[:, -1], np.full(batch, n - 1, np.int32))
    dec.feed(pr[:, :-1])
    again, _ = dec.step(pr[:, -1], np.full(batch, n - 1, np.int32))
    assert np.array_equal(np.asarray(got).view(np.uint32), np.asarray(again).view(np.uint32))
    for p in range(n):
        want = om.step(pr[:, p], np.full(batch, p, np.int32))
    compare_logits(got, want, label)
    dec.close()
    om.close()


@pytest.mark.parametrize("family,wd,heads,kv,hd,batch,n", [
    ("opt", "i8", 12, 12, 64, 4, 391), ("opt", "bf16", 4, 4, 64, 64, 33), ("whisper", "i8", 12, 12, 64, 30, 51),
    ("gemma", "i8", 16, 8, 128, 8, 131), ("gemma", "bfp16", 16, 4, 256, 8, 151), ("gemma", "i8", 4, 1, 256, 256, 9)])
def test_prompt_attention_of_64_rows(gpu, xe, monkeypatch, family, wd, heads, kv, hd, batch, n):
    monkeypatch.delenv("XE_STEP", raising=False)
    cfg = prompt_cfg(xe, family, wd).replace(n_heads=heads, n_kv_heads=kv, head_dim=hd)
    if family != "gemma":
        cfg = cfg.replace(d_model=heads * hd, max_pos=448, max_ctx=448)
    print("[case] 64-row attention %s %s %d/%d x %d batch %d, %d tokens" % (family, wd, heads, kv, hd, batch, n), flush=True)
    assert blocks64(cfg, batch, n - 1) >= 256
    check(xe, gpu, cfg, batch, n, "prompt64-%s-%s-hd%d-b%d-n%d" % (family, wd, hd, batch, n))


@pytest.mark.parametrize("family,wd,batch,n", [("gemma", "i8", 1, 2150), ("gemma_hd128", "bf16", 1, 2101), ("gemma", "i8", 16, 200),
                                               ("opt", "i8", 1, 2080)])
def test_prompt_beyond_one_pass(gpu, xe, monkeypatch, family, wd, batch, n):
    monkeypatch.delenv("XE_STEP", raising=False)
    cfg = prompt_cfg(xe, family, wd).replace(max_ctx=2304, max_pos=2304)
    print("[case] beyond one pass %s %s batch %d, %d tokens" % (family, wd, batch, n), flush=True)
    assert batch * (n - 1) > PASS_ROWS
    check(xe, gpu, cfg, batch, n, "prompt-long-%s-%s-b%d-n%d" % (family, wd, batch, n))
