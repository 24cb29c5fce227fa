"""Device memory that a pass takes besides the model's."""
import numpy as np
import pytest

from tests import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw,bits", [(dict(), False), (dict(tensor_types={"attn_k": O.Q8_0}), True)])
def test_exact_prompt_keeps_no_room_for_copies_of_weights(kw, bits):
    """A prompt in the host's order runs its MatMuls from packed activations: the pass's workspace is a few rows of activations and scores, not the fp16 copy of the
    largest weight matrix (90 MB at this width) -- with the steps fused around the MatMuls, and operator by operator (wq and wk of different types).
    The latter's logits have the oracle's bits."""
    from spy_amd import _lib as H
    from spy_amd import model as M
    from tests.model_util import OracleModel
    cfg = M.Config.llama2_7b(n_ctx=128, wtype=O.Q4_0, **kw)
    cfg.n_layer, cfg.n_vocab = 1, 512
    tensors = M.synth_model(cfg, seed=3)
    prompt = np.random.default_rng(2).integers(0, cfg.n_vocab, 40).astype(np.int32)
    eng = M.Engine(cfg, tensors)
    prev = H.load().spy_hip_set_exact_order(1)               # a model whose wq and wk differ has no passes of order 1: the library-wide switch then
    try:
        H.sync()
        before = H.device_info()["free_mem"]
        logits = eng.forward_last(prompt, 0)
        taken = before - H.device_info()["free_mem"]
    finally:
        H.load().spy_hip_set_exact_order(prev)
    print("workspace of a 40-token pass: %.1f MB" % (taken / 1e6), flush=True)
    # 40 tokens: 10 rows of n_embd, 3 of n_ff and the packed n_ff as floats, 32 heads x 128 scores and probabilities: 13 MB (and what
    # the process's first pass loads, some 20 MB)
    assert taken < 60e6
    if bits:
        want = OracleModel(cfg, tensors, nthread=8).forward(prompt, 0)[-1]
        assert np.array_equal(logits.view(np.uint32), want.view(np.uint32))
    eng.close()


def test_own_order_prompt_where_only_the_embedding_is_whole_super_blocks(monkeypatch):
    """n_embd a multiple of 256, n_ff not: wq, wk, wv, wo, gate and up run from packed activations (2.25 bytes per element) and down from Q8_0 blocks of rows that are hardly
    longer (1.06), so the workspace has to be sized by the former.  The same bits as the tile kernels, and the next allocation, made right behind, stays as it is."""
    from spy_amd import _lib as H
    from spy_amd import model as M
    from tests.gpu_util import dev_empty
    cfg = M.Config.llama2_7b(n_ctx=512, wtype=O.Q4_0)
    cfg.n_layer, cfg.n_vocab, cfg.n_ff = 1, 512, 4160
    tensors = M.synth_model(cfg, seed=5)
    prompt = np.random.default_rng(3).integers(0, cfg.n_vocab, 400).astype(np.int32)
    got = {}
    for forced in (None, "tile"):
        if forced: monkeypatch.setenv("SPY_HIP_GEMM", forced)
        else: monkeypatch.delenv("SPY_HIP_GEMM", raising=False)
        eng = M.Engine(cfg, tensors)
        eng.set_order(0)
        eng.forward(prompt, 0, want_logits=False)            # the workspace is allocated here
        guard = dev_empty(64 << 20, 0xA5)
        got[forced] = eng.forward_last(prompt, 0)
        H.sync()
        assert (guard.download(np.uint8) == 0xA5).all()
        eng.close()
    assert np.isfinite(got[None]).all() and np.array_equal(got[None].view(np.uint32), got["tile"].view(np.uint32))
