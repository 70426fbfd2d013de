"""The code predictor's layer stack as persistent launches (csrc/cp_chain.hip) against the launch-per-op path of the SAME
library: the chain keeps tiles, k-step ownership, accumulation order and rounding points, so codes AND logits must be
bit-identical; no wait may time out (error word 0).  Reference function: the decoder loop of
qwen3_tts_code_predictor_vllm.py:480-561 (parity of either schedule with the oracle: tests/test_gpu_engine.py)."""
import ctypes as C

import pytest
import torch

from ht_vllm_omni_amd import _lib as L
from ht_vllm_omni_amd.config import get_dims
from ht_vllm_omni_amd.weights import make_weights
from oracle import talker_oracle as O
from tests.util import BF16, assert_e2e_close

pytestmark = pytest.mark.gpu


def _engine(d, w, **kw):
    from ht_vllm_omni_amd.engine import TalkerEngine
    return TalkerEngine(d, w, **kw)


def _inputs(d, w, B, seed):
    g = torch.Generator().manual_seed(seed)
    code0 = torch.randint(1, d.codebook, (B,), generator=g)
    return code0, w["embed"][code0], torch.randn(B, d.hidden, generator=g).to(BF16)


@pytest.mark.parametrize("model,B,span,split48",
                         [(m, B, span, 0) for m, B in (("tts-1.7b", 64), ("tts-1.7b", 37), ("tts-1.7b", 5), ("tts-0.6b", 16), ("tts-1.7b", 32), ("tts-1.7b", 48),
                                                       ("tts-1.7b", 17)) for span in (2, 1)] + [("tts-1.7b", 64, 2, 1), ("tts-1.7b", 53, 2, 1)])
def test_chain_is_bit_identical_to_the_launch_chain(model, B, span, split48):
    """span 1 = one persistent launch per pass (layer stack only), 2 = ONE launch for every pass with its head GEMM and sampler.  split48: above 48 rows
    too the split of the stages that 33 to 48 rows have (16-row gate_up tiles): the bits do not depend on a tile's height (gemm_frag.cuh SlabOrder)."""
    d = get_dims(model).with_(layers=1, max_model_len=256)          # the released predictor: 5 layers, 16 groups
    w = make_weights(d, seed=33, std=0.02)
    code0, e0, lh = _inputs(d, w, B, B)
    res = {}
    with L.debug_library() as lib:
        lib.omni_debug_cp_chain.argtypes = [C.c_int]; lib.omni_debug_cp_chain.restype = None
        lib.omni_debug_chain_mode.argtypes = [C.c_int, C.c_int, C.c_int]; lib.omni_debug_chain_mode.restype = None
        try:
            for on in (0, 1):
                lib.omni_debug_cp_chain(span if on else 0)
                lib.omni_debug_chain_mode(0, int(not split48), 0)
                eng = _engine(d, w, kv_dtype="bf16", num_blocks=8, max_batch=64)
                for rep in range(3):                                 # flags and hand-off buffers carry over from call to call
                    codes, lg = eng.code_predictor(code0.to(torch.int32).cuda(), e0.cuda(), lh.cuda(), greedy=True, return_logits=True)
                    steps = torch.full((B,), 3 + rep, dtype=torch.int32)
                    sampled = eng.code_predictor(code0.to(torch.int32).cuda(), e0.cuda(), lh.cuda(), greedy=False, temperature=0.9,
                                                 top_k=50, seed=7, steps=steps.cuda())
                assert eng.chain_error() == 0 and eng.chains_ran() == on
                res[on] = (codes.cpu(), lg.cpu(), sampled.cpu())
        finally:
            lib.omni_debug_cp_chain(2)
            lib.omni_debug_chain_mode(0, 1, 0)
    bad = (res[1][0] != res[0][0]).any(dim=1).nonzero().flatten().tolist()
    assert torch.equal(res[1][0], res[0][0]), f"greedy codes differ between the persistent chain and the launch chain in rows {bad}: first differing group per row {[int((res[1][0][b] != res[0][0][b]).nonzero()[0]) for b in bad]}"
    assert torch.equal(res[1][1], res[0][1]), "logits differ between the persistent chain and the launch chain"
    assert torch.equal(res[1][2], res[0][2]), "sampled codes differ between the persistent chain and the launch chain"


@pytest.mark.parametrize("top_p", [0.0, 0.9], ids=["top-k", "top-p"])
@pytest.mark.parametrize("B", [1, 15, 31, 33, 49, 63])
def test_all_pass_chain_at_the_edges_of_its_row_splits(B, top_p):
    """The all-pass launch splits its stages over the workgroups by rows (up to 16, 32, 48, 64): at the edges of each, sampled codes (both picks: one
    wave a row, four waves with top-p), greedy codes and logits are the launch path's."""
    d = get_dims("tts-1.7b").with_(layers=1, max_model_len=256)
    w = make_weights(d, seed=12, std=0.02)
    code0, e0, lh = (t.cuda() for t in _inputs(d, w, B, 7 * B))
    res = {}
    with L.debug_library() as lib:
        lib.omni_debug_cp_chain.argtypes = [C.c_int]; lib.omni_debug_cp_chain.restype = None
        try:
            for on in (0, 2):
                lib.omni_debug_cp_chain(on)
                eng = _engine(d, w, kv_dtype="bf16", num_blocks=8, max_batch=64)
                steps = torch.full((B,), 5, dtype=torch.int32, device="cuda")
                sampled = [eng.code_predictor(code0.to(torch.int32), e0, lh, greedy=False, temperature=0.9, top_k=50, top_p=top_p, seed=3, steps=steps) for _ in range(2)]
                codes, lg = eng.code_predictor(code0.to(torch.int32), e0, lh, greedy=True, return_logits=True)
                assert eng.chain_error() == 0 and eng.chains_ran() == (1 if on else 0)
                res[on] = [t.cpu() for t in (*sampled, codes, lg)]
        finally:
            lib.omni_debug_cp_chain(2)
    for x, y in zip(res[0], res[2]):
        assert torch.equal(x, y)


@pytest.mark.parametrize("chain,fused_norm", [(0, None), (2, None), (0, False)], ids=["launches", "chain", "separate-norms"])
@pytest.mark.parametrize("B", [5, 24, 40, 64])
def test_a_row_of_nans_leaves_nothing_behind(B, chain, fused_norm):
    """One row's input is NaN for one call.  What the private K / V cache keeps of it lies past the position of every later pass that has not written
    there again yet: the row's next call, with finite inputs, gives what it gave before."""
    d = get_dims("tts-1.7b").with_(layers=1, max_model_len=256)
    w = make_weights(d, seed=12, std=0.02)
    code0, e0, lh = (t.cuda() for t in _inputs(d, w, B, 3 * B))
    bad = lh.clone()
    bad[B // 2] = float("nan")
    with L.debug_library() as lib:
        lib.omni_debug_cp_chain.argtypes = [C.c_int]; lib.omni_debug_cp_chain.restype = None
        try:
            lib.omni_debug_cp_chain(chain)
            eng = _engine(d, w, kv_dtype="bf16", num_blocks=8, max_batch=64, fused_norm=fused_norm)
            outs = [eng.code_predictor(code0.to(torch.int32), e0, x, greedy=True, return_logits=True) for x in (lh, bad, lh)]
            assert eng.chain_error() == 0
            assert eng.chains_ran() == (1 if chain else 0)
        finally:
            lib.omni_debug_cp_chain(2)
    other = [b for b in range(B) if b != B // 2]
    assert outs[1][1][B // 2].isnan().all(), "the NaN row's logits"
    for first, poisoned, again in zip(*outs):
        assert torch.equal(poisoned[other], first[other]), "another row changed"
        assert torch.equal(again, first), "the NaN row's next call differs"


def test_chain_matches_oracle_at_full_predictor_depth():
    """Product library, chain on (the default): greedy codes / logits of the 5-layer, 16-group predictor vs the oracle."""
    d = get_dims("tts-1.7b").with_(layers=1, max_model_len=256)
    w = make_weights(d, seed=21, std=0.02)
    B = 48
    code0, e0, lh = _inputs(d, w, B, 5)
    eng = _engine(d, w, kv_dtype="bf16", num_blocks=8, max_batch=64)
    codes, lg = eng.code_predictor(code0.to(torch.int32).cuda(), e0.cuda(), lh.cuda(), greedy=True, return_logits=True)
    assert eng.chain_error() == 0
    ref_codes, ref_lg = O.TalkerOracle(d, w).code_predictor(code0, e0, lh, do_sample=False, return_logits=True)
    assert_e2e_close(lg.cpu()[:, 0], ref_lg[:, 0], mean_tol=6e-3, max_ulps=3, what="chain: code predictor logits, group 1 (5 layers)")
    assert (codes.cpu()[:, 1] == ref_codes[:, 1]).float().mean().item() >= 0.9


def _decode_engine(d, w, B, kv="fp8"):
    eng = _engine(d, w, kv_dtype=kv, num_blocks=256, max_batch=64)
    g = torch.Generator().manual_seed(9)
    eng.input_ids[:B] = torch.randint(1, d.codebook, (B,), generator=g).to(torch.int32).cuda()
    eng.last_hidden[:B] = torch.randn(B, d.hidden, generator=g).to(BF16).cuda()
    eng.text_step[:B] = (torch.randn(B, d.hidden, generator=g) * 0.02).to(BF16).cuda()
    eng.positions[:B] = 17
    eng.seq_lens[:B] = 18
    for b in range(B):
        eng.block_table[b, :3] = torch.tensor([1 + 3 * b, 2 + 3 * b, 3 + 3 * b], dtype=torch.int32)
    for c in eng.kv_caches:        # a history to attend to (same bytes in every engine built from this seed)
        c.view(torch.uint8).copy_(torch.randint(0, 120, c.view(torch.uint8).shape, generator=g, dtype=torch.uint8).cuda())
    eng.set_sampling(greedy=0, temperature=0.9, top_k=50, rep_penalty=1.05, seed=42, cp_greedy=0, cp_temperature=0.9, cp_top_k=50)
    return eng


# the released 1.7B width, and one NO released checkpoint has (the stage sets are instantiated from the shape: csrc/bb_chain.hip BB_SHAPES): hidden 1536,
# intermediate 4608, 12 q / 6 kv heads (qkv 3072 wide)
UNRELEASED = dict(hidden=1536, inter=4608, q_heads=12, kv_heads=6)


@pytest.mark.parametrize("mode,B,kv,shape", [("engine", 64, "fp8", None), ("plain-chain", 64, "fp8", None),
                                             ("engine", 49, "bf16", None), ("plain-chain", 49, "bf16", None),
                                             ("plain-chain", 64, "fp8", UNRELEASED), ("plain-chain", 41, "int8", UNRELEASED)])
def test_backbone_segment_chain_against_the_launch_path(B, kv, mode, shape):
    """o_proj -> gate_up -> down_proj -> next qkv as one persistent launch per layer against the launch-per-op backbone of the
    same library at the 1.7B shape.  The chain (csrc/bb_chain.hip bb_flow_kernel) and the debug library's loader / consumer engine (bb_engine.hip) keep the
    launch path's tiles and summation order: logits, hidden state, sampled ids, codes and every KV byte of three decode steps are identical.  No wait
    times out in any mode."""
    d = get_dims("tts-1.7b").with_(layers=3, max_model_len=256, **(shape or {}))
    w = make_weights(d, seed=8, std=0.02)
    res = {}
    with L.debug_library() as lib:
        for fn in (lib.omni_debug_bb_chain, lib.omni_debug_bb_engine):
            fn.argtypes = [C.c_int]; fn.restype = None
        try:
            for on in (0, 1):
                lib.omni_debug_bb_chain(on)
                lib.omni_debug_bb_engine(int(mode == "engine"))
                eng = _decode_engine(d, w, B, kv)
                outs = []
                for _ in range(3):
                    eng.decode_step(B)
                    outs.append((eng.logits[:B].clone(), eng.last_hidden[:B].clone(), eng.input_ids[:B].clone(), eng.audio_codes[:B].clone()))
                torch.cuda.synchronize()
                assert eng.chain_error() == 0
                assert eng.chains_ran() == (3 if on else 1), (on, eng.chains_ran(), "the shape must run BOTH persistent chains")
                res[on] = (outs, [c.view(torch.uint8).clone() for c in eng.kv_caches])
        finally:
            lib.omni_debug_bb_chain(1)
            lib.omni_debug_bb_engine(0)
    for s, (a, b) in enumerate(zip(res[1][0], res[0][0])):
        for name, x, y in zip(("logits", "hidden", "ids", "codes"), a, b):
            assert torch.equal(x, y), f"step {s}: {name} differ between the backbone chain and the launch path"
    for l, (x, y) in enumerate(zip(res[1][1], res[0][1])):
        assert torch.equal(x, y), f"KV cache of layer {l} differs"


@pytest.mark.parametrize("B,kv,shape", [(32, "fp8", None), (23, "bf16", None), (16, "fp8", None), (9, "int8", None), (1, "fp8", None), (40, "fp8", None),
                                        (48, "bf16", None), (33, "int8", None), (27, "fp8", UNRELEASED), (7, "bf16", UNRELEASED)])
def test_backbone_segment_chain_at_1_to_48_rows_against_the_launch_path(B, kv, shape):
    """The backbone segment as a persistent launch at 1 to 48 rows (csrc/bb_chain.hip bb_flow_kernel, split by rows: 16, 32, 64), its last row tile
    partly filled, at the 1.7B width and one that no released checkpoint has: logits, hidden state, ids, codes and every KV byte of three decode steps
    are the launch path's; both chains reported as launched."""
    d = get_dims("tts-1.7b").with_(layers=3, max_model_len=256, **(shape or {}))
    w = make_weights(d, seed=8, std=0.02)
    res = {}
    with L.debug_library() as lib:
        lib.omni_debug_bb_chain.argtypes = [C.c_int]; lib.omni_debug_bb_chain.restype = None
        try:
            for on in (0, 1):
                lib.omni_debug_bb_chain(on)
                eng = _decode_engine(d, w, B, kv)
                outs = []
                for _ in range(3):
                    eng.decode_step(B)
                    outs.append((eng.logits[:B].clone(), eng.last_hidden[:B].clone(), eng.input_ids[:B].clone(), eng.audio_codes[:B].clone()))
                torch.cuda.synchronize()
                assert eng.chain_error() == 0
                assert eng.chains_ran() == (3 if on else 1), (on, eng.chains_ran())
                res[on] = (outs, [c.view(torch.uint8).clone() for c in eng.kv_caches])
        finally:
            lib.omni_debug_bb_chain(1)
    for s, (a, b) in enumerate(zip(res[1][0], res[0][0])):
        for name, x, y in zip(("logits", "hidden", "ids", "codes"), a, b):
            assert torch.equal(x, y), f"step {s}: {name} differ between the small-batch backbone chain and the launch path"
    for l, (x, y) in enumerate(zip(res[1][1], res[0][1])):
        assert torch.equal(x, y), f"KV cache of layer {l} differs"


@pytest.mark.parametrize("B", [64, 37, 32, 16, 5, 1])
def test_backbone_segment_chain_at_the_0p6b_shape_against_the_launch_path(B):
    """The 0.6B backbone (hidden 1024, intermediate 3072: the code predictor's layer dimensions) runs the per-layer segment on the code predictor's split
    of the stages (csrc/bb_chain.hip bb_flow_small_kernel) at EVERY batch size: logits, hidden state, sampled ids, codes and every KV byte of three decode
    steps are the launch path's, no wait times out, and the native step reports both chains as launched.
    Reference shape: configuration_qwen3_tts.py:192-216,376-409 (read from the checkpoint, never hard-coded: the chain is chosen
    by the shape, every other shape keeps the launch path)."""
    d = get_dims("tts-0.6b").with_(layers=3, max_model_len=256)
    w = make_weights(d, seed=8, std=0.02)
    res = {}
    with L.debug_library() as lib:
        lib.omni_debug_bb_chain.argtypes = [C.c_int]; lib.omni_debug_bb_chain.restype = None
        try:
            for on in (0, 1):
                lib.omni_debug_bb_chain(on)
                eng = _decode_engine(d, w, B, "bf16")
                outs = []
                for _ in range(3):
                    eng.decode_step(B)
                    outs.append((eng.logits[:B].clone(), eng.last_hidden[:B].clone(), eng.input_ids[:B].clone(), eng.audio_codes[:B].clone()))
                torch.cuda.synchronize()
                assert eng.chain_error() == 0
                assert eng.chains_ran() == (3 if on else 1), (on, eng.chains_ran())
                res[on] = (outs, [c.view(torch.uint8).clone() for c in eng.kv_caches])
        finally:
            lib.omni_debug_bb_chain(1)
    for s, (a, b) in enumerate(zip(res[1][0], res[0][0])):
        for name, x, y in zip(("logits", "hidden", "ids", "codes"), a, b):
            assert torch.equal(x, y), f"step {s}: {name} differ between the 0.6B backbone chain and the launch path"
    for l, (x, y) in enumerate(zip(res[1][1], res[0][1])):
        assert torch.equal(x, y), f"KV cache of layer {l} differs"


@pytest.mark.parametrize("model,shape", [("tts-0.6b", None), ("tts-1.7b", None), ("tts-1.7b", UNRELEASED)], ids=["0.6b", "1.7b", "unreleased"])
@pytest.mark.parametrize("layers", [1, 4])
def test_backbone_launches_of_changing_batches(model, shape, layers):
    """One engine, steps of batches on either side of every row split (16, 32, 48, 64) in turn: a layer's launch empties the hand-off buffers of the next
    one's, the first layer's its own, so what a batch of another size left there must not matter.  Bits of the launch path throughout."""
    d = get_dims(model).with_(layers=layers, max_model_len=256, **(shape or {}))
    w = make_weights(d, seed=9, std=0.02)
    res = {}
    with L.debug_library() as lib:
        lib.omni_debug_bb_chain.argtypes = [C.c_int]; lib.omni_debug_bb_chain.restype = None
        try:
            for on in (0, 1):
                lib.omni_debug_bb_chain(on)
                eng = _decode_engine(d, w, 64, "bf16")
                outs = []
                for B in (64, 16, 33, 1, 49, 17, 48, 32, 15, 64):
                    eng.decode_step(B)
                    outs += [eng.logits[:B].clone(), eng.last_hidden[:B].clone(), eng.audio_codes[:B].clone()]
                    assert eng.chains_ran() == (3 if on else 1), (on, B, eng.chains_ran())
                torch.cuda.synchronize()
                assert eng.chain_error() == 0
                res[on] = outs + [c.view(torch.uint8).clone() for c in eng.kv_caches]
        finally:
            lib.omni_debug_bb_chain(1)
    for i, (x, y) in enumerate(zip(res[1], res[0])):
        assert torch.equal(x, y), i


def _same(x, y):
    """equal bit for bit but for the payload of NaNs"""
    return bool(((x == y) | (x.isnan() & y.isnan())).all()) if x.is_floating_point() else torch.equal(x, y)


def _all_ones(t):
    t.view(torch.int16).fill_(-1)


@pytest.mark.parametrize("model", ["tts-1.7b", "tts-0.6b"])
@pytest.mark.parametrize("B", [5, 24, 40, 64])
def test_words_of_all_ones_pass_the_predictors_hand_offs(model, B):
    """An empty word of a hand-off buffer is two bf16 NaNs, 0xffff each (csrc/chain_flow.cuh).  Such words as data -- one row's hidden state, the projected
    row of a code that the last row draws -- are stored as other NaNs: nobody waits for them, and every output is the launch path's."""
    d = get_dims(model).with_(layers=1, max_model_len=256)
    w = make_weights(d, seed=12, std=0.02)
    code0, e0, lh = (t.cuda() for t in _inputs(d, w, B, 5 * B))
    lh = lh.clone()
    _all_ones(lh[1])
    res = {}
    with L.debug_library() as lib:
        lib.omni_debug_cp_chain.argtypes = [C.c_int]; lib.omni_debug_cp_chain.restype = None
        try:
            for on in (0, 2):
                lib.omni_debug_cp_chain(on)
                eng = _engine(d, w, kv_dtype="bf16", num_blocks=8, max_batch=64)
                clean = eng.code_predictor(code0.to(torch.int32), e0, lh, greedy=True)
                g = d.num_code_groups // 2
                _all_ones(eng.cp_proj_table[g - 1, clean[B - 1, g]])
                codes, lg = eng.code_predictor(code0.to(torch.int32), e0, lh, greedy=True, return_logits=True)
                assert eng.chain_error() == 0 and eng.chains_ran() == (1 if on else 0)
                assert lg[1].isnan().all() and lg[B - 1, g:].isnan().all() and lg[B - 1, :g].isfinite().all()
                res[on] = (clean, codes, lg)
        finally:
            lib.omni_debug_cp_chain(2)
    for x, y in zip(res[2], res[0]):
        assert _same(x, y)


@pytest.mark.parametrize("model", ["tts-1.7b", "tts-0.6b"])
@pytest.mark.parametrize("B", [5, 24, 40, 64])
def test_words_of_all_ones_pass_the_backbones_hand_offs(model, B):
    """The same words in one row's input of the backbone: a step, and the next one, in which the predictor gets that row's hidden state."""
    d = get_dims(model).with_(layers=3, max_model_len=256)
    w = make_weights(d, seed=8, std=0.02)
    res = {}
    with L.debug_library() as lib:
        for fn in (lib.omni_debug_bb_chain, lib.omni_debug_cp_chain):
            fn.argtypes = [C.c_int]; fn.restype = None
        try:
            for on in (0, 1):
                lib.omni_debug_bb_chain(on)
                lib.omni_debug_cp_chain(2 * on)
                eng = _decode_engine(d, w, B, "bf16")
                _all_ones(eng.text_step[1])
                outs = []
                for _ in range(2):
                    eng.decode_step(B)
                    assert eng.chains_ran() == (3 if on else 0), (on, eng.chains_ran())
                    assert eng.last_hidden[1].isnan().all() and eng.last_hidden[:1].isfinite().all() and eng.last_hidden[2:B].isfinite().all()
                    outs += [eng.logits[:B].clone(), eng.last_hidden[:B].clone(), eng.input_ids[:B].clone(), eng.audio_codes[:B].clone()]
                assert eng.chain_error() == 0
                res[on] = outs
        finally:
            lib.omni_debug_bb_chain(1)
            lib.omni_debug_cp_chain(2)
    for i, (x, y) in enumerate(zip(res[1], res[0])):
        assert _same(x, y), i


@pytest.mark.parametrize("B,kv,base", [(64, "fp8", "launch-path"), (49, "bf16", "layer-chain"), (57, "int8", "launch-path"), (51, "fp16", "layer-chain")])
def test_whole_backbone_launch_against_the_launch_path(B, kv, base):
    """The whole decoder stack -- qkv(0), then attention -> o_proj -> gate_up -> down_proj -> next qkv per layer -- as ONE persistent
    launch (csrc/bb_all.hip: the paged attention is a stage of the grid, two (row, kv head) pairs per workgroup) against the
    launch-per-op backbone and against the per-layer chain of the same library: pa_body.cuh / chain_gemm.cuh are the launch
    path's arithmetic, so logits, hidden state, sampled ids, codes, slot mapping and every KV byte of three decode steps are
    identical; no flag wait times out.  Reference: the vLLM Qwen3 decoder stack behind qwen3_tts_talker.py:341,414-422."""
    d = get_dims("tts-1.7b").with_(layers=3, max_model_len=256)
    w = make_weights(d, seed=8, std=0.02)
    res = {}
    with L.debug_library() as lib:
        for fn in (lib.omni_debug_bb_chain, lib.omni_debug_bb_all, lib.omni_debug_pa_tail):
            fn.argtypes = [C.c_int]; fn.restype = None
        try:
            lib.omni_debug_pa_tail(0)          # (the in-grid attention stage keeps the interleaved tail round: compare like with like)
            for on in (0, 1):
                lib.omni_debug_bb_all(on)
                lib.omni_debug_bb_chain(1 if (on or base == "layer-chain") else 0)
                eng = _decode_engine(d, w, B, kv)
                outs = []
                for _ in range(3):
                    eng.decode_step(B)
                    outs.append((eng.logits[:B].clone(), eng.last_hidden[:B].clone(), eng.input_ids[:B].clone(), eng.audio_codes[:B].clone(),
                                 eng.slot_mapping[:B].clone()))
                torch.cuda.synchronize()
                assert eng.chain_error() == 0
                res[on] = (outs, [c.view(torch.uint8).clone() for c in eng.kv_caches])
        finally:
            lib.omni_debug_bb_chain(1)
            lib.omni_debug_bb_all(0)
            lib.omni_debug_pa_tail(1)
    for s, (a, b) in enumerate(zip(res[1][0], res[0][0])):
        for name, x, y in zip(("logits", "hidden", "ids", "codes", "slots"), a, b):
            assert torch.equal(x, y), f"step {s}: {name} differ between the one-launch backbone and the {base}"
    for l, (x, y) in enumerate(zip(res[1][1], res[0][1])):
        assert torch.equal(x, y), f"KV cache of layer {l} differs"


@pytest.mark.parametrize("B,kv", [(64, "int8"), (37, "fp8"), (8, "bf16"), (1, "int8")])
def test_moe_layer_chain_against_the_launch_path(B, kv):
    """The Omni talker's sparse-MoE layer as TWO persistent launches around its
    expert GEMMs (csrc/moe_chain.hip) -- o_proj -> { router GEMM + normalised rows | shared-expert gate_up } -> { shared-expert down_proj,
    top-k routing }, and { combine into the residual stream -> the next layer's qkv } -- against the seven launches they replace (mode 2:
    the first chain alone): the launch path's tiles, k-step ownership, combine orders and the routing / combine kernels' arithmetic, so three
    decode steps at the released Omni talker width (3 layers) agree bit for bit in logits, hidden state, sampled ids, code frames and every
    KV byte; no flag wait times out; the step reports the chain as launched.  Reference: HF Qwen3OmniMoeTalkerTextSparseMoeBlock behind
    qwen3_omni.py:586-649."""
    d = get_dims("omni-talker").with_(layers=3, max_model_len=256)
    w = make_weights(d, seed=8, std=0.02)
    res = {}
    with L.debug_library() as lib:
        lib.omni_debug_moe_chain.argtypes = [C.c_int]; lib.omni_debug_moe_chain.restype = None
        try:
            for on in (0, 2, 1):
                lib.omni_debug_moe_chain(on)
                eng = _decode_engine(d, w, B, kv)
                outs = []
                for _ in range(3):
                    eng.decode_step(B)
                    outs.append((eng.logits[:B].clone(), eng.last_hidden[:B].clone(), eng.input_ids[:B].clone(), eng.audio_codes[:B].clone()))
                torch.cuda.synchronize()
                assert eng.chain_error() == 0
                assert bool(eng.chains_ran() & 2) == bool(on), (on, eng.chains_ran())
                res[on] = (outs, [c.view(torch.uint8).clone() for c in eng.kv_caches])
        finally:
            lib.omni_debug_moe_chain(1)
    for on, what in ((2, "the first MoE chain"), (1, "both MoE chains")):
        for s, (a, b) in enumerate(zip(res[on][0], res[0][0])):
            for name, x, y in zip(("logits", "hidden", "ids", "codes"), a, b):
                assert torch.equal(x, y), f"step {s}: {name} differ between {what} and the launch path"
        for l, (x, y) in enumerate(zip(res[on][1], res[0][1])):
            assert torch.equal(x, y), f"KV cache of layer {l} differs ({what})"


def test_chain_steps_replay_in_a_graph_and_stay_deterministic():
    """Whole decode steps with the chain inside a captured hipGraph: two engines fed the same requests produce the same
    codes step after step (flags and epochs advance on the device across replays), error word stays 0."""
    d = get_dims("tts-1.7b").with_(layers=2, max_model_len=256)
    w = make_weights(d, seed=4, std=0.02)
    B = 64
    outs = []
    for _ in range(2):
        eng = _engine(d, w, kv_dtype="fp8", num_blocks=256, max_batch=64)
        g = torch.Generator().manual_seed(9)
        eng.input_ids[:B] = torch.randint(1, d.codebook, (B,), generator=g).to(torch.int32).cuda()
        eng.last_hidden[:B] = torch.randn(B, d.hidden, generator=g).to(BF16).cuda()
        eng.text_step[:B] = (torch.randn(B, d.hidden, generator=g) * 0.02).to(BF16).cuda()
        eng.positions[:B] = 17
        eng.seq_lens[:B] = 18
        for b in range(B):
            eng.block_table[b, :2] = torch.tensor([1 + 2 * b, 2 + 2 * b], dtype=torch.int32)
        eng.set_sampling(greedy=0, temperature=0.9, top_k=50, rep_penalty=1.05, seed=42, cp_greedy=0, cp_temperature=0.9, cp_top_k=50)
        eng.decode_step(B); torch.cuda.synchronize()
        gr = torch.cuda.CUDAGraph()
        with torch.cuda.graph(gr):
            eng.decode_step(B)
        frames = []
        for _ in range(6):
            gr.replay()
            frames.append(eng.audio_codes[:B].clone())
        torch.cuda.synchronize()
        assert eng.chain_error() == 0
        outs.append(torch.stack(frames).cpu())
    assert torch.equal(outs[0], outs[1])
    assert (outs[0][1:] != outs[0][:-1]).any(), "steps did not advance"
