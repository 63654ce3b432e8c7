"""Routing of few tokens (experts over workgroups, one wave per token's
choice) at the edges of its tiles and of its rule, and the expert weight
gradients of small experts over chunks of 128 tokens, at the chunks' edges."""
import numpy as np
import pytest

import helpers
import oracle
from neuralscript_amd import runtime, synth

pytestmark = pytest.mark.gpu


# tokens around a wave (63-65) and the rule's lines (2048: two experts per
# workgroup, above it four; above 4096 the tiled kernel); 9 and 64 experts are
# the rule's ends, 8 and 65 lie outside; 36 and 100 columns are remainders of
# every wider load; 30 columns are refused
@pytest.mark.parametrize("M,D,E,masked", [(1, 36, 9, False), (63, 100, 10, True), (64, 64, 33, False),
                                          (65, 1024, 64, True), (2048, 36, 63, True), (2049, 36, 11, False),
                                          (4096, 36, 64, False), (4097, 36, 64, True), (65, 30, 33, True),
                                          (65, 36, 8, False), (65, 36, 65, True)])
def test_routing_of_few_tokens_is_bit_exact(M, D, E, masked):
    print(f"few-token routing M={M} D={D} E={E}", flush=True)
    H, live = 4, E // 2 if masked else E
    ir = ("ns.func @MOE {\n"
          f"  ns.tensor.alloc %moe_g_w : Tensor[{D}, {E}] float32\n"
          f"  ns.tensor.alloc %moe_e1_w : Tensor[{E}, {D * H}] float32\n"
          f"  ns.tensor.alloc %moe_e2_w : Tensor[{E}, {H * D}] float32\n"
          f"  ns.layer.moe %moe0 %x %moe_g_w %moe_e1_w %moe_e2_w : Tensor[Dynamic, {D}] float32 "
          f"// moe(x, experts={E}, ffn={H}) initial={live}\n"
          "  ns.return %moe0\n}\n")
    Wg = synth.normal(M + 1, D * E, float(1 / np.sqrt(D)))
    We1, We2 = synth.normal(M + 2, E * D * H, 0.05), synth.normal(M + 3, E * H * D, 0.05)
    x = synth.normal(M + 4, M * D)
    x[:D] = 0.0  # a token whose logits are all equal: the first live expert
    active = np.zeros(E, np.uint8)
    active[:live] = 1
    model = runtime.Model(runtime.Plan(ir), np.concatenate([Wg, We1, We2]))
    out = model.eval_infer(x)[: M * D]
    best, prob, lg = model.last_routing(M, E)
    rbest, rprob, rlg = oracle.moe_route(x, Wg, active if masked else None, M, D, E, want_logits=True)
    assert helpers.bitwise_equal(lg, rlg), "router logits differ"
    assert np.array_equal(best, rbest), f"expert choice differs at {np.flatnonzero(best != rbest)[:10]}"
    helpers.assert_close(prob, rprob, "routing probability")
    ref, _, _ = oracle.moe_fwd(x, Wg, We1, We2, active if masked else None, M, D, H, E)
    helpers.assert_close(out, ref, "moe output")
    model.free()


# one live expert takes every token: its chunks are full, one over, one short;
# 8209 tokens: the chunk has grown past 128
@pytest.mark.parametrize("rows,live", [(127, 1), (128, 1), (129, 1), (257, 1), (1025, 6), (8209, 1)])
def test_small_expert_gradients_over_token_chunks(rows, live):
    print(f"expert gradient chunks rows={rows} live={live}", flush=True)
    ir = helpers.ir_text("moet")
    assert "initial=6" in ir
    ir = ir.replace("initial=6", f"initial={live}")
    net = oracle.Net(ir)
    x, y = helpers.net_inputs(net, "moet", rows, rows), helpers.net_labels(net, rows, rows)
    w = helpers.net_weights_for(net, 900 + rows)
    om = oracle.Model(net, w)
    rec = {}
    om.train_step(x, y, 0.02, rec)
    model = runtime.Model(runtime.Plan(ir), w)
    model.train_step(x, y, 0.02)
    for ins in net.train.instrs:
        if ins.op.startswith("ns.grad.moe."):
            ref = rec["buf"][ins.result]
            helpers.assert_close(model.read_value(ins.result, ref.size), ref, f"{ins.op} rows={rows}")
    # the weights come back the same from the staged copy (the first call
    # after a step) and from the model's own (the second)
    first = model.get_weights()
    assert not helpers.bitwise_equal(first, w)
    assert helpers.bitwise_equal(first, model.get_weights())
    model.train_step(x, y, 0.02)
    again = model.get_weights()
    assert not helpers.bitwise_equal(again, first)
    assert helpers.bitwise_equal(again, model.get_weights())
    model.free()
