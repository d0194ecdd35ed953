"""GPU parity of the whole block step (TransformerBlock::forward on the cached
step, src/quantized_transformer.rs:258-285) through qimm_block_create /
qimm_block_forward, against the oracle on identical seeded inputs, in both
activation modes of the block (gpu_util.check_block):
- QIMM_ACT_CANDLE (the default: the reference CPU path's int8 rounding of every
  quantized-matmul input) against the oracle's candle mode: the output reaches
  cosine >= 0.9999 and max|a-b|/max|b| <= 2e-2, and its update x_out - x lies
  at least as close to candle's as the bf16 mode's does;
- QIMM_ACT_BF16 against the oracle's exact mode (f32 activations, f64
  accumulation): cosine >= 0.9999 on the output and on the stricter update,
  max|a-b|/max|b| <= 2e-2.
The own k / v the block returns are checked against the matching oracle mode.
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O
import qimm
import synth
from gpu_util import check_block, cos_sim, dev, host, kv_close, max_abs_rel, stream

pytestmark = pytest.mark.gpu


def block_tensors(w, keep):
    T = qimm.BlockTensors()
    for name, field in (("to_q", "to_q"), ("to_k", "to_k"), ("to_v", "to_v"), ("to_out", "to_out"),
                        ("gate_up", "gate_up"), ("proj", "proj"), ("gate_layer", "gate_layer"),
                        ("down", "mlp_out")):
        if name in w:
            t, data, rows, cols = w[name]
            setattr(T, field, qimm.make_tensor(t, rows, cols, data.tobytes(), keep))
    for name in ("norm_q", "norm_k"):
        arr = np.ascontiguousarray(w[name], dtype=np.float32)
        setattr(T, name, qimm.make_tensor(synth.F32, arr.size, 1, arr.tobytes(), keep))
    return T


def run_block(torch, qctx, cfg, w, x, mod, pe, kpre=None, vpre=None, alias=False, want_kv=False,
              act=qimm.ACT_CANDLE):
    keep = []
    c = qimm.BlockConfig(cfg["hidden"], cfg["heads"], cfg["head_dim"], cfg["mlp"])
    blk = qctx.block_create(c, block_tensors(w, keep))
    assert blk.act_mode == qimm.ACT_CANDLE  # the default
    blk.set_act_mode(act)
    b, s, hid = x.shape
    x_dev = dev(torch, x)
    x_out = x_dev if alias else torch.empty_like(x_dev)
    kv = None
    mod_d, pe_d = dev(torch, mod), dev(torch, pe)  # device buffers stay referenced until the step ran
    if kpre is not None:
        kv = qctx.kv_create(3, b, cfg["heads"], kpre.shape[2])
        k_d, v_d = dev(torch, kpre.view(np.int16)), dev(torch, vpre.view(np.int16))
        kv.store(2, k_d.data_ptr(), v_d.data_ptr(), stream(torch))
    k_out = v_out = None
    if want_kv:
        k_out = torch.empty((b, cfg["heads"], s, 128), dtype=torch.bfloat16, device="cuda")
        v_out = torch.empty_like(k_out)
    blk.forward(x_dev.data_ptr(), x_out.data_ptr(), b, s, mod_d.data_ptr(), pe_d.data_ptr(),
                kv, 2, k_out.data_ptr() if want_kv else None, v_out.data_ptr() if want_kv else None, stream(torch))
    out = host(x_out)
    kvs = (host(k_out.float()), host(v_out.float())) if want_kv else (None, None)
    blk.free()
    if kv is not None:
        kv.free()
    return out, kvs


def run_modes(torch, qctx, cfg, w, x, mod, pe, kpre=None, vpre=None, alias=False, want_kv=False):
    """The block in the candle and the bf16 activation mode: ((out, kv), (out, kv))."""
    return tuple(run_block(torch, qctx, cfg, w, x, mod, pe, kpre, vpre, alias, want_kv, act)
                 for act in (qimm.ACT_CANDLE, qimm.ACT_BF16))


def oracle_modes(cfg, w, x, mod, pe, kpre, vpre):
    return tuple(O.block_forward(cfg, w, x, mod, pe, kpre, vpre, mode=m) for m in (O.CANDLE, O.EXACT))


def check_modes(cfg, w, x, mod, pe, kpre, vpre, runs, want_kv=False, refs=None):
    """Both modes' outputs (and own k / v) against the oracle's matching modes."""
    (got_c, kv_c), (got_b, kv_b) = runs
    (ref, kr, vr), (ref_e, kre, vre) = refs or oracle_modes(cfg, w, x, mod, pe, kpre, vpre)
    hid = cfg["hidden"]
    check_block(*(a.reshape(-1, hid) for a in (got_c, got_b, ref, ref_e, x)))
    if want_kv:
        for (k, v), (kk, vv) in ((kv_c, (kr, vr)), (kv_b, (kre, vre))):
            kv_close(k, kk)
            kv_close(v, vv)


def make_case(seed, cfg, b, s, p, attn_type, down_type, fused=True):
    rng = np.random.default_rng(seed)
    w = synth.block_weights(seed, cfg["hidden"], cfg["heads"], cfg["mlp"], attn_type, down_type, fused)
    x = rng.standard_normal((b, s, cfg["hidden"])).astype(np.float32)
    mod = (rng.standard_normal((b, 1, 4 * cfg["hidden"])) * 0.5).astype(np.float32)
    gh = int(np.sqrt(s))
    while s % gh:
        gh -= 1
    pe = O.rope_table([(1, gh, s // gh)], [0] * p + [1] * s)[p:]
    kpre = vpre = None
    if p:
        kpre = O.f32_to_bf16(rng.standard_normal((b, cfg["heads"], p, 128)))
        vpre = O.f32_to_bf16(rng.standard_normal((b, cfg["heads"], p, 128)))
    return w, x, mod, pe, kpre, vpre


SMALL = dict(hidden=256, heads=2, head_dim=128, mlp=768)


def check(got, ref, x, exact=False):
    """exact=False: cosine on the output; exact=True: cosine on the update."""
    cs = cos_sim(got - x, ref - x) if exact else cos_sim(got, ref)
    mr = max_abs_rel(got, ref)
    assert cs >= 0.9999 and mr <= 2e-2, (cs, mr)


@pytest.mark.parametrize("attn_type,down_type", [(synth.Q8_0, synth.Q8_0), (synth.Q4_K, synth.Q6_K),
                                                 (synth.Q6_K, synth.Q4_K)])
@pytest.mark.parametrize("b,s,p", [(1, 16, 8), (2, 24, 16),  # M <= 64: split-K weight-streaming GEMM
                                   (1, 96, 40), (2, 64, 64), (1, 130, 0),
                                   # more than one tile of tokens: partial tiles, a batch
                                   # boundary inside a tile, S % 4 != 0, and sequences shorter
                                   # than a tile (three in one tile)
                                   (1, 520, 24), (2, 300, 16), (1, 514, 0), (3, 200, 8)])
def test_block_matches_oracle(torch_cuda, qctx, attn_type, down_type, b, s, p):
    w, x, mod, pe, kpre, vpre = make_case(b * 1000 + s + p, SMALL, b, s, p, attn_type, down_type)
    runs = run_modes(torch_cuda, qctx, SMALL, w, x, mod, pe, kpre, vpre, want_kv=True)
    check_modes(SMALL, w, x, mod, pe, kpre, vpre, runs, want_kv=True)


@pytest.mark.parametrize("b,s,p,act", [(1, 77, 203, "candle"), (2, 147, 33, "candle"), (2, 523, 65, "bf16"),
                                       (1, 1031, 131, "candle")])
def test_block_ragged_tokens_ignore_row_padding(torch_cuda, qctx, b, s, p, act):
    """Token counts and prefixes that are no multiple of 8 leave V^T row padding in
    the workspace. A larger call on NaN inputs fills the workspace with NaN first:
    the output is the one of a context of its own, bit for bit, and the oracle's."""
    torch = torch_cuda
    w, x, mod, pe, kpre, vpre = make_case(b + s + p, SMALL, b, s, p, synth.Q4_K, synth.Q6_K)
    mode = qimm.ACT_CANDLE if act == "candle" else qimm.ACT_BF16
    own = qimm.Context(0)
    alone, _ = run_block(torch, own, SMALL, w, x, mod, pe, kpre, vpre, act=mode)
    own.close()
    wn, xn, modn, pen, _, _ = make_case(3, SMALL, 1, 2048, 0, synth.Q4_K, synth.Q6_K)
    run_block(torch, qctx, SMALL, wn, np.full_like(xn, np.nan), modn, pen)
    got, _ = run_block(torch, qctx, SMALL, w, x, mod, pe, kpre, vpre, act=mode)
    assert np.array_equal(got, alone)
    ref, _, _ = O.block_forward(SMALL, w, x, mod, pe, kpre, vpre, mode=O.CANDLE if act == "candle" else O.EXACT)
    check(got, ref, x, exact=act == "bf16")


def test_block_in_place_and_separate_mlp_inputs(torch_cuda, qctx):
    w, x, mod, pe, kpre, vpre = make_case(7, SMALL, 1, 64, 16, synth.Q8_0, synth.Q8_0, fused=False)
    runs = run_modes(torch_cuda, qctx, SMALL, w, x, mod, pe, kpre, vpre, alias=True)
    check_modes(SMALL, w, x, mod, pe, kpre, vpre, runs)


def test_block_mixed_qkv_types_unfused_path(torch_cuda, qctx):
    """to_v in Q8_0 beside Q4_K to_q / to_k: unfused q/k/v GEMMs, and in candle
    mode the norm1 output rounded per 256 values for q and k, per 32 for v."""
    w, x, mod, pe, kpre, vpre = make_case(8, SMALL, 1, 64, 32, synth.Q4_K, synth.Q6_K)
    rng = np.random.default_rng(80)
    w["to_v"] = synth.weight(rng, synth.Q8_0, SMALL["hidden"], SMALL["hidden"])
    runs = run_modes(torch_cuda, qctx, SMALL, w, x, mod, pe, kpre, vpre, want_kv=True)
    check_modes(SMALL, w, x, mod, pe, kpre, vpre, runs, want_kv=True)


def test_block_large_norm_weights_running_max_path(torch_cuda, qctx):
    """q/k RmsNorm weights of magnitude ~3 (a score bound of ~150 in log2 units,
    above the attention's fixed-reference limit of 64): the attention keeps the
    running maximum; the small-weight cases elsewhere take the fixed reference.
    Both modes against the oracle, with a prefix cache and without."""
    for p in (32, 0):
        w, x, mod, pe, kpre, vpre = make_case(13 + p, SMALL, 1, 96, p, synth.Q4_K, synth.Q6_K)
        rng = np.random.default_rng(131 + p)
        w["norm_q"] = (3.0 + 0.3 * rng.standard_normal(128)).astype(np.float32)
        w["norm_k"] = (3.0 + 0.3 * rng.standard_normal(128)).astype(np.float32)
        runs = run_modes(torch_cuda, qctx, SMALL, w, x, mod, pe, kpre, vpre, want_kv=True)
        check_modes(SMALL, w, x, mod, pe, kpre, vpre, runs, want_kv=True)


@pytest.mark.parametrize("s,p,norm", [(700, 65, 1.0), (700, 65, 3.0), (257, 260, 3.0), (1100, 0, 1.0)])
@pytest.mark.parametrize("padded", [False, True])
def test_block_attention_split_over_keys(torch_cuda, qctx, s, p, norm, padded):
    """Few query tiles: the attention splits their keys over workgroups and merges the
    parts' sums, against the fixed reference (norm weights 1) and relative to each
    part's own maximum (3: beyond its bound), and, padded, with whole 64-key windows
    of a part masked; both activation modes against the oracle."""
    w, x, mod, pe, kpre, vpre = make_case(17 + s + p, SMALL, 1, s, p, synth.Q8_0, synth.Q8_0)
    rng = np.random.default_rng(s + p)
    for n in ("norm_q", "norm_k"):
        w[n] = (norm * (1 + 0.1 * rng.standard_normal(128))).astype(np.float32)
    if not padded:
        check_modes(SMALL, w, x, mod, pe, kpre, vpre, run_modes(torch_cuda, qctx, SMALL, w, x, mod, pe, kpre, vpre, want_kv=True),
                    want_kv=True)
        return
    torch = torch_cuda
    valid = np.ones((1, p + s), dtype=np.uint8)
    valid[0, 5:min(200, p + s // 2)] = 0
    outs = []
    for act in (qimm.ACT_CANDLE, qimm.ACT_BF16):
        keep = []
        blk = qctx.block_create(qimm.BlockConfig(256, 2, 128, 768), block_tensors(w, keep))
        blk.set_act_mode(act)
        xd, md, pd, vd = dev(torch, x), dev(torch, mod), dev(torch, pe), dev(torch, valid)
        out, kv = torch.empty_like(xd), None
        if p:
            kv = qctx.kv_create(1, 1, 2, p)
            kd, vvd = dev(torch, kpre.view(np.int16)), dev(torch, vpre.view(np.int16))
            kv.store(0, kd.data_ptr(), vvd.data_ptr(), stream(torch))
        blk.forward_masked(xd.data_ptr(), out.data_ptr(), 1, s, md.data_ptr(), 1, pd.data_ptr(), None, vd.data_ptr(), kv, 0,
                           stream=stream(torch))
        outs.append(host(out))
        blk.free()
        if kv:
            kv.free()
    mask = np.broadcast_to(valid[:, None, :], (1, s, p + s))
    refs = [O.block_forward(SMALL, w, x, mod, pe, kpre, vpre, mask=mask, mode=m)[0] for m in (O.CANDLE, O.EXACT)]
    check_block(*(a.reshape(-1, 256) for a in (outs[0], outs[1], refs[0], refs[1], x)))


def exact_softmax_error(q, k, v, see):
    """Relative error against 64 bits that bf16 probabilities relative to the running maximum
    (windows of 64 keys), f32 sums of the unrounded ones and a bf16 output have, and the 64-bit
    values; q, k, v [n, 128] f64 (scores in log2 units), see [queries, keys] bool."""
    def bf(a):
        return O.bf16_round(a.astype(np.float32)).astype(np.float64)

    s = np.where(see, q @ k.T, -np.inf)
    w = np.exp2(s - s.max(1, keepdims=True))
    want = w @ v / w.sum(1, keepdims=True)
    m, l, o = np.full(len(q), -np.inf), np.zeros(len(q)), np.zeros((len(q), 128))
    for j in range(0, len(k), 64):
        new = np.maximum(m, s[:, j:j + 64].max(1))
        ref = np.where(np.isinf(new), 0.0, new)
        a, pr = np.exp2(m - ref), np.exp2(s[:, j:j + 64] - ref[:, None])
        m, l, o = new, l * a + pr.sum(1), o * a[:, None] + bf(pr) @ v[j:j + 64]
    return bf(o / l[:, None]) - want, want


@pytest.mark.parametrize("s,p,mask", [(77, 0, None), (77, 0, "ids"), (131, 61, None), (131, 61, "valid"), (64, 77, None),
                                      (700, 65, None), (701, 64, "valid"), (1031, 0, "ids")])
def test_block_attention_precision_at_odd_lengths(torch_cuda, qctx, s, p, mask):
    """Lengths that are no multiple of 8: the block's attention rounds its probabilities
    relative to the running maximum and sums them unrounded, whatever its norms bound.
    to_out is the identity, gate1 opens fully and gate2 is shut, so that x_out - x is the
    attention's bf16 output; to_q is to_k and norm_q undoes
    the softmax scale, so that q is k. Its error
    against 64 bits is the emulated one (the fixed reference's is 1.09-1.2 times that
    here). 64 and more query tiles over few CUs split over the keys (700 tokens and more)."""
    torch = torch_cuda
    w, x, mod, pe, kpre, vpre = make_case(s + p, SMALL, 1, s, p, synth.BF16, synth.BF16)
    rng = np.random.default_rng(s)
    eye = O.f32_to_bf16(np.eye(256, dtype=np.float32))
    w["to_out"] = (synth.BF16, eye.view(np.uint8).reshape(-1), 256, 256)
    w["to_q"] = w["to_k"]
    w["norm_k"] = (0.2 * (1 + 0.1 * rng.standard_normal(128))).astype(np.float32)
    w["norm_q"] = (w["norm_k"] / np.float32(128 ** -0.5 * np.log2(np.e))).astype(np.float32)
    mod[..., 256:512], mod[..., 768:] = 30.0, 0.0
    if p:
        kpre = O.f32_to_bf16(0.2 * rng.standard_normal((1, 2, p, 128)))
    n = p + s
    ids = np.r_[np.full(s // 3, -1), np.zeros(s // 3), np.full(s - 2 * (s // 3), -1)].astype(np.int32) if mask == "ids" else None
    valid = np.ones((1, n), dtype=np.uint8)
    if mask == "valid":
        valid[0, 3:p - 2] = 0
    see = np.broadcast_to(valid[0] != 0, (s, n))
    if ids is not None:
        i, j = np.arange(s)[:, None], np.arange(s)[None, :]
        see = (i >= j) | ((ids[:, None] >= 0) & (ids[:, None] == ids[None, :]))
    keep = []
    blk = qctx.block_create(qimm.BlockConfig(256, 2, 128, 768), block_tensors(w, keep))
    blk.set_act_mode(qimm.ACT_BF16)
    xd, md, pd = dev(torch, x), dev(torch, mod), dev(torch, pe)
    idd, vd = (None if ids is None else dev(torch, ids)), dev(torch, valid)
    kd, vdv = (dev(torch, a.view(np.int16)) if p else None for a in (kpre, vpre))
    kv = qctx.kv_create(1, 1, 2, p) if p else None
    if p:
        kv.store(0, kd.data_ptr(), vdv.data_ptr(), stream(torch))
    out = torch.empty_like(xd)
    k = torch.empty((2, s, 128), dtype=torch.bfloat16, device="cuda")
    v = torch.empty_like(k)
    args = (xd.data_ptr(), out.data_ptr(), 1, s, md.data_ptr())
    tail = (k.data_ptr(), v.data_ptr(), stream(torch))
    if mask:
        blk.forward_masked(*args, 1, pd.data_ptr(), None if ids is None else idd.data_ptr(),
                           vd.data_ptr() if mask == "valid" else None, kv, 0, *tail)
    else:
        blk.forward(*args, pd.data_ptr(), kv, 0, *tail)
    got = (host(out).astype(np.float64) - x)[0]
    k, v = host(k.float()).astype(np.float64), host(v.float()).astype(np.float64)
    blk.free()
    if kv is not None:
        kv.free()
    err, emu, size = 0.0, 0.0, 0.0
    for h in range(2):
        pk, pv = ((O.bf16_to_f32(a)[0, h].astype(np.float64) for a in (kpre, vpre)) if p else (np.zeros((0, 128)),) * 2)
        e, want = exact_softmax_error(k[h], np.concatenate([pk, k[h]]), np.concatenate([pv, v[h]]), see)
        err += np.sum((got[:, 128 * h:128 * (h + 1)] - want) ** 2)
        emu += np.sum(e ** 2)
        size += np.sum(want ** 2)
    print(f"error against 64 bits {np.sqrt(err / size):.3e}, emulated {np.sqrt(emu / size):.3e}", flush=True)
    assert err <= 1.04 ** 2 * emu


def test_block_deterministic(torch_cuda, qctx):
    w, x, mod, pe, kpre, vpre = make_case(9, SMALL, 1, 96, 32, synth.Q4_K, synth.Q6_K)
    a, _ = run_block(torch_cuda, qctx, SMALL, w, x, mod, pe, kpre, vpre)
    b, _ = run_block(torch_cuda, qctx, SMALL, w, x, mod, pe, kpre, vpre)
    assert np.array_equal(a, b)


def test_block_config1_shape(torch_cuda, qctx):
    """Hidden 3072, 24 heads x 128, MLP 9216, 256 image tokens over a 64-token
    prefix, Q8_0 weights: the reference CPU-path configuration."""
    cfg = dict(hidden=3072, heads=24, head_dim=128, mlp=9216)
    w, x, mod, pe, kpre, vpre = make_case(11, cfg, 1, 256, 64, synth.Q8_0, synth.Q8_0)
    runs = run_modes(torch_cuda, qctx, cfg, w, x, mod, pe, kpre, vpre)
    check_modes(cfg, w, x, mod, pe, kpre, vpre, runs)


@pytest.mark.parametrize("b,s,p,mlp", [(1, 8, 16, 512), (2, 6, 0, 1024), (2, 8, 8, 1024), (1, 16, 0, 2048),
                                       (2, 20, 8, 1024), (1, 64, 16, 1024),
                                       # MLP 12288: gate_up (24576 x 4096) keeps six groups per CU over the
                                       # whole K (SwiGLU epilogue at 40 and at 2 x 12 tokens)
                                       (1, 40, 16, 12288), (2, 12, 8, 12288)])
def test_block_hidden4096_short_m(torch_cuda, qctx, b, s, p, mlp):
    """Hidden 4096 (32 heads) at M <= 64 tokens: the fused QKV (12288 x 4096),
    output (4096 x 4096) and gate_up (2 mlp x 4096) projections and, for
    mlp % 1024 == 0, the Q6_K down projection take the one-launch kernel with
    its q/k/v (RmsNorm + RoPE + layouts, batch boundaries inside the token
    tile), residual and SwiGLU epilogues; mlp 512 sends the down projection to
    the split-K dequantizing kernel. Short MLPs keep the oracle quick; the
    model's MLP 12288 runs at 40 and 24 tokens."""
    cfg = dict(hidden=4096, heads=32, head_dim=128, mlp=mlp)
    w, x, mod, pe, kpre, vpre = make_case(21 + b + s, cfg, b, s, p, synth.Q4_K, synth.Q6_K)
    runs = run_modes(torch_cuda, qctx, cfg, w, x, mod, pe, kpre, vpre, want_kv=True)
    check_modes(cfg, w, x, mod, pe, kpre, vpre, runs, want_kv=True)


@pytest.mark.parametrize("b,s,p,mlp,attn_type,down_type", [
    (1, 1028, 16, 1024, synth.Q4_K, synth.Q6_K),  # a 4-row last tile row
    (2, 520, 8, 1024, synth.Q4_K, synth.Q6_K),    # batch boundary inside the third 256-row tile
    (2, 523, 8, 1024, synth.Q8_0, synth.Q8_0),    # V^T rows of 523 tokens, stored 528 apart
    (1, 2100, 0, 384, synth.Q8_0, synth.Q8_0),    # down over K = 384, half a super-block over
    (1, 1024, 0, 2048, synth.Q8_0, synth.Q8_0),   # four full tile rows, no prefix
    (1, 2820, 0, 4096, synth.Q4_K, synth.Q6_K)])  # out, gate_up and down on 256 x 256 tiles too
def test_block_hidden4096_large_m(torch_cuda, qctx, qctx_codes, b, s, p, mlp, attn_type, down_type):
    """Hidden 4096 (32 heads) at M >= 1024 tokens, over bf16 rows and with the
    codes alone, where the q/k/v projection has enough 256 x 256 tiles for the
    decoding large-M kernel: the fused q/k/v epilogues over 32 heads (head =
    column / 128 across 48 column tiles, V written transposed) and the XCD-aware
    tile order, with partial tiles and a batch boundary inside a tile; at 2820
    tokens (12 tile rows) also the residual (out, Q6_K down) and SwiGLU
    epilogues, on a 4-row last tile row; at 2100 tokens the four-wave kernel's
    residual epilogue for the codes alone. Output, k and v against both oracle
    modes. Short MLPs keep the oracle quick."""
    cfg = dict(hidden=4096, heads=32, head_dim=128, mlp=mlp)
    cus, m = torch_cuda.cuda.get_device_properties(0).multi_processor_count, b * s
    assert qimm.qmatmul_route(attn_type, 12288, 4096, m, cus).kernel == qimm.GEMM_BF16_ROWS
    assert qimm.qmatmul_route(attn_type, 12288, 4096, m, cus, False).kernel == qimm.GEMM_WIDE
    if m > 2048:
        large = qimm.GEMM_WIDE if mlp % 256 == 0 else qimm.GEMM_LARGE
        assert qimm.qmatmul_route(down_type, 4096, mlp, m, cus, False).kernel == large
    w, x, mod, pe, kpre, vpre = make_case(61 + b + s, cfg, b, s, p, attn_type, down_type)
    refs = oracle_modes(cfg, w, x, mod, pe, kpre, vpre)
    for ctx in (qctx, qctx_codes):
        runs = run_modes(torch_cuda, ctx, cfg, w, x, mod, pe, kpre, vpre, want_kv=True)
        check_modes(cfg, w, x, mod, pe, kpre, vpre, runs, want_kv=True, refs=refs)


def test_block_bf16_weights_hidden256_large_m(torch_cuda, qctx):
    """Float-stored (bf16) weights, hidden 256, MLP 12288, 2112 tokens: gate_up (24576 x
    256) in the four-wave kernel with its SwiGLU epilogue, a 64-row last tile row."""
    cfg = dict(hidden=256, heads=2, head_dim=128, mlp=12288)
    cus = torch_cuda.cuda.get_device_properties(0).multi_processor_count
    assert qimm.qmatmul_route(synth.BF16, 24576, 256, 2112, cus).kernel == qimm.GEMM_LARGE
    w, x, mod, pe, kpre, vpre = make_case(71, cfg, 1, 2112, 8, synth.BF16, synth.BF16)
    got, _ = run_block(torch_cuda, qctx, cfg, w, x, mod, pe, kpre, vpre)
    ref_e, _, _ = O.block_forward(cfg, w, x, mod, pe, kpre, vpre, mode=O.EXACT)
    check(got, ref_e, x)
    check(got, ref_e, x, exact=True)


@pytest.mark.parametrize("s,mlp", [(2820, 4096), (2100, 192)])
def test_block_hidden4096_large_m_bf16_weights(torch_cuda, qctx, s, mlp):
    """Float-stored (bf16) weights, hidden 4096: the kernel over bf16 rows under
    its fused q/k/v, residual and SwiGLU epilogues (2820 tokens, MLP 4096: 12 tile
    rows, a 4-row last one), and the down projection of an MLP of 192 (an odd
    number of 64-k steps) in the four-wave kernel's bf16 form, whose weight tile
    goes global -> LDS by direct loads like the activations. Candle multiplies
    float-stored weights in plain f32 (no int8 activations), so exact mode alone
    is the reference here."""
    cfg = dict(hidden=4096, heads=32, head_dim=128, mlp=mlp)
    cus = torch_cuda.cuda.get_device_properties(0).multi_processor_count
    down = qimm.qmatmul_route(synth.BF16, 4096, mlp, s, cus).kernel
    assert down == (qimm.GEMM_BF16_ROWS if mlp % 128 == 0 else qimm.GEMM_LARGE)
    b, p = 1, 0
    w, x, mod, pe, kpre, vpre = make_case(67, cfg, b, s, p, synth.BF16, synth.BF16)
    got, (k, v) = run_block(torch_cuda, qctx, cfg, w, x, mod, pe, kpre, vpre, want_kv=True)
    ref_e, kre, vre = O.block_forward(cfg, w, x, mod, pe, kpre, vpre, mode=O.EXACT)
    check(got, ref_e, x)
    check(got, ref_e, x, exact=True)
    assert cos_sim(k, kre) >= 0.9999 and max_abs_rel(k, kre) <= 2e-2
    assert cos_sim(v, vre) >= 0.9999 and max_abs_rel(v, vre) <= 2e-2


@pytest.mark.parametrize("attn_type,down_type", [(synth.Q8_0, synth.Q8_0), (synth.Q4_K, synth.Q6_K)])
def test_block_mid_m_split_k(torch_cuda, qctx, attn_type, down_type):
    """Hidden 1024 (8 heads), MLP 2048, 128 tokens over a 16-token prefix: every
    projection's 128x128 tiles leave CUs idle, so each runs split over K (2
    shares of whole 512-value groups) with its partial sums added by the q/k/v,
    SwiGLU and residual epilogues of the reduction kernel."""
    cfg = dict(hidden=1024, heads=8, head_dim=128, mlp=2048)
    w, x, mod, pe, kpre, vpre = make_case(31, cfg, 1, 128, 16, attn_type, down_type)
    runs = run_modes(torch_cuda, qctx, cfg, w, x, mod, pe, kpre, vpre, want_kv=True)
    check_modes(cfg, w, x, mod, pe, kpre, vpre, runs, want_kv=True)
    again, _ = run_block(torch_cuda, qctx, cfg, w, x, mod, pe, kpre, vpre)
    assert np.array_equal(runs[0][0], again)


def test_block_rejects_bad_config(torch_cuda, qctx):
    keep = []
    w = synth.block_weights(1, 256, 2, 768, synth.Q8_0)
    bad = qimm.BlockConfig(256, 4, 64, 768)   # head_dim 64 unsupported
    with pytest.raises(qimm.QimmError, match="QIMM_ERR_SHAPE"):
        qctx.block_create(bad, block_tensors(w, keep))
    c = qimm.BlockConfig(256, 2, 128, 768)
    T = block_tensors(w, keep)
    T.to_q = qimm.make_tensor(synth.Q8_0, 256, 256, b"\0" * 100, keep)   # wrong byte count
    with pytest.raises(qimm.QimmError, match="QIMM_ERR_SHAPE"):
        qctx.block_create(c, T)


def test_block_reserve_then_forward(torch_cuda, qctx):
    """qimm_block_reserve pre-sizes the context scratch: forwards at the reserved
    size and below give the same bits as forwards that grow the scratch themselves,
    and bad sizes are rejected."""
    w, x, mod, pe, kpre, vpre = make_case(12, SMALL, 1, 96, 16, synth.Q4_K, synth.Q6_K)
    a, _ = run_block(torch_cuda, qctx, SMALL, w, x, mod, pe, kpre, vpre)
    keep = []
    blk = qctx.block_create(qimm.BlockConfig(256, 2, 128, 768), block_tensors(w, keep))
    blk.reserve(2, 600)
    with pytest.raises(qimm.QimmError, match="QIMM_ERR_SHAPE"):
        blk.reserve(1, 64, 3)
    with pytest.raises(qimm.QimmError, match="QIMM_ERR_ARG"):
        blk.set_act_mode(2)
    blk.free()
    b, _ = run_block(torch_cuda, qctx, SMALL, w, x, mod, pe, kpre, vpre)
    assert np.array_equal(a, b)


def test_block_reserve_covers_smaller_forwards(torch_cuda):
    """After a reserve, forwards of fewer tokens need no more scratch either, though
    they may split over K or over keys where the reserved size does not: they can be
    captured (an allocation or a synchronize would fail the capture)."""
    torch = torch_cuda
    ctx, keep = qimm.Context(0), []
    w, x, mod, pe, _, _ = make_case(21, SMALL, 1, 300, 0, synth.Q4_K, synth.Q6_K)
    blk = ctx.block_create(qimm.BlockConfig(256, 2, 128, 768), block_tensors(w, keep))
    blk.reserve(1, 4096)
    md = dev(torch, mod)
    for s in (300, 130, 77, 20):
        xd, pd = dev(torch, x[:, :s]), dev(torch, pe[:s])
        out = torch.empty_like(xd)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            blk.forward(xd.data_ptr(), out.data_ptr(), 1, s, md.data_ptr(), pd.data_ptr(), None, 0, stream=stream(torch))
        eager = torch.empty_like(xd)
        blk.forward(xd.data_ptr(), eager.data_ptr(), 1, s, md.data_ptr(), pd.data_ptr(), None, 0, stream=stream(torch))
        for _ in range(3):
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager)
    blk.free()
    ctx.close()


@pytest.mark.parametrize("case", ["config1_128x128", "wide_ragged", "two_k_shares"])
@pytest.mark.parametrize("rows_kept", [True, False])
def test_hidden_q8_0_rounding_in_gate_up_epilogue_bit_identical(torch_cuda, qctx, qctx_codes, monkeypatch, case, rows_kept):
    """Q8_0 down weights in candle mode: the Q8_0 rounding of the SwiGLU hidden
    state (the down projection's input, one scale per 32 columns of a token row)
    done by the gate_up kernel's epilogue against the same rounding as the
    rows-quantizer pass (QIMM_SEPARATE_ROUNDING=1): bit-identical block outputs.
    Cases: config 1 (MLP 9216 at 256 tokens over 64), hidden 1024 / MLP 4096 at
    1100 tokens (a last token tile of 76 rows), and the same block at 256 tokens
    (two K shares: the f32 state and the rows quantizer on both sides); over bf16
    rows, whose epilogue rounds a block across four lanes, and with the codes
    alone: the undivided 128x128 kernel (four lanes per block) and the 256x256
    kernel (two waves per block)."""
    if not rows_kept:
        qctx = qctx_codes
    if case == "config1_128x128":
        cfg, b, s, p = dict(hidden=3072, heads=24, head_dim=128, mlp=9216), 1, 256, 64
    else:
        cfg, b, s, p = dict(hidden=1024, heads=8, head_dim=128, mlp=4096), 1, 1100 if case == "wide_ragged" else 256, 64
    print(f"case: {case}, hidden {cfg['hidden']}, MLP {cfg['mlp']}, {s} tokens", flush=True)
    w, x, mod, pe, kpre, vpre = make_case(43, cfg, b, s, p, synth.Q8_0, synth.Q8_0)
    fused, _ = run_block(torch_cuda, qctx, cfg, w, x, mod, pe, kpre, vpre)
    monkeypatch.setenv("QIMM_SEPARATE_ROUNDING", "1")
    separate, _ = run_block(torch_cuda, qctx, cfg, w, x, mod, pe, kpre, vpre)
    assert np.isfinite(fused).all()
    diff = np.count_nonzero(fused.view(np.uint32) != separate.view(np.uint32))
    print(f"{case}: outputs differing in any bit: {diff} of {fused.size}", flush=True)
    assert diff == 0


@pytest.mark.parametrize("case", ["config1_fast_4wave", "ragged_any_length"])
def test_attention_q8_0_rounding_in_epilogue_bit_identical(torch_cuda, qctx, monkeypatch, case):
    """Q8_0 weights in candle mode: the attention output's Q8_0 rounding (to_out's
    input, 32 values of one head per block) done by the attention kernel's
    epilogue against the same rounding as the rows-quantizer pass
    (QIMM_SEPARATE_ROUNDING=1): bit-identical block outputs. Cases: config 1
    (hidden 3072, 24 heads, MLP 9216, 256 tokens over 64: the 4-wave fast
    kernel) and a prefix and token count that are not multiples of 8 (the
    exact form of the softmax)."""
    if case == "config1_fast_4wave":
        cfg, b, s, p = dict(hidden=3072, heads=24, head_dim=128, mlp=9216), 1, 256, 64
    else:
        cfg, b, s, p = SMALL, 2, 100, 61
    w, x, mod, pe, kpre, vpre = make_case(41, cfg, b, s, p, synth.Q8_0, synth.Q8_0)
    fused, _ = run_block(torch_cuda, qctx, cfg, w, x, mod, pe, kpre, vpre)
    monkeypatch.setenv("QIMM_SEPARATE_ROUNDING", "1")
    separate, _ = run_block(torch_cuda, qctx, cfg, w, x, mod, pe, kpre, vpre)
    assert np.isfinite(fused).all()
    diff = np.count_nonzero(fused.view(np.uint32) != separate.view(np.uint32))
    print(f"{case}: outputs differing in any bit: {diff} of {fused.size}", flush=True)
    assert diff == 0
