"""Parity at the full sizes of the benchmark's workloads, where the fp32 oracle of the whole problem would
take minutes: sampled rows against the oracle (a row of a GEMM or of an attention output only needs that
row of the left operand), and properties that hold at any size -- softmax of a constant V returns V, the
order of the key/value segments does not matter, adaLN-Zero with a zero modulation projection is the
identity, a PipeFusion patch against a K/V buffer that holds this very step's values equals the rows of
the full-sequence pass."""
import pytest
import torch

from oracle import ops as O
from tests.util import assert_parity, bf16_round

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def dev_randn(shape, seed, scale=1.0):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(shape, generator=gen, device=DEV) * scale).to(torch.bfloat16)


@pytest.fixture(autouse=True)
def fresh_state():
    from hetu_dit_amd.cache_manager import reset_cache_manager
    from hetu_dit_amd.runtime_state import reset_runtime_state

    reset_runtime_state()
    yield
    reset_cache_manager()
    reset_runtime_state()
    torch.cuda.empty_cache()


def sample_rows(m, count, seed):
    gen = torch.Generator().manual_seed(seed)
    idx = torch.randint(0, m, (count,), generator=gen)
    idx[0], idx[1] = 0, m - 1  # the corners of the first and the last tile
    return idx


# (image rows, text rows, n, k, epilogue): the four GEMM calls of an SD3 joint block at 1024 x 1024, the
# out-projection and second MLP call of a PipeFusion patch (2048 image rows: the planner gives them the
# 128x128 ring alone, with 24 and 96 slabs per tile), the QKV+MLP call of a Flux single block at 1024 x 1024, the FF1
# call of a CogVideoX block at 49 frames of 480 x 720
GEMM_CASES = [
    (8192, 666, 4608, 1536, "bias"),
    (8192, 666, 1536, 1536, "gate"),
    (8192, 666, 6144, 1536, "gelu"),
    (8192, 666, 1536, 6144, "gate"),
    (2048, 0, 1536, 1536, "gate"),
    (2048, 0, 1536, 6144, "gate"),
    (4608, 0, 9216, 3072, "bias"),
    (17776, 0, 12288, 3072, "gelu"),
]


@pytest.mark.parametrize("m_img,m_txt,n,k,epi", GEMM_CASES)
def test_gemm_full_size_sampled_rows(hdit, m_img, m_txt, n, k, epi):
    print(f"gemm full size m={m_img}+{m_txt} n={n} k={k} epi={epi}", flush=True)
    ops = hdit.ops
    probs, checks = [], []
    for i, m in enumerate([m for m in (m_img, m_txt) if m]):
        a, w, b = dev_randn((m, k), 10 + i), dev_randn((n, k), 20 + i, 0.02), dev_randn((n,), 30 + i)
        rows = sample_rows(m, 48, 40 + i)
        if epi == "gate":
            res = dev_randn((m, n), 50 + i)
            gate = torch.randn(2, n, generator=torch.Generator(device=DEV).manual_seed(60 + i), device=DEV)
            out = res.clone()
            probs.append(ops.gemm_problem(a, w, out, b, ops.EPI_GATE_RESIDUAL, resid=out, gate=gate, rows_per_batch=m // 2))
        else:
            res = gate = None
            out = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
            probs.append(ops.gemm_problem(a, w, out, b, ops.EPI_BIAS_GELU if epi == "gelu" else ops.EPI_BIAS))
        checks.append((a, w, b, res, gate, out, rows, m))
    ops.gemm_launch(probs)
    torch.cuda.synchronize()
    for a, w, b, res, gate, out, rows, m in checks:
        lin = O.linear(a[rows.to(DEV)].float().cpu(), w.float().cpu(), b.float().cpu())
        if epi == "gelu":
            want = O.gelu_tanh(lin)
        elif epi == "gate":
            g = gate.cpu()[(rows // (m // 2)).clamp(max=1)]
            want = res[rows.to(DEV)].float().cpu() + g * lin
        else:
            want = lin
        assert_parity(out[rows.to(DEV)], want, what=f"{epi} rows of m={m}")
        assert torch.isfinite(out.float()).all()


# One launch per case, a list of problems (rows, n, k, epilogue, f32 stream?, problems that share the left operand
# with the first one): the launches of the Flux and CogVideoX blocks whose tile shapes and
# two-phase plans differ from the SD3 ones -- the Flux single block's [q|k|v] + GELU(proj_mlp) call on one operand,
# its proj_out (k = 15360, gated onto the fp32 stream), the Flux double block's QKV and FF2 (k = 12288, gated fp32)
# over image + text rows, and CogVideoX's QKV / out-projection / FF2 over 226 text + 17550 video rows.
WIDE_GEMM_CASES = {
    "flux_single_qkv_mlp": [(4608, 9216, 3072, "bias", False, False), (4608, 12288, 3072, "gelu", False, True)],
    "flux_single_proj_out": [(4608, 3072, 15360, "gate", True, False)],
    "flux_double_qkv": [(4096, 9216, 3072, "bias", False, False), (512, 9216, 3072, "bias", False, False)],
    "flux_double_ff2": [(4096, 3072, 12288, "gate", True, False), (512, 3072, 12288, "gate", True, False)],
    "cogvideox_qkv": [(17776, 9216, 3072, "bias", False, False)],
    "cogvideox_out": [(226, 3072, 3072, "gate", True, False), (17550, 3072, 3072, "gate", True, False)],
    "cogvideox_ff2": [(226, 3072, 12288, "gate", True, False), (17550, 3072, 12288, "gate", True, False)],
}


@pytest.mark.parametrize("case", sorted(WIDE_GEMM_CASES))
def test_gemm_full_size_flux_cogvideox_launches(hdit, case):
    print(f"gemm full size launch {case}", flush=True)
    ops = hdit.ops
    probs, checks, first_a = [], [], None
    for i, (m, n, k, epi, f32, share) in enumerate(WIDE_GEMM_CASES[case]):
        a = first_a if share else dev_randn((m, k), 10 + i)
        first_a = a if first_a is None else first_a
        w, b = dev_randn((n, k), 20 + i, 0.02), dev_randn((n,), 30 + i)
        rows = sample_rows(m, 40, 40 + i)
        res = gate = None
        if epi == "gate":
            res = dev_randn((m, n), 50 + i)
            res = res.float() + 2.0 ** -12 if f32 else res  # an fp32 stream value that bf16 cannot hold
            gate = torch.randn(1, n, generator=torch.Generator(device=DEV).manual_seed(60 + i), device=DEV)
            out = torch.empty(m, n, dtype=res.dtype, device=DEV)
            probs.append(ops.gemm_problem(a, w, out, b, ops.EPI_GATE_RESIDUAL, resid=res, gate=gate, rows_per_batch=m))
        else:
            out = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
            probs.append(ops.gemm_problem(a, w, out, b, ops.EPI_BIAS_GELU if epi == "gelu" else ops.EPI_BIAS))
        checks.append((a, w, b, res, gate, out, rows, m, epi))
    ops.gemm_launch(probs)
    torch.cuda.synchronize()
    for a, w, b, res, gate, out, rows, m, epi in checks:
        lin = O.linear(a[rows.to(DEV)].float().cpu(), w.float().cpu(), b.float().cpu())
        if epi == "gelu":
            want = O.gelu_tanh(lin)
        elif epi == "gate":
            want = res[rows.to(DEV)].float().cpu() + gate.cpu() * lin
        else:
            want = lin
        assert_parity(out[rows.to(DEV)], want, what=f"{case}: {epi} rows of m={m}")
        assert torch.isfinite(out.float()).all()


@pytest.mark.parametrize("S,n_txt,H,hd,kind,axes", [(4608, 512, 24, 128, 1, (16, 56, 56)), (17776, 226, 48, 64, 2, (16, 24, 24))])
def test_qk_norm_rope_full_size_sampled_rows(hdit, S, n_txt, H, hd, kind, axes):
    """``hdit_qk_norm_rope`` on q and k of a packed [1, S, 3 H d] projection at the Flux (RMS norm, d 128, 4608
    rows) and CogVideoX (LayerNorm, d 64, 17776 rows) sizes: sampled rows against the oracle, text rows not rotated,
    and the v columns untouched."""
    print(f"qk_norm_rope full size S={S} H={H} d={hd} kind={kind}", flush=True)
    ops = hdit.ops
    inner = H * hd
    qkv = dev_randn((1, S, 3 * inner), 1)
    before = qkv.clone()
    wq, wk = dev_randn((hd,), 2, 0.1) + 1.0, dev_randn((hd,), 3, 0.1) + 1.0
    bq, bk = (dev_randn((hd,), 4, 0.1), dev_randn((hd,), 5, 0.1)) if kind == 2 else (None, None)
    pos = torch.stack([torch.zeros(S - n_txt), (torch.arange(S - n_txt) // 64).float(), (torch.arange(S - n_txt) % 64).float()], 1)
    cos, sin = O.flux_rope_table(pos, axes)
    q = qkv[:, :, :inner].view(1, S, H, hd)
    k = qkv[:, :, inner : 2 * inner].view(1, S, H, hd)
    jobs = [ops.qk_norm_rope_job(q, kind, wq, bq, cos.to(DEV), sin.to(DEV), rope_row0=n_txt),
            ops.qk_norm_rope_job(k, kind, wk, bk, cos.to(DEV), sin.to(DEV), rope_row0=n_txt)]
    ops.qk_norm_rope(jobs, 1, H, hd, eps=1e-6)
    torch.cuda.synchronize()
    assert torch.equal(qkv[:, :, 2 * inner :], before[:, :, 2 * inner :])
    rows = sample_rows(S, 64, 6)
    rows[2], rows[3] = n_txt - 1, n_txt  # last text row (not rotated), first rotated row
    for col0, w, b, name in ((0, wq, bq, "q"), (inner, wk, bk, "k")):
        x = before[0, rows.to(DEV), col0 : col0 + inner].float().cpu().view(-1, H, hd)
        wf = w.float().cpu()
        xn = O.rms_norm(x, 1e-6, wf) if kind == 1 else O.layer_norm(x, 1e-6, wf, b.float().cpu())
        want = xn.clone()
        for j, r in enumerate(rows.tolist()):
            if r >= n_txt:
                want[j] = O.apply_rotary_emb(xn[j][None, :, None, :], cos[r - n_txt][None], sin[r - n_txt][None])[0, :, 0]
        got = qkv[0, rows.to(DEV), col0 : col0 + inner].view(-1, H, hd)
        assert_parity(got, want, what=f"qk_norm_rope {name} rows")


def test_flux_blocks_full_size_against_oracle(hdit):
    """Flux at 1024 x 1024 -- B1, 512 text + 4096 image tokens (64 x 64 grid), D 3072, 24 heads of 128 --
    one double-stream block and one single-stream block, each against the fp32 oracle (about 1.3 TFLOP of CPU
    work apiece).  At this width the planner picks tile shapes and two-phase launches the small-width block tests
    never see."""
    import oracle
    from hetu_dit_amd import blocks, synthetic
    from hetu_dit_amd.runtime_state import get_runtime_state
    from tests.util import oracle_params

    cfg = synthetic.CONFIGS["flux_1024"]
    B, Ni, Nt, D, H, hd = cfg["batch"], cfg["n_img"], cfg["n_txt"], cfg["dim"], cfg["heads"], cfg["head_dim"]
    ids = synthetic.flux_ids(Nt, *cfg["grid"])
    cos, sin = synthetic.rope_table(ids, (16, 56, 56))
    rope = (cos.to(DEV), sin.to(DEV))
    x, e, t = synthetic.randn_bf16((B, Ni, D), 23), synthetic.randn_bf16((B, Nt, D), 24), synthetic.randn_bf16((B, D), 25)
    print("flux double block full size", flush=True)
    dbl = synthetic.init_module_(blocks.FluxTransformerBlock(D, H, hd), 21)
    p_dbl = oracle_params(dbl)
    dbl = dbl.to(DEV)
    enc, hid = dbl(hidden_states=x.to(DEV), encoder_hidden_states=e.to(DEV), temb=t.to(DEV), image_rotary_emb=rope)
    torch.cuda.synchronize()
    o_enc, o_hid = oracle.flux_double_block(p_dbl, x.float(), e.float(), t.float(), (cos, sin), H)
    assert_parity(hid, o_hid, what="flux double hidden (full size)")
    assert_parity(enc, o_enc, what="flux double encoder (full size)")
    # the same block through its one-call entry point: same launches, same bits
    enc2, hid2 = hdit.ops.block_flux_double(dbl, x.to(DEV), e.to(DEV), t.to(DEV), rope)
    torch.cuda.synchronize()
    assert torch.equal(hid2, hid) and torch.equal(enc2, enc)
    del dbl, p_dbl, o_enc, o_hid
    print("flux single block full size", flush=True)
    sgl = synthetic.init_module_(blocks.FluxSingleTransformerBlock(D, H, hd), 22)
    p_sgl = oracle_params(sgl)
    sgl = sgl.to(DEV)
    get_runtime_state().max_condition_sequence_length = Nt
    joint = torch.cat([e, x], dim=1)
    out = sgl(hidden_states=joint.to(DEV), temb=t.to(DEV), image_rotary_emb=rope)
    torch.cuda.synchronize()
    o_out = oracle.flux_single_block(p_sgl, joint.float(), t.float(), (cos, sin), H, n_text=Nt)
    assert_parity(out, o_out, what="flux single (full size)")
    out2 = hdit.ops.block_flux_single(sgl, joint.to(DEV), t.to(DEV), rope)
    torch.cuda.synchronize()
    assert torch.equal(out2, out)


# (batch, heads, image tokens, text tokens, head dim): SD3 and Flux at 1024 x 1024, CogVideoX
ATTN_CASES = [(2, 24, 4096, 333, 64), (1, 24, 4096, 512, 128), (1, 48, 17550, 226, 64)]


@pytest.mark.parametrize("B,H,n_img,n_txt,hd", ATTN_CASES)
def test_attention_full_size(hdit, B, H, n_img, n_txt, hd):
    print(f"attention full size B={B} H={H} {n_img}+{n_txt} hd={hd}", flush=True)
    ops = hdit.ops
    qi, qt = dev_randn((B, n_img, H, hd), 1), dev_randn((B, n_txt, H, hd), 2)
    ki, kt = dev_randn((B, n_img, H, hd), 3), dev_randn((B, n_txt, H, hd), 4)
    vi, vt = dev_randn((B, n_img, H, hd), 5), dev_randn((B, n_txt, H, hd), 6)
    oi, ot = ops.attention([qi, qt], [ki, kt], [vi, vt])
    torch.cuda.synchronize()
    # sampled (batch, head, query) rows against the oracle: one row needs that query and all keys/values
    S = n_img + n_txt
    q = torch.cat([qi, qt], 1)
    k = torch.cat([ki, kt], 1).float().cpu()
    v = torch.cat([vi, vt], 1).float().cpu()
    o = torch.cat([oi, ot], 1)
    rows = sample_rows(S, 24, 7)
    rows[2], rows[3] = n_img - 1, n_img  # both sides of the segment boundary
    for b, h in ((0, 0), (B - 1, H - 1)):
        want = O.attention(q[b, rows.to(DEV), h].float().cpu()[None, None], k[b, :, h][None, None], v[b, :, h][None, None])[0, 0]
        assert_parity(o[b, rows.to(DEV), h], want, what=f"attention rows b={b} h={h}")
    # the order of the key/value segments does not matter (SD3 joins [image, text], Flux [text, image])
    oi2, ot2 = ops.attention([qi, qt], [kt, ki], [vt, vi])
    torch.cuda.synchronize()
    assert_parity(oi2, oi.float(), rel=4e-3, what="segment order (image queries)")
    assert_parity(ot2, ot.float(), rel=4e-3, what="segment order (text queries)")
    # a value that is the same for every key comes back unchanged, whatever the scores
    const = dev_randn((B, 1, H, hd), 8)
    ci, ct = ops.attention([qi, qt], [ki, kt], [const.expand(B, n_img, H, hd).contiguous(), const.expand(B, n_txt, H, hd).contiguous()])
    torch.cuda.synchronize()
    assert_parity(ci, const.expand(B, n_img, H, hd).float(), rel=4e-3, what="constant V (image)")
    assert_parity(ct, const.expand(B, n_txt, H, hd).float(), rel=4e-3, what="constant V (text)")


def test_sd3_stack_full_size_properties(hdit):
    """The SD3 step and its PipeFusion form at full size (24 blocks, B2, 4096 + 333 tokens)."""
    from hetu_dit_amd import synthetic, transformer
    from hetu_dit_amd.layers.modules import AdaLayerNormContinuous, AdaLayerNormZero
    from hetu_dit_amd.runtime_state import get_runtime_state

    cfg = synthetic.CONFIGS["sd3_pipefusion"]
    B, Ni, Nt, D, L, P = cfg["batch"], cfg["n_img"], cfg["n_txt"], cfg["dim"], cfg["layers"], cfg["patches"]
    with torch.device(DEV):
        stack = transformer.SD3TransformerBlocks(L, D, cfg["heads"], cfg["head_dim"])
    gen = torch.Generator(device=DEV).manual_seed(3)
    for _, p in sorted(stack.named_parameters(), key=lambda kv: kv[0]):
        p.data = (torch.randn(p.shape, generator=gen, device=DEV) * 0.02).to(torch.bfloat16)
    x, e, t = dev_randn((B, Ni, D), 11), dev_randn((B, Nt, D), 12), dev_randn((B, D), 13)

    # a PipeFusion patch whose K/V buffer holds this very input's keys and values sees what the full pass saw:
    # its output is the matching rows of the full-sequence output
    rs = get_runtime_state()
    rs.set_token_patches([Ni // P * i for i in range(P + 1)])
    rs.set_patched_mode(False)
    full = stack(x, e, t)
    torch.cuda.synchronize()
    assert torch.isfinite(full.float()).all()
    rs.set_patched_mode(True)
    for p in range(P):
        sl = slice(Ni // P * p, Ni // P * (p + 1))
        got = stack(x[:, sl].contiguous(), e, t)
        torch.cuda.synchronize()
        assert_parity(got, full[:, sl].float(), what=f"patch {p} against the rows of the full pass")
        rs.next_patch()
    # the same step with neighbouring patches one block apart on two streams: the bits of one patch after the other
    from hetu_dit_amd.cache_manager import get_cache_manager

    buffers = [b for entry in get_cache_manager().cache.values() for b in entry.tensors if b is not None]
    saved = [b.clone() for b in buffers]
    xs = [dev_randn((B, Ni // P, D), 20 + p) for p in range(P)]
    want = []
    for p in range(P):
        want.append(stack(xs[p], e, t).clone())
        rs.next_patch()
    torch.cuda.synchronize()
    after = [b.clone() for b in buffers]
    for b, s0 in zip(buffers, saved):
        b.copy_(s0)
    got = stack.forward_patches(xs, e, t, num_streams=2)
    torch.cuda.synchronize()
    for p in range(P):
        assert torch.equal(got[p], want[p]), f"overlapped patch {p}"
    assert all(torch.equal(a, b) for a, b in zip(buffers, after))
    rs.set_patched_mode(False)

    # adaLN-Zero: with the modulation projections zeroed every gate is zero and the stack is the identity
    for m in stack.modules():
        if isinstance(m, (AdaLayerNormZero, AdaLayerNormContinuous)):
            m.linear.weight.data.zero_()
            m.linear.bias.data.zero_()
    out = stack(x, e, t)
    torch.cuda.synchronize()
    assert torch.equal(out, x)


def test_attention_fp8_full_size_cogvideox(hdit):
    """CogVideoX on the fp8 path at its real length: 48 heads, 226 text + 17550 video tokens (17776 keys).  Sampled
    query rows against the fp32 oracle at the kernel-level fp8 bound (zero-mean random V: nothing averages the
    e4m3 rounding of V and P away relative to the signal), and a V that is the same for every key and exactly
    representable in e4m3: the output must then be V itself, which holds only if the row sum is taken over the
    same rounded probabilities the P.V product consumes -- a mismatch between the two grows with the number of
    keys."""
    print("attention fp8 full size 1x48x17776 d64", flush=True)
    ops = hdit.ops
    B, H, n_txt, n_img, hd = 1, 48, 226, 17550, 64
    S = n_txt + n_img
    q, k, v = dev_randn((B, S, H, hd), 1), dev_randn((B, S, H, hd), 2), dev_randn((B, S, H, hd), 3)
    (o,) = ops.attention([q], [k], [v], fp8=True)
    torch.cuda.synchronize()
    rows = sample_rows(S, 24, 7)
    for h in (0, 17, H - 1):
        want = O.attention(q[0, rows.to(DEV), h].float().cpu()[None, None], k[0, :, h].float().cpu()[None, None],
                           v[0, :, h].float().cpu()[None, None])[0, 0]
        assert_parity(o[0, rows.to(DEV), h], want, rel=6e-2, cos=0.998, what=f"fp8 attention rows, head {h}")
    # constant, e4m3-representable V (absmax 1 maps to 448 = 1.75 * 2^8; +-1, +-0.5, +-0.25 stay exact)
    gen = torch.Generator(device=DEV).manual_seed(9)
    vals = torch.tensor([1.0, -1.0, 0.5, -0.5, 0.25, -0.25], device=DEV)
    const = vals[torch.randint(0, 6, (B, 1, H, hd), generator=gen, device=DEV)].to(torch.bfloat16)
    const[..., 0] = 1.0  # every head's absmax is 1
    (oc,) = ops.attention([q], [k], [const.expand(B, S, H, hd).contiguous()], fp8=True)
    torch.cuda.synchronize()
    err = (oc.float() - const.float()).abs().max().item()
    print(f"constant V: max |out - V| = {err:.3e}", flush=True)
    assert err <= 2.0 ** -8, f"softmax weights do not sum to one over {S} keys: max |out - V| = {err:.3e}"
