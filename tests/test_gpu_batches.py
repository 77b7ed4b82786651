"""Batches of many sequences on the GPU: the plan's limits (64 sequences, one
per lane; 256, four per lane; above, more), rows cut over
splits and rows held whole, empty sequences among them, through the finished
partial, the split step with a host partial and its merge, and the W_UV
epilogue.  Against fp64 over the same bf16 inputs.
"""
import numpy as np
import pytest
import torch

from scope_amd import ops
from tests.gpu_pool import page_layout
from tests.helpers import LSE_ATOL, LSE_RTOL, OUT_ATOL, OUT_RTOL, assert_close, bf16_randn, bits

pytestmark = pytest.mark.gpu
DEV = "cuda"
PS = 32


def _lens(B, seed, longest):
    """Mostly short lengths around block edges, every seventh sequence empty,
    a few long ones that several splits share."""
    rng = np.random.default_rng(seed)
    lens = rng.integers(1, 130, B)
    lens[::7] = 0
    lens[[1, B // 2, B - 1]] = longest, longest - 31, longest // 2
    return [int(x) for x in lens]


def _pool(lens, shape, seed):
    """A paged pool of random tokens (the reference gathers them back)."""
    table, pages = page_layout([n + 1 for n in lens], PS, seed)
    pool = bf16_randn((pages,) + shape, seed + 1, 0.5).to(DEV)
    return pool, torch.from_numpy(np.maximum(table, 0)).to(DEV)


def _attend(q, k, v, scale):
    """fp64 (out, lse) of q [.., G, Dk] over k [.., L, Dk], v [.., L, Dv]."""
    q, k, v = (x.cpu().double() for x in (q, k, v))
    x = torch.matmul(q, k.transpose(-1, -2)) * scale
    return torch.matmul(torch.softmax(x, -1), v), torch.logsumexp(x, -1)


def _merged(o, l, ho, hl):
    both = torch.logaddexp(l, hl)
    return (o * torch.exp(l - both)[..., None] + ho * torch.exp(hl - both)[..., None]), both


@pytest.mark.parametrize("B,Hkv,G,wg", [(65, 1, 4, 0), (65, 3, 2, 7), (130, 2, 8, 0),
                                        (256, 1, 1, 300), (256, 2, 4, 0), (257, 2, 4, 0),
                                        (700, 1, 2, 64)])
def test_gqa_many_sequences(B, Hkv, G, wg):
    D = 64
    lens = _lens(B, B, 3000)
    print(f"gqa B={B} Hkv={Hkv} G={G} wg={wg}", flush=True)
    kp, pt = _pool(lens, (Hkv, PS, D), 11)
    vp = bf16_randn(kp.shape, 13).to(DEV)
    q = bf16_randn((B, Hkv * G, D), 14).to(DEV)
    kn, vn = (bf16_randn((B, Hkv, 1, D), s).to(DEV) for s in (15, 16))
    gl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    lo = torch.zeros_like(gl)
    scale, max_len = D ** -0.5, max(lens) + 1

    def rows(b, n):
        t = torch.arange(n, device=DEV)
        at = pt[b, t // PS].long()
        return kp[at, :, t % PS].transpose(0, 1), vp[at, :, t % PS].transpose(0, 1)

    # the lengths as they are (empty sequences stay empty), then a fused step
    out, lse = ops.gqa_decode_partial(q, kp, vp, pt, gl, scale, max_len, n_workgroups=wg)
    for b, n in enumerate(lens):
        k, v = rows(b, n)
        if n:
            o, l = _attend(q[b].view(Hkv, G, D), k, v, scale)
        else:
            o, l = torch.zeros(Hkv, G, D), torch.full((Hkv, G), float("-inf"))
        assert_close(out[b].cpu().view(Hkv, G, D), o, OUT_ATOL, OUT_RTOL, f"partial out {b}")
        assert_close(lse[b].cpu().view(Hkv, G), l, LSE_ATOL, LSE_RTOL, f"partial lse {b}")
    ho = bf16_randn((B * Hkv * G, D), 17, 0.1).to(DEV)
    hl = torch.linspace(-2, 8, B * Hkv * G, device=DEV)
    st = ops.gqa_append_decode_split(q, kn, vn, kp, vp, pt, gl, lo, scale, max_len,
                                     n_workgroups=wg)
    mo, ml = ops.merge_split(st, (ho, hl), ops.PARTIAL_LSE_BF16, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert lo.cpu().tolist() == [n + 1 for n in lens]
    ho, hl = ho.cpu().double().view(B, Hkv, G, D), hl.cpu().double().view(B, Hkv, G)
    mo, ml = mo.cpu().view(B, Hkv, G, D), ml.cpu().view(B, Hkv, G)
    for b, n in enumerate(lens):
        k, v = rows(b, n + 1)  # with the appended token, now in its page
        assert np.array_equal(bits(k[:, n]), bits(kn[b, :, 0])), b
        assert np.array_equal(bits(v[:, n]), bits(vn[b, :, 0])), b
        o, l = _merged(*_attend(q[b].view(Hkv, G, D), k, v, scale), ho[b], hl[b])
        assert_close(mo[b], o, OUT_ATOL, OUT_RTOL, f"merged out {b}")
        assert_close(ml[b], l, LSE_ATOL, LSE_RTOL, f"merged lse {b}")


@pytest.mark.parametrize("B,H,wg", [(65, 16, 0), (200, 16, 0), (257, 16, 40), (100, 32, 0),
                                    (65, 128, 0), (96, 128, 300), (140, 128, 9), (256, 128, 0),
                                    # one pass for all heads (B * H >= 1024) and its edges
                                    (31, 32, 0), (32, 32, 0), (1024, 32, 0), (22, 48, 7),
                                    (16, 64, 0), (64, 80, 300), (11, 96, 0), (10, 112, 5)])
def test_mla_many_sequences(B, H, wg):
    lens = _lens(B, B + H, 2500)
    scale = 192 ** -0.5
    print(f"mla B={B} H={H} wg={wg}", flush=True)
    lat, pt = _pool(lens, (PS, 576), 21)
    qn = bf16_randn((B * H, 512), 22, 0.5).to(DEV)
    qp = bf16_randn((B * H, 64), 23, 0.5).to(DEV)
    new = bf16_randn((B, 1, 576), 24, 0.5).to(DEV)
    gl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    lo = torch.zeros_like(gl)
    max_len = max(lens) + 1

    def rows(b, n):
        t = torch.arange(n, device=DEV)
        return lat[pt[b, t // PS].long(), t % PS]

    q = torch.cat([qn, qp], 1).view(B, H, 576)
    out, lse = ops.mla_decode_partial(qn, qp, lat, pt, gl, scale, max_len, n_workgroups=wg)
    out, lse = out.cpu().view(B, H, 512), lse.cpu().view(B, H)
    for b, n in enumerate(lens):
        x = rows(b, n)
        if n:
            o, l = _attend(q[b], x, x[:, :512], scale)
        else:
            o, l = torch.zeros(H, 512), torch.full((H,), float("-inf"))
        assert_close(out[b], o, OUT_ATOL, OUT_RTOL, f"partial out {b}")
        assert_close(lse[b], l, LSE_ATOL, LSE_RTOL, f"partial lse {b}")
    ho = bf16_randn((B * H, 512), 25, 0.1).to(DEV)
    hl = torch.linspace(-2, 8, B * H, device=DEV)
    w_uv = bf16_randn((H, 32, 512), 26, 0.05).to(DEV)
    st = ops.mla_append_decode_split(qn, qp, new[..., :512], new[..., 512:], lat, pt, gl, lo,
                                     scale, max_len, n_workgroups=wg)
    mo, ml = ops.merge_split(st, (ho, hl), ops.PARTIAL_LSE_BF16, out_dtype=torch.float32)
    ov, latent, ul = ops.merge_split_uv(st, w_uv, (ho, hl), ops.PARTIAL_LSE_BF16,
                                        want_latent=True, want_lse=True)
    torch.cuda.synchronize()
    assert lo.cpu().tolist() == [n + 1 for n in lens]
    assert np.array_equal(bits(latent), bits(mo.to(torch.bfloat16)))
    assert torch.equal(ul, ml)
    ho, hl = ho.cpu().double().view(B, H, 512), hl.cpu().double().view(B, H)
    mo, ml, ov = mo.cpu().view(B, H, 512), ml.cpu().view(B, H), ov.float().cpu().view(B, H, 32)
    w = w_uv.cpu().double()
    for b, n in enumerate(lens):
        x = rows(b, n + 1)  # with the appended token, now in its page
        assert np.array_equal(bits(x[n]), bits(new[b, 0])), b
        o, l = _merged(*_attend(q[b], x, x[:, :512], scale), ho[b], hl[b])
        assert_close(mo[b], o, OUT_ATOL, OUT_RTOL, f"merged out {b}")
        assert_close(ml[b], l, LSE_ATOL, LSE_RTOL, f"merged lse {b}")
        assert_close(ov[b], torch.einsum("hk,hvk->hv", o, w), OUT_ATOL, OUT_RTOL, f"out_v {b}")


@pytest.mark.parametrize("B,H", [(128, 32), (64, 64), (65, 128)])
def test_mla_many_sequences_round_only_their_probabilities(B, H):
    """Batches whose rows the one-pass kernel cuts over workgroups: the pieces
    are fp32, so an output's error is that of bf16 probabilities alone.  Rounding
    to 8 significant bits errs by up to 2^-8 / m of a value of significand m, in
    rms over m log-uniform on [1, 2) by 2^-8 / sqrt(3) * sqrt(0.541) = 0.00166, and
    over random values the output errs by no more.  A bf16 piece adds as much
    again (0.0020 measured)."""
    L, scale = 2047, 192 ** -0.5
    print(f"mla precision B={B} H={H}", flush=True)
    lat, pt = _pool([L] * B, (PS, 576), 31)
    qn = bf16_randn((B * H, 512), 32, 0.5).to(DEV)
    qp = bf16_randn((B * H, 64), 33, 0.5).to(DEV)
    gl = torch.full((B,), L, dtype=torch.int32, device=DEV)
    out, _ = ops.mla_decode_partial(qn, qp, lat, pt, gl, scale, L)
    st = ops.mla_append_decode_split(qn, qp, bf16_randn((B, 1, 512), 34, 0.5).to(DEV),
                                     bf16_randn((B, 1, 64), 35, 0.5).to(DEV), lat, pt, gl,
                                     torch.zeros_like(gl), scale, L + 1)
    merged, _ = ops.merge_split(st, None, out_dtype=torch.float32)
    q = torch.cat([qn, qp], 1).view(B, H, 576)
    t = torch.arange(L + 1, device=DEV)
    for got, n in ((out, L), (merged, L + 1)):
        err = ref = 0.0
        for b in range(0, B, 8):
            x = lat[pt[b, t[:n] // PS].long(), t[:n] % PS].double()
            w = torch.softmax(torch.matmul(q[b].double(), x.t()) * scale, -1)
            o = torch.matmul(w, x[:, :512])
            err += float((got.view(B, H, 512)[b] - o).square().sum())
            ref += float(o.square().sum())
        assert (err / ref) ** 0.5 <= 0.00166, (n, (err / ref) ** 0.5)


@pytest.mark.parametrize("L,wg", [(60, 0), (3000, 12), (3000, 200)])  # whole rows, 1, 4 waves
def test_uv_merge_writes_its_lse_over_the_steps(L, wg):
    """lse_out may be the step's lse_g: both waves of a row read it before either
    result is written.  The bits of the merge with buffers of its own."""
    B, H, scale = 24, 16, 192 ** -0.5
    print(f"uv merge in place L={L} wg={wg}", flush=True)
    lat, pt = _pool([L] * B, (PS, 576), 41)
    gl = torch.full((B,), L, dtype=torch.int32, device=DEV)
    st = ops.mla_append_decode_split(bf16_randn((B * H, 512), 42, 0.5).to(DEV),
                                     bf16_randn((B * H, 64), 43, 0.5).to(DEV),
                                     bf16_randn((B, 1, 512), 44, 0.5).to(DEV),
                                     bf16_randn((B, 1, 64), 45, 0.5).to(DEV), lat, pt, gl,
                                     torch.zeros_like(gl), scale, L + 1, n_workgroups=wg)
    w_uv = bf16_randn((H, 32, 512), 46, 0.05).to(DEV)
    ho = bf16_randn((B * H, 512), 47, 0.1).to(DEV)
    hl = torch.full((B * H,), 7.0, device=DEV)
    want, _, wl = ops.merge_split_uv(st, w_uv, (ho, hl), ops.PARTIAL_LSE_BF16, want_lse=True)
    got = torch.empty_like(want)
    ws = st.workspace
    rc = ops.lib().ws_mla_merge_split_uv(
        st.gpu_len.data_ptr(), B, H, st.cap, st.nwg, st.out_g.data_ptr(), st.lse_g.data_ptr(),
        ws.data_ptr(), ws.numel(), ho.data_ptr(), hl.data_ptr(), None, ops.PARTIAL_LSE_BF16,
        w_uv.data_ptr(), 32, None, got.data_ptr(), st.lse_g.data_ptr(),
        torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0 and torch.equal(got, want) and torch.equal(st.lse_g.view(-1), wl)


@pytest.mark.parametrize("n,tokens,shape", [(1, 0, (1, 1, 1)), (3, 5, (3, 100, 1)),
                                            (256, 4097, (256, 1, 1)), (2049, 7, (2049, 1, 1)),
                                            (0, 3, (0, 4, 1))])
def test_dense_paging(n, tokens, shape):
    table, lens, ones = ops.dense_paging(n, tokens, shape, torch.device(DEV))
    assert table.shape == (n, 1) and table.view(-1).tolist() == list(range(n))
    assert lens.tolist() == [tokens] * n
    assert ones.shape == shape and bool((ones == 1).all())
