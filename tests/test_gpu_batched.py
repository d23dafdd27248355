"""GPU: the batched drafting path -- many requests per launch, no per-request host loop.

* the fp16 MFMA GEMM head (cfh_head_gemm16_topk, the drafter's head above 8 rows): logits within two
  fp16 ulps of the oracle plus the fp32 dot product's rounding, with the markov bias added at the GEMV
  head's rounding points; top-k ids equal where the margin exceeds 1e-3; log-sum-exp to 1e-5;
* the grouped GEMV head (cfh_head_topk_grouped, pass B of the two-pass head for a batch): bit for bit
  equal to the same kernel called once per request; the batched path residual (one
  cfh_path_residual over every request's beams, each with its own marginal hidden; above 16 rows
  the wide path streams each weight once for up to 128 rows): within fp16 rounding of the per-request
  calls and of the oracle;
* whole batched drafts -- 32 chains, 3 trees, 4 two-pass chains -- against the oracle's search on the
  same predicted hiddens, request by request (ids equal unless a decision was within 1e-3 of a tie).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import rel_err, to64
from chain_flow_amd.config import flownet
from chain_flow_amd.drafter import Drafter
from chain_flow_amd.head import PathHead, ShortlistHead
from chain_flow_amd.weights import make_weights, synthetic_context
from oracle import beam as obeam
from oracle import head as ohead


def _setup(d=512, V=4096, n=1024, seed=7):
    cfg = flownet(d, layers=1, flow_steps=2)
    W = make_weights(cfg, V, init="test", base_seed=seed)
    W["lm_head.weight"] = (W["lm_head.weight"].float() * 8).half()
    sl = torch.randperm(V, generator=torch.Generator().manual_seed(3))[:n].sort().values.to(torch.int32)
    return cfg, W, sl


def _bound(h64, w64, ref):
    ulp = np.spacing(np.abs(ref).astype(np.float16)).astype(np.float64)
    return 2 * ulp + 2.0 ** -20 * (np.abs(h64) @ np.abs(w64).T)


@pytest.mark.gpu
@pytest.mark.parametrize("M,n,d,stride", [(9, 777, 256, 1), (64, 1024, 512, 4), (65, 1000, 256, 1), (128, 300, 768, 3)])
def test_gemm16_markov_equals_two_calls(cuda, M, n, d, stride):
    """The markov bias computed inside the head's launch (up to 128 rows) against the bias as a launch of
    its own: logits, top-k and log-sum-exp bit for bit, at both row counts' edges, ragged shortlists,
    odd and even counts of head chunks and strided parents (one of them absent: -1 reads row 0)."""
    from chain_flow_amd import _lib
    g = torch.Generator().manual_seed(M + n)
    V, r = 1500, 256
    lm, w1, w2 = (torch.randn(V, x, generator=g).mul(0.1).half().to(cuda) for x in (d, r, r))
    sl = torch.randperm(V, generator=g)[:n].sort().values.to(torch.int32).to(cuda)
    head = ShortlistHead(lm, sl, w1, w2)
    h = torch.randn(M, d, generator=g).half().to(cuda)
    prev = torch.randint(0, V, (M, stride), generator=g, dtype=torch.int32).to(cuda)
    prev[M // 2, 0] = -1
    got_l, ref_l = (torch.empty(M, n, dtype=torch.float16, device=cuda) for _ in range(2))
    print(f"[gemm16 markov] M={M} n={n} d={d} stride={stride}", flush=True)
    got = head.topk(h, 4, prev=prev.view(-1), prev_stride=stride, logits=got_l)
    L, st = _lib.lib(), _lib.stream_handle()
    a = w1.index_select(0, prev[:, 0].clamp_min(0).long())
    bias = torch.empty(M, n, dtype=torch.float16, device=cuda)
    w2img = head.image.data_ptr() + int(L.cfh_head_packed_bytes(n, d, 0))
    _lib.check(L.cfh_head_gemm16_topk(a.data_ptr(), M, r, w2img, n, None, 0, bias.data_ptr(), None, None, None, None,
                                      st), "markov")
    vals, ids, lse = (torch.empty(M, 4, device=cuda), torch.empty(M, 4, dtype=torch.int32, device=cuda),
                      torch.empty(M, device=cuda))
    _lib.check(L.cfh_head_gemm16_topk(h.data_ptr(), M, d, head.image.data_ptr(), n, bias.data_ptr(), 4,
                                      ref_l.data_ptr(), vals.data_ptr(), ids.data_ptr(), lse.data_ptr(),
                                      head.workspace(M, 4, cuda).data_ptr(), st), "head")
    torch.cuda.synchronize()
    assert torch.equal(got_l, ref_l) and torch.equal(got[0], vals) and torch.equal(got[1], ids)
    assert torch.equal(got[2], lse)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [8, 128, 129, 256])
def test_out_of_range_markov_parents_read_the_nearest_row(cuda, M):
    """A parent of -1 (a beam row without one), and above 8 rows one past the table, at the row counts
    where the head's launches change (GEMV, the bias in the GEMM, the bias before it): the same
    result as the nearest row of w1, bit for bit."""
    g = torch.Generator().manual_seed(M)
    V, r, n, d = 600, 256, 500, 256
    lm, w1, w2 = (torch.randn(V, x, generator=g).mul(0.1).half().to(cuda) for x in (d, r, r))
    sl = torch.randperm(V, generator=g)[:n].sort().values.to(torch.int32).to(cuda)
    head = ShortlistHead(lm, sl, w1, w2)
    h = torch.randn(M, d, generator=g).half().to(cuda)
    prev = torch.randint(0, V, (M,), generator=g, dtype=torch.int32)
    prev[0], prev[M - 1] = -1, -1
    if M > 8:
        prev[M // 2] = V
    print(f"[markov parents] M={M}", flush=True)
    got = head.topk(h, 4, prev=prev.to(cuda))
    ref = head.topk(h, 4, prev=prev.clamp(0, V - 1).to(cuda))
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(got, ref))


@pytest.mark.gpu
@pytest.mark.parametrize("M,n,markov", [(9, 1024, True), (40, 1000, False), (160, 1024, True), (256, 777, True)])
def test_gemm16_head_matches_oracle(cuda, M, n, markov):
    cfg, W, _ = _setup(n=n)
    V = W["lm_head.weight"].shape[0]
    sl = torch.randperm(V, generator=torch.Generator().manual_seed(M))[:n].sort().values.to(torch.int32)
    head = ShortlistHead(W["lm_head.weight"].to(cuda), sl.to(cuda), W["markov.w1.weight"].to(cuda),
                         W["markov.w2.weight"].to(cuda))
    g = torch.Generator().manual_seed(M + 1)
    h = (torch.randn(M, 512, generator=g) * 0.5).half()
    prev = torch.randint(0, V, (M,), generator=g, dtype=torch.int32)
    k = 8
    logits = torch.empty(M, n, dtype=torch.float16, device=cuda)
    print(f"[gemm16] M={M} n={n} markov={markov}", flush=True)
    vals, ids, lse = head.topk(h.to(cuda), k, prev=prev.to(cuda) if markov else None, logits=logits)
    torch.cuda.synchronize()
    s64 = sl.long().numpy()
    h64, w64 = to64(h), to64(W["lm_head.weight"])[s64]
    hw = ohead.head_logits(h64, w64)
    if markov:
        mb = ohead.markov_bias(to64(W["markov.w1.weight"]), to64(W["markov.w2.weight"])[s64], prev.long().numpy())
        ref = ohead.r16(hw + mb, "fp16")
        bound = _bound(h64, w64, hw) + np.spacing(np.abs(mb).astype(np.float16)) + \
            np.spacing(np.abs(ref).astype(np.float16))
    else:
        ref = hw
        bound = _bound(h64, w64, hw)
    got = to64(logits)
    assert (np.abs(got - ref) <= bound).all()
    lsm = ohead.log_softmax(ref)
    _, want = ohead.topk(lsm, k)
    ok = ohead.margins(lsm, k) > 1e-3
    assert (ids.cpu().numpy()[ok] == want[ok]).all()
    # the kernel's own log-softmax of its own logits, exactly as the GEMV head computes it
    gl = got.astype(np.float64)
    m = gl.max(1)
    want_lse = m + np.log(np.exp(gl - m[:, None]).sum(1))
    assert np.allclose(lse.cpu().numpy(), want_lse, atol=1e-5, rtol=0)
    assert np.allclose(vals.cpu().numpy(), np.take_along_axis(gl, ids.cpu().long().numpy(), 1) - want_lse[:, None],
                       atol=1e-5, rtol=0)


@pytest.mark.gpu
def test_grouped_head_and_batched_path_match_per_request_calls(cuda):
    cfg, W, sl = _setup()
    dr = Drafter(cfg, {k: v.to(cuda) for k, v in W.items()}, sl.to(cuda), device=cuda)
    B, F, Mc, d = 5, 4, 300, 512
    g = torch.Generator().manual_seed(5)
    rows = (torch.randn(B * F, d, generator=g) * 0.5).half().to(cuda)
    cand = torch.stack([torch.randperm(4096, generator=g)[:Mc].sort().values for _ in range(B)]).to(torch.int32)
    cand = cand.to(cuda)
    lastp = torch.randint(0, 4096, (B * F, 4), generator=g, dtype=torch.int32)
    lastp[1, 2:] = -1
    lastp = lastp.to(cuda)
    print("[grouped head / batched path]", flush=True)
    v, i, l = dr.head.topk_groups(rows, 6, cand, prev=lastp.view(-1), prev_stride=4)
    pred = (torch.randn(B, 8, d, generator=g) * 0.5).half().to(cuda)
    hb = dr.path.hidden(lastp, 3, pred[:, 2])
    torch.cuda.synchronize()
    W64 = {k: to64(v_) for k, v_ in W.items() if k.startswith("path_head.")}
    emb64 = to64(W["embed_tokens.weight"])
    for b in range(B):
        rv, ri, rl = dr.head.topk_rows(rows[b * F:(b + 1) * F], 6, cand[b].contiguous(),
                                       prev=lastp[b * F:(b + 1) * F].contiguous().view(-1), prev_stride=4)
        hr = dr.path.hidden(lastp[b * F:(b + 1) * F].contiguous(), 3, pred[b, 2].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(v[b * F:(b + 1) * F], rv) and torch.equal(i[b * F:(b + 1) * F], ri), b
        assert torch.equal(l[b * F:(b + 1) * F], rl), b
        res = ohead.path_residual(W64, emb64, lastp[b * F:(b + 1) * F].long().cpu().numpy(), 3, cfg.path_order)
        ref = ohead.r16(to64(pred[b, 2])[None] + res, "fp16")
        got = to64(hb[b * F:(b + 1) * F])
        e_req, e_or = rel_err(got, to64(hr)), rel_err(got, ref)
        print(f"  request {b}: batched path vs per-request {e_req:.2e}, vs oracle {e_or:.2e}", flush=True)
        assert e_req < 2e-3 and e_or < 2e-3, b


@pytest.mark.gpu
@pytest.mark.parametrize("d,M,nlive", [(2560, 17, 1), (2560, 128, 3), (5120, 64, 2), (5120, 97, 4)])
def test_wide_path_residual_and_head_match_oracle(cuda, d, M, nlive):
    """The path residual of 17-128 rows at the served widths, one to four live offsets, absent ancestors
    mixed in, within fp16 rounding of the oracle; then the head with the markov bias over the rows it
    returned: ids equal wherever the oracle's margin exceeds twice the logits' error bound (two ulps
    and the fp32 dot product of each term, one ulp of their sum)."""
    V, n, k = 2048, 1000, 4
    cfg = flownet(d, layers=1, flow_steps=1)
    g = torch.Generator().manual_seed(d + M)
    mat = lambda r, c, s: (torch.randn(r, c, generator=g) * s).half()  # noqa: E731
    W = {f"path_head.{p}": v for p, v in [
        ("norm.weight", 1 + mat(1, d, 0.1)[0]), ("norm.bias", mat(1, d, 0.1)[0]),
        ("mlp.0.weight", mat(2 * d, d, d ** -0.5)), ("mlp.0.bias", mat(1, 2 * d, 0.05)[0]),
        ("mlp.3.weight", mat(d, 2 * d, (2 * d) ** -0.5)), ("mlp.3.bias", mat(1, d, 0.05)[0])]}
    for j in range(cfg.path_order):
        W[f"path_head.offset_proj.{j}.weight"] = mat(d, d, d ** -0.5)
        W[f"path_head.offset_proj.{j}.bias"] = mat(1, d, 0.05)[0]
    emb, lm, w1, w2 = mat(V, d, 0.5), mat(V, d, 3 * d ** -0.5), mat(V, 256, 1.0), mat(V, 256, 1 / 16)
    sl = torch.randperm(V, generator=g)[:n].sort().values.to(torch.int32)
    lastp = torch.randint(0, V, (M, cfg.path_order), generator=g, dtype=torch.int32)
    lastp[1, 1:] = -1
    lastp[M - 1, 2:] = -1
    pred = torch.randn(d, generator=g).half()
    print(f"[wide path] d={d} M={M} nlive={nlive}", flush=True)
    ph = PathHead({n_: v.to(cuda) for n_, v in W.items()}, emb.to(cuda), cfg.path_order, cfg.path_ffn_multiplier, cuda)
    head = ShortlistHead(lm.to(cuda), sl.to(cuda), w1.to(cuda), w2.to(cuda))
    lastp_d = lastp.to(cuda)
    rows = ph.hidden(lastp_d, nlive, pred.to(cuda))
    vals, ids, _ = head.topk(rows, k, prev=lastp_d.view(-1), prev_stride=cfg.path_order)
    torch.cuda.synchronize()
    res = ohead.path_residual({n_: to64(v) for n_, v in W.items()}, to64(emb), lastp.long().numpy(), nlive,
                              cfg.path_order)
    got = to64(rows)
    e = rel_err(got, ohead.r16(to64(pred)[None] + res, "fp16"))
    print(f"  hidden {e:.2e}", flush=True)
    assert e < 2e-3
    s64 = sl.long().numpy()
    lm64 = to64(lm)[s64]
    prev = lastp[:, 0].long().numpy()
    hw, mb = ohead.head_logits(got, lm64), ohead.markov_bias(to64(w1), to64(w2)[s64], prev)
    ref = ohead.r16(hw + mb, "fp16")
    bound = _bound(got, lm64, hw) + _bound(to64(w1)[prev], to64(w2)[s64], mb) + \
        np.spacing(np.abs(ref).astype(np.float16)).astype(np.float64)
    order = np.argsort(-ref, axis=-1, kind="stable")[:, :k + 1]
    near = np.take_along_axis(bound, order, -1).max(-1, keepdims=True)
    ok = ohead.margins(ref, k) > 2 * near
    print(f"  ids compared {ok.mean():.2f}", flush=True)
    assert ok.any() and (ids.cpu().numpy()[ok] == order[:, :k][ok]).all()


def _oracle(W, sl, cfg):
    W64 = {k: to64(v) for k, v in W.items()}
    s64 = sl.long().numpy()

    def score(h, prev):
        if prev is None:
            return ohead.head_logits(h, W64["lm_head.weight"][s64])
        return ohead.head_with_bias(h, W64["lm_head.weight"][s64], W64["markov.w1.weight"],
                                    W64["markov.w2.weight"][s64], prev)

    resid = lambda lp, nl: ohead.path_residual(W64, W64["embed_tokens.weight"], lp, nl, cfg.path_order)
    return s64, score, resid


def _near(trace, k1, k2):
    return any((ohead.margins(t["lp"], k1) <= 1e-3).any() or (ohead.margins(t["cand"], k2) <= 1e-3).any()
               for t in trace)


@pytest.mark.gpu
@pytest.mark.parametrize("search,B,twopass", [("chain", 32, 0), ("tree", 3, 0), ("chain", 4, 256), ("tree", 4, 256),
                                              ("chain", 8, 256), ("tree", 6, 256)])
def test_batched_drafts_match_oracle(cuda, search, B, twopass):
    cfg, W, sl = _setup()
    dr = Drafter(cfg, {k: v.to(cuda) for k, v in W.items()}, sl.to(cuda), device=cuda, twopass_m=twopass,
                 twopass_shared=True)
    ctx = synthetic_context(B, cfg.context_size, 512, seed=9)
    known0 = sl[torch.randperm(len(sl), generator=torch.Generator().manual_seed(B))[:B]].long()
    print(f"[batched {search}] B={B} twopass={twopass}", flush=True)
    pred = dr.predict_hidden(ctx.to(cuda))
    if search == "chain":
        got = dr.beam_chains(None, known0.to(cuda), 5, 4, pred=pred).cpu().numpy()
    else:
        got = dr.beam_tree(None, known0.to(cuda), keep=4, topb=8, depth=4, pred=pred).cpu().numpy()
    torch.cuda.synchronize()
    s64, score, resid = _oracle(W, sl, cfg)
    pr = to64(pred)
    bad = 0
    for b in range(B):
        if search == "chain":
            ref, tr = obeam.beam_chains(pr[b:b + 1], known0[b:b + 1].numpy(), s64, 4, 5, cfg.path_order, score,
                                        resid, return_trace=True, twopass_m=twopass, shared=True)
            k1, k2 = 4, 4
        else:
            ref, tr = obeam.beam_tree(pr[b:b + 1], known0[b:b + 1].numpy(), s64, 4, 8, 4, cfg.path_order, score,
                                      resid, return_trace=True, twopass_m=twopass, shared=True)
            k1, k2 = 8, 4
        if got[b].tolist() != ref[0].tolist():
            print(f"  b={b} gpu {got[b].tolist()} oracle {ref[0].tolist()}", flush=True)
            assert _near(tr, k1, k2), b
            bad += 1
    print(f"  {B - bad}/{B} requests equal to the oracle, the rest at near ties", flush=True)


@pytest.mark.gpu
@pytest.mark.parametrize("search,B", [("chain", 80), ("tree", 70)])
def test_batches_past_256_beam_rows_equal_smaller_batches(cuda, search, B):
    """80 width-4 chains (320 beam rows a depth) and 70 keep-4 trees (280): the path residual and
    the head take every row in one call (16-row path chunks, 256-row head launches), and each
    request's draft equals the same request drafted in a batch of half the size, bit for bit (every
    kernel computes a row from that row's inputs alone)."""
    cfg, W, sl = _setup()
    dr = Drafter(cfg, {k: v.to(cuda) for k, v in W.items()}, sl.to(cuda), device=cuda)
    ctx = synthetic_context(B, cfg.context_size, 512, seed=21).to(cuda)
    known0 = sl[torch.randperm(len(sl), generator=torch.Generator().manual_seed(B))[:B]].long().to(cuda)
    print(f"[batched {search}] B={B}: {4 * B} beam rows a depth", flush=True)
    pred = dr.predict_hidden(ctx)

    def run(lo, hi):
        if search == "chain":
            return dr.beam_chains(None, known0[lo:hi], 5, 4, pred=pred[lo:hi].contiguous())
        return dr.beam_tree(None, known0[lo:hi], keep=4, topb=8, depth=4, pred=pred[lo:hi].contiguous())

    whole = run(0, B)
    h = B // 2
    parts = torch.cat([run(0, h), run(h, B)])
    torch.cuda.synchronize()
    assert torch.equal(whole, parts)


@pytest.mark.gpu
@pytest.mark.parametrize("F,k", [(4, 4), (1, 8)])
def test_passb_over_the_shortlist_equals_grouped_rows(cuda, F, k):
    """Pass B of a large batch (B M > shortlist rows): one full-shortlist head pass, each row's
    log-softmax top-k over its request's candidates gathered from the logits, against the grouped
    in-place pass B over the same candidates: log-probs within 2e-3, ids equal away from ties."""
    cfg, W, sl = _setup()
    dr = Drafter(cfg, {k_: v.to(cuda) for k_, v in W.items()}, sl.to(cuda), device=cuda, twopass_m=256,
                 twopass_shared=True)
    B, d, M = 8, 512, 256
    g = torch.Generator().manual_seed(F)
    hm = (torch.randn(B, 4, d, generator=g)).half().to(cuda)
    local, glob = dr.head.candidates(hm, M, True)
    rows = (torch.randn(B * F, d, generator=g)).half().to(cuda)
    prev = sl[torch.randint(0, len(sl), (B * F * cfg.path_order,), generator=g)].to(torch.int32).to(cuda)
    v1, i1, _ = dr._scores(rows, k, prev, cfg.path_order, glob, B, None, None)
    v2, i2, _ = dr._scores(rows, k, prev, cfg.path_order, glob, B, None, local)
    torch.cuda.synchronize()
    v1, v2, i1, i2 = v1.cpu().numpy(), v2.cpu().numpy(), i1.cpu().numpy(), i2.cpu().numpy()
    print(f"  max |dlogp| {np.abs(v1 - v2).max():.2e}, ids equal {(i1 == i2).mean():.3f}", flush=True)
    assert np.abs(v1 - v2).max() < 2e-3
    gaps = np.diff(-v1, axis=1)
    for r in range(B * F):
        for j in range(k):
            if i1[r, j] != i2[r, j]:   # only where a neighbouring rank is within 1e-3
                near = (j > 0 and gaps[r, j - 1] <= 1e-3) or (j < k - 1 and gaps[r, j] <= 1e-3)
                assert near, (r, j)
