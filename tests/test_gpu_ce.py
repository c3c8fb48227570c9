"""GPU parity of the fused linear cross-entropy (through the C ABI).

Small shapes against the fp64 CPU oracle; the full BASELINE shape against an
fp32 torch reference computed in row chunks on the GPU.  Tolerance: relative
Frobenius error <= 2e-2 for loss, dhidden, dweight; the valid-row count and the
zero rows of ignored labels are exact.
"""

import numpy as np
import pytest
import torch

from oracle import cross_entropy as oc
from siq_vl_amd import _lib
from siq_vl_amd import cross_entropy as C
from siq_vl_amd import workloads as W

pytestmark = pytest.mark.gpu

TOL = 2e-2
DEV = "cuda"


def rel(x, ref) -> float:
    x = np.asarray(x, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    return float(np.linalg.norm(x - ref) / max(np.linalg.norm(ref), 1e-30))


def make(n, hdim, vocab, seed=0, ignore_frac=0.3, wscale=0.05):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(n, hdim, generator=g).to(torch.bfloat16)
    w = (wscale * torch.randn(vocab, hdim, generator=g)).to(torch.bfloat16)
    y = torch.randint(0, vocab, (n,), generator=g)
    y[torch.rand(n, generator=g) < ignore_frac] = -100
    return h, w, y


def run(h, w, y, chunk, divisor=None, need_dw=True):
    div = None if divisor is None else torch.tensor(float(divisor), device=DEV)
    loss, count, bad, dh, dw = C.flce_fwd_bwd(h.to(DEV), w.to(DEV), y.to(DEV), -100, div, need_dw, chunk)
    torch.cuda.synchronize()
    return (float(loss), int(count), int(bad), dh.float().cpu().numpy(),
            None if dw is None else dw.float().cpu().numpy())


@pytest.mark.parametrize("chunk", [128, 4096])
def test_small_vs_oracle(chunk):
    h, w, y = make(300, 256, 1000, seed=1)
    y[5] = 1000  # out of range: counted as bad, treated as ignored
    print(f"flce small chunk={chunk}", flush=True)
    loss, count, bad, dh, dw = run(h, w, y, chunk)
    ref = oc.linear_ce(h, w, y)
    assert count == ref["count"] and bad == ref["bad"] == 1
    assert abs(loss - ref["loss"]) <= TOL * abs(ref["loss"])
    assert rel(dh, ref["dh"]) <= TOL
    assert rel(dw, ref["dw"]) <= TOL
    ignored = (y == -100) | (y >= 1000)
    assert np.all(dh[ignored.numpy()] == 0.0)


@pytest.mark.parametrize("hdim,vocab", [(896, 2000), (320, 1000)])
def test_hidden_sizes_off_the_tile_grid(hdim, vocab):
    """hdim 896 (Qwen2.5-0.5B: three whole 256-wide tiles of the gradient
    GEMMs and a half one) and 320 (one whole tile and a quarter), with a
    vocabulary that ends inside a tile, over three chunks."""
    h, w, y = make(300, hdim, vocab, seed=31)
    print(f"flce hdim={hdim} V={vocab}", flush=True)
    loss, count, bad, dh, dw = run(h, w, y, 128)
    ref = oc.linear_ce(h, w, y)
    assert count == ref["count"] and bad == 0
    assert abs(loss - ref["loss"]) <= TOL * abs(ref["loss"])
    assert rel(dh, ref["dh"]) <= TOL and rel(dw, ref["dw"]) <= TOL
    assert np.all(dh[(y == -100).numpy()] == 0.0)


def test_sum_reduction_with_divisor():
    h, w, y = make(200, 128, 520, seed=2)
    loss, count, _, dh, dw = run(h, w, y, 64, divisor=517.0)
    ref = oc.linear_ce(h, w, y, divisor=517.0)
    assert count == ref["count"]
    assert abs(loss - ref["loss"]) <= TOL * abs(ref["loss"])
    assert rel(dh, ref["dh"]) <= TOL and rel(dw, ref["dw"]) <= TOL


def test_all_ignored_gives_nan_and_zero_grads():
    h, w, y = make(64, 64, 256, seed=3)
    y[:] = -100
    loss, count, bad, dh, dw = run(h, w, y, 4096)
    assert count == 0 and bad == 0 and np.isnan(loss)
    assert np.all(dh == 0.0) and np.all(dw == 0.0)


def test_no_ignored_rows_several_chunks():
    h, w, y = make(600, 256, 1000, seed=8, ignore_frac=0.0)
    loss, count, bad, dh, dw = run(h, w, y, 256)
    ref = oc.linear_ce(h, w, y)
    assert count == ref["count"] == 600 and bad == 0
    assert abs(loss - ref["loss"]) <= TOL * abs(ref["loss"])
    assert rel(dh, ref["dh"]) <= TOL and rel(dw, ref["dw"]) <= TOL


@pytest.mark.parametrize("chunk", [4096, 512])
def test_ignored_rows_cost_nothing_but_a_zero_row(chunk):
    """Rows whose label is ignored are compacted away before the GEMMs: the batch
    gives bitwise the loss, dW and valid-row dH of the valid rows alone."""
    g = torch.Generator().manual_seed(9)
    h = torch.randn(2048, 512, generator=g).to(torch.bfloat16)
    w = (0.05 * torch.randn(4096, 512, generator=g)).to(torch.bfloat16)
    y = W.span_masked_labels(2048, 4096, 0.3, g)
    valid = (y != -100).numpy()
    print(f"flce compaction chunk={chunk} valid={int(valid.sum())}", flush=True)
    full = run(h, w, y, chunk)
    sub = run(h[valid], w, y[valid], chunk)
    assert full[1] == sub[1] == int(valid.sum())
    assert full[0] == sub[0]
    assert np.array_equal(full[3][valid], sub[3]) and np.all(full[3][~valid] == 0.0)
    if chunk >= 2048:  # one chunk either way: the same rows in the same k-steps
        assert np.array_equal(full[4], sub[4])
    else:
        assert rel(full[4], sub[4]) <= 1e-2


def test_qwen_vocab_vs_oracle():
    h, w, y = make(256, 1536, W.QWEN_VOCAB, seed=4, wscale=0.02)
    print("flce qwen vocab n=256", flush=True)
    loss, count, _, dh, dw = run(h, w, y, 4096)
    ref = oc.linear_ce(h, w, y, block=64)
    assert count == ref["count"]
    assert abs(loss - ref["loss"]) <= TOL * abs(ref["loss"])
    assert rel(dh, ref["dh"]) <= TOL and rel(dw, ref["dw"]) <= TOL


def test_vocab_past_one_factor_segment_vs_oracle():
    """V = 270000: 1055 vocab tiles, of which the last holds 176 columns, with
    labels in it and on both sides of its 1024th tile's end.  Two chunks, so dW
    is also summed over chunks."""
    h, w, y = make(96, 64, 270000, seed=9, wscale=0.05)
    y[7] = 269999  # the last column of the partial last tile
    y[8] = 262143  # the last column of tile 1023
    y[9] = 262144  # the first column of tile 1024
    print("flce vocab 270000 n=96 chunk=64", flush=True)
    loss, count, _, dh, dw = run(h, w, y, 64)
    ref = oc.linear_ce(h, w, y, block=32)
    assert count == ref["count"]
    assert abs(loss - ref["loss"]) <= TOL * abs(ref["loss"])
    assert rel(dh, ref["dh"]) <= TOL and rel(dw, ref["dw"]) <= TOL
    # the labelled columns' dW rows are dominated by the -g term: check them alone too
    for v in (269999, 262143, 262144):
        assert rel(dw[v], ref["dw"][v]) <= TOL, v


def test_large_logits_keep_relative_precision():
    # logits of magnitude ~30: the exp-normalised chunk buffer keeps precision
    h, w, y = make(128, 256, 2048, seed=6, wscale=2.0)
    loss, _, _, dh, dw = run(h, w, y, 4096)
    ref = oc.linear_ce(h, w, y)
    assert abs(loss - ref["loss"]) <= TOL * abs(ref["loss"])
    assert rel(dh, ref["dh"]) <= TOL and rel(dw, ref["dw"]) <= TOL


@pytest.mark.parametrize("n,hdim,vocab,chunk", [(300, 256, 1000, 128), (300, 256, 1000, 4096),
                                                (256, 1536, W.QWEN_VOCAB, 4096)])
def test_dh_only_vs_oracle(n, hdim, vocab, chunk):
    """The call of a frozen lm_head (dweight = NULL: the reference's stage 1,
    siq_vl/model/modeling.py:329-330, and stage 2's LoRA, which leaves lm_head
    out of its targets, :377-386): loss and dH against the oracle, ignored
    rows exactly zero, and bitwise the loss and dH of the call that also
    forms dW."""
    h, w, y = make(n, hdim, vocab, seed=21, wscale=0.05 if vocab < 4096 else 0.02)
    y[5] = vocab + 1  # out of range: counted as bad, treated as ignored
    print(f"flce dH only n={n} V={vocab} chunk={chunk}", flush=True)
    loss, count, bad, dh, dw = run(h, w, y, chunk, need_dw=False)
    assert dw is None
    ref = oc.linear_ce(h, w, y, block=64)
    assert count == ref["count"] and bad == ref["bad"] == 1
    assert abs(loss - ref["loss"]) <= TOL * abs(ref["loss"])
    assert rel(dh, ref["dh"]) <= TOL
    ignored = ((y == -100) | (y >= vocab)).numpy()
    assert np.all(dh[ignored] == 0.0)
    both = run(h, w, y, chunk, need_dw=True)
    assert both[0] == loss and np.array_equal(both[3], dh)


def test_frozen_lm_head_autograd_takes_the_dh_only_call():
    """hidden requires grad, the weight does not: the autograd op forms no dW
    and hidden's gradient is the raw dH-only call's, scaled."""
    h, w, y = make(200, 128, 768, seed=22)
    hg = h.to(DEV).requires_grad_(True)
    wd = w.to(DEV)
    loss = C.fused_linear_cross_entropy(hg, wd, y.to(DEV), chunk_tokens=64)
    (2.0 * loss).backward()
    assert wd.grad is None
    _, _, _, dh, dw = run(h, w, y, 64, need_dw=False)
    assert dw is None
    assert np.array_equal(hg.grad.float().cpu().numpy(), (torch.from_numpy(dh) * 2.0).to(torch.bfloat16).float().numpy())


def test_autograd_matches_raw_and_scales():
    h, w, y = make(96, 128, 512, seed=8)
    hg = h.to(DEV).requires_grad_(True)
    wg = w.to(DEV).requires_grad_(True)
    loss = C.fused_linear_cross_entropy(hg, wg, y.to(DEV), chunk_tokens=64)
    (3.0 * loss).backward()
    _, _, _, dh, dw = run(h, w, y, 64)
    assert np.allclose(hg.grad.float().cpu().numpy(), 3.0 * dh, rtol=1e-2, atol=1e-6)
    assert np.allclose(wg.grad.float().cpu().numpy(), 3.0 * dw, rtol=1e-2, atol=1e-6)


@pytest.mark.slow
def test_full_size_vs_torch_fp32():
    """Config 4 at full size, both the training call (dH and dW) and the
    frozen-lm_head call (dH only), against one fp32 torch reference."""
    cfg = W.CONFIG4
    print(f"flce full size n={cfg.n} hdim={cfg.hdim} V={cfg.vocab}", flush=True)
    x = W.ce_inputs(cfg, device=DEV)
    loss, count, bad, dh, dw = C.flce_fwd_bwd(x["hidden"], x["weight"], x["labels"])
    loss_h, count_h, bad_h, dh_h, dw_h = C.flce_fwd_bwd(x["hidden"], x["weight"], x["labels"], need_dweight=False)
    assert dw_h is None and int(count_h) == int(count) and int(bad_h) == int(bad)
    assert float(loss_h) == float(loss) and torch.equal(dh_h, dh)
    del dh_h
    hf = x["hidden"].float()
    wf = x["weight"].float()
    y = x["labels"]
    valid = y != -100
    cnt = int(valid.sum())
    assert int(count) == cnt and int(bad) == 0
    ref_loss = torch.zeros((), device=DEV, dtype=torch.float64)
    ref_dh = torch.empty_like(hf)
    ref_dw = torch.zeros_like(wf)
    for r0 in range(0, cfg.n, 2048):
        z = hf[r0:r0 + 2048] @ wf.t()
        yb = y[r0:r0 + 2048]
        ref_loss += torch.nn.functional.cross_entropy(z, yb, ignore_index=-100, reduction="sum").double()
        p = torch.softmax(z, -1)
        vb = yb != -100
        idx = torch.nonzero(vb).reshape(-1)
        p[idx, yb[idx]] -= 1.0
        p[~vb] = 0.0
        p /= cnt
        ref_dh[r0:r0 + 2048] = p @ wf
        ref_dw += p.t() @ hf[r0:r0 + 2048]
        del z, p
    ref_loss = float(ref_loss / cnt)
    r_loss = abs(float(loss) - ref_loss) / abs(ref_loss)
    r_dh = float((dh.float() - ref_dh).norm() / ref_dh.norm())
    r_dw = float((dw.float() - ref_dw).norm() / ref_dw.norm())
    print(f"  loss {float(loss):.6f} ref {ref_loss:.6f} rel {r_loss:.2e}; dh rel {r_dh:.2e}; dw rel {r_dw:.2e}",
          flush=True)
    assert r_loss <= TOL and r_dh <= TOL and r_dw <= TOL
    assert bool((dh[~valid] == 0).all())


@pytest.mark.parametrize("n,hdim,vocab,chunk", [(70, 64, 1032, 4096), (4500, 128, 1032, 4096), (700, 192, 520, 300),
                                                (200, 64, 20008, 4096)])
def test_row_references_and_label_terms(n, hdim, vocab, chunk):
    """Rows whose label logit is near the maximum, 2^60 below it in every tile
    or in some (their tiles are redone relative to their own maximum), labels
    that come once, often, in several sorted runs of 2048 rows, and rows whose
    label holds all the mass.  Per element: dH one rounding of each softmax
    numerator (a second one in redone rows) and of the result, dW one of f H
    besides; the label terms are exact."""
    print(f"flce references n={n} hdim={hdim} V={vocab} chunk={chunk}", flush=True)
    h, w, y = make(n, hdim, vocab, seed=n, ignore_frac=0.2, wscale=1.0)
    g = torch.Generator().manual_seed(n + 1)
    valid = torch.nonzero((y >= 0)).flatten()
    y[valid[torch.rand(valid.numel(), generator=g) < 0.4]] = 7  # a frequent label
    scale = torch.tensor([0.01, 0.2, 3.0, 12.0])[torch.randint(0, 4, (n,), generator=g)]
    h = (h.float() * scale[:, None]).to(torch.bfloat16)
    for r in valid[::5].tolist():  # the label far above the rest
        h[r] = w[y[r]] * 2.0
    for r in valid[1::7].tolist():  # one vocab tile far above the label's, the others not
        h[r] = (0.02 * h[r].float() + 3.0 * w[300 + r % 100].float()).to(torch.bfloat16)
    loss, count, bad, dh, dw = run(h, w, y, chunk)
    ref = oc.linear_ce(h, w, y)
    assert count == ref["count"] and bad == 0
    assert abs(loss - ref["loss"]) <= 1e-5 * abs(ref["loss"])
    hf, wf = h.double().numpy()[valid], w.double().numpy()
    z = hf @ wf.T
    p = np.exp(z - z.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True) * count
    # fp32 logits: p's relative error is the logit's absolute one
    slack = 2.0**-8 + hdim * 2.0**-22 * float((np.abs(hf) @ np.abs(wf).T).max())
    mag_h, mag_w = p @ np.abs(wf), p.T @ np.abs(hf)
    assert np.all(np.abs(dh[valid] - ref["dh"][valid]) <= 2**-8 * np.abs(ref["dh"][valid]) + slack * mag_h + 1e-30)
    steps = -(-count // chunk)
    assert np.all(np.abs(dw - ref["dw"]) <= (2**-8 if steps == 1 else 2**-7) * np.abs(ref["dw"]) + 2 * slack * mag_w
                  + (0 if steps == 1 else 2**-8 * 2 * np.abs(mag_w).max()) + 1e-30)
    alone, c2, _ = C.flce_loss(h.to(DEV), w.to(DEV), y.to(DEV))
    assert float(alone) == loss and int(c2) == count


@pytest.mark.parametrize("n,hdim,vocab", [(300, 64, 8), (2100, 1024, 712), (1800, 1280, 5000), (20000, 1024, 520),
                                          (32600, 4096, 264)])
def test_dh_ranges_and_parts(n, hdim, vocab):
    """dH's vocab ranges: fewer k-steps than ranges and parts, token tiles with
    whole ranges and with cut ones in one call, a valid-row count well below
    the chunk, 7 ranges, and 1.  Per element: one rounding of each softmax
    numerator, one of the result, and the fp32 logit's error."""
    print(f"flce dH ranges n={n} hdim={hdim} V={vocab}", flush=True)
    h, w, y = make(n, hdim, vocab, seed=n, ignore_frac=0.6 if n == 1800 else 0.05, wscale=2.0 / hdim**0.5)
    hd, wd, yd = h.to(DEV), w.to(DEV), y.to(DEV)
    loss, count, bad, dh, _ = C.flce_fwd_bwd(hd, wd, yd, -100, None, False, n)
    wf, total = wd.double(), 0.0
    valid = yd >= 0
    assert int(count) == int(valid.sum()) and int(bad) == 0
    assert bool((dh[~valid] == 0).all())
    for r0 in range(0, n, 4096):
        hb, yb, vb = hd[r0:r0 + 4096].double(), yd[r0:r0 + 4096], valid[r0:r0 + 4096]
        z = hb @ wf.t()
        rows = torch.arange(hb.shape[0], device=DEV)
        zy = z[rows, yb.clamp(min=0)]
        total += float((torch.logsumexp(z, 1) - zy)[vb].sum())
        p = torch.softmax(z, 1) / int(count)
        slack = 2.0**-8 + hdim * 2.0**-22 * float((hb.abs() @ wf.abs().t()).max())
        mag = p @ wf.abs()
        ref = p @ wf - wf[yb.clamp(min=0)] / int(count)
        err = (dh[r0:r0 + 4096].double() - ref).abs()
        assert bool((err <= 2.0**-8 * ref.abs() + slack * mag + 1e-30)[vb].all())
    assert abs(float(loss) - total / int(count)) <= 1e-5 * abs(total / int(count))


@pytest.mark.parametrize("n,chunk,valid", [(300, 100, 250), (600, 300, 505), (700, 300, 500), (2000, 1000, 96),
                                           (700, 300, 600), (512, 512, 512), (90, 1, 70)])
def test_dw_reads_no_row_that_the_call_did_not_write(n, chunk, valid):
    """Chunks that start off the 64-row grid: dW's last k-step reaches past the
    valid rows, there to zero rows only, whatever the workspace held before
    (large finite values here)."""
    hdim, vocab = 128, 520
    h, w, y = make(n, hdim, vocab, seed=valid, ignore_frac=0.0)
    g = torch.Generator().manual_seed(n)
    y[torch.randperm(n, generator=g)[valid:]] = -100
    print(f"flce workspace contents n={n} chunk={chunk} valid={valid}", flush=True)
    L = _lib.lib()
    hd, wd, yd = h.to(DEV), w.to(DEV), y.to(DEV)
    dh, dw = torch.empty_like(hd), torch.empty_like(wd)
    loss, count, bad = (torch.empty((), dtype=t, device=DEV) for t in (torch.float32, torch.int64, torch.int64))
    nbytes = L.siq_flce_workspace_bytes(n, hdim, vocab, chunk, 1)
    ws = torch.full((nbytes // 2,), 3.0, dtype=torch.bfloat16, device=DEV)
    rc = L.siq_flce_fwd_bwd(hd.data_ptr(), wd.data_ptr(), yd.data_ptr(), n, hdim, vocab, -100, 0, None,
                            loss.data_ptr(), count.data_ptr(), bad.data_ptr(), dh.data_ptr(), dw.data_ptr(), chunk,
                            ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "siq_flce_fwd_bwd")
    ref = oc.linear_ce(h, w, y)
    assert int(count) == ref["count"] == valid
    assert abs(float(loss) - ref["loss"]) <= 1e-5 * abs(ref["loss"])
    # bf16 operands, a few roundings each; over two chunks the first one's sum is rounded besides
    assert rel(dh.float().cpu().numpy(), ref["dh"]) <= 2.0**-7
    assert rel(dw.float().cpu().numpy(), ref["dw"]) <= 2.0**-7


@pytest.mark.parametrize("n,hdim,vocab,chunks", [(8192, 1536, 151936, (None, 8192, 4096, 1000)),
                                                 (3000, 896, 1032, (None, 1500, 1024, 700, 100))])
def test_loss_and_dh_do_not_depend_on_the_chunk(n, hdim, vocab, chunks):
    """Bitwise: the cut of dH's vocab ranges goes by the batch's token tiles,
    also in chunks that start inside one or hold more than one run of them
    (151936 columns: runs of 27 tiles; all chunks have 8 ranges)."""
    g = torch.Generator(device=DEV).manual_seed(hdim)
    h = torch.randn(n, hdim, device=DEV, generator=g).to(torch.bfloat16)
    w = (0.05 * torch.randn(vocab, hdim, device=DEV, generator=g)).to(torch.bfloat16)
    y = torch.randint(0, vocab, (n,), device=DEV, generator=g)
    y[torch.rand(n, device=DEV, generator=g) < 0.1] = -100
    want = None
    for chunk in chunks:
        print(f"flce chunk n={n} hdim={hdim} V={vocab} chunk={chunk}", flush=True)
        loss, _, _, dh, _ = C.flce_fwd_bwd(h, w, y, -100, None, False, chunk)
        want = want or (loss, dh)
        assert torch.equal(loss, want[0])
        assert torch.equal(dh.view(torch.int16), want[1].view(torch.int16))


@pytest.mark.parametrize("n,vocab,peaked", [(1024, 32008, False), (1024, 32008, True), (1600, 32008, True),
                                            (2100, 151936, False), (2100, 151936, True)])
def test_redone_rows_are_rounded_no_more_often_than_others(n, vocab, peaked):
    """Labels far below their rows' other logits, so that tiles are redone.
    Rows of dW without a label (no exact label term) see a rounding of E, one on
    the way to the gradient and one of the result, each 2^-9.2 in the root mean
    square of a relative error; where one logit holds a row's mass, its E is 1
    and the first rounding falls away.  With 151936 columns a workgroup of the
    row pass brings more tiles to the rows' reference than it keeps factors of."""
    hdim = 896
    g = torch.Generator(device=DEV).manual_seed(5)
    h = torch.randn(n, hdim, device=DEV, generator=g).to(torch.bfloat16)
    w = (0.02 * torch.randn(vocab, hdim, device=DEV, generator=g)).to(torch.bfloat16)
    y = torch.arange(n, device=DEV)
    if peaked:
        h *= 40
    else:
        w[:n] = (-0.05 * h.float()).to(torch.bfloat16)
    print(f"flce redone rows n={n} hdim={hdim} V={vocab} peaked={peaked}", flush=True)
    z = h.double() @ w.double().t()
    low = float((z.max(1).values - z[y, y] > 60 * 0.6931).double().mean())
    print(f"  redone rows {low:.3f}", flush=True)
    assert low > 0.95
    _, _, _, dh, dw = C.flce_fwd_bwd(h, w, y, -100, None, True)
    p = torch.softmax(z, 1)
    p[y, y] -= 1.0
    p /= n
    for got, ref in ((dh, p @ w.double()), (dw[n:], p[:, n:].t() @ h.double())):
        err = float((got.double() - ref).norm() / ref.norm())
        print(f"  rel {err:.3e}", flush=True)
        assert err <= (2 if peaked else 3) ** 0.5 * 2.0**-9.2


@pytest.mark.parametrize("n,hdim,counts", [(1500, 64, (255, 256, 257, 512, 1)), (6000, 832, (5000, 600)),
                                           (2048, 1600, (2048,)), (140000, 64, ())])
def test_label_terms_of_frequent_labels(n, hdim, counts):
    """dW's label terms: labels with a sum's 256 rows and a few more or less,
    labels that hold nearly all rows over three sorted runs, and labels spread
    over more runs than a wave searches at once (69).  Where the softmax part is
    small (p = 1 / 8192) a missing row shows: the error is that of bf16 operands."""
    vocab = 8192 if n < 100000 else 520
    g = torch.Generator(device=DEV).manual_seed(n)
    h = torch.randn(n, hdim, device=DEV, generator=g).to(torch.bfloat16)
    w = (0.2 / hdim**0.5 * torch.randn(vocab, hdim, device=DEV, generator=g)).to(torch.bfloat16)
    y = torch.randint(0, vocab, (n,), device=DEV, generator=g)
    order, at = torch.randperm(n, device=DEV, generator=g), 0
    for i, c in enumerate(counts):
        y[y == 9 + i] = 0
        y[order[at:at + c]] = 9 + i
        at += c
    print(f"flce frequent labels n={n} hdim={hdim}", flush=True)
    _, count, bad, _, dw = C.flce_fwd_bwd(h, w, y, -100, None, True)
    assert int(count) == n and int(bad) == 0
    ref = torch.zeros(vocab, hdim, dtype=torch.float64, device=DEV)
    for r0 in range(0, n, 4096):
        hb = h[r0:r0 + 4096].double()
        p = torch.softmax(hb @ w.double().t(), 1)
        p[torch.arange(hb.shape[0], device=DEV), y[r0:r0 + 4096]] -= 1.0
        ref += (p / n).t() @ hb
    err = (dw.double() - ref).norm(dim=1) / ref.norm(dim=1)
    print(f"  largest relative error of a row {float(err.max()):.2e}", flush=True)
    assert float(err.max()) <= 2.0**-6  # (sums that nearly cancel: bf16 errors of the terms over the result)
    again = C.flce_fwd_bwd(h, w, y, -100, None, True)[4]
    assert torch.equal(dw.view(torch.int16), again.view(torch.int16))


@pytest.mark.parametrize("n,chunk", [(700, 4096), (700, 256)])
def test_dhidden_in_the_place_of_hidden(n, chunk):
    """The C ABI with dhidden == hidden: bitwise the results of separate buffers."""
    hdim, vocab = 128, 1032
    h, w, y = make(n, hdim, vocab, seed=77)
    y[::3] = 5
    print(f"flce dhidden in place chunk={chunk}", flush=True)
    hd, wd, yd = h.to(DEV), w.to(DEV), y.to(DEV)
    loss, _, _, dh, dw = C.flce_fwd_bwd(hd, wd, yd, -100, None, True, chunk)
    L = _lib.lib()
    nbytes = L.siq_flce_workspace_bytes(n, hdim, vocab, chunk, 1)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    dw2, loss2 = torch.empty_like(wd), torch.empty_like(loss)
    count, bad = (torch.empty((), dtype=torch.int64, device=DEV) for _ in range(2))
    rc = L.siq_flce_fwd_bwd(hd.data_ptr(), wd.data_ptr(), yd.data_ptr(), n, hdim, vocab, -100, 0, None,
                            loss2.data_ptr(), count.data_ptr(), bad.data_ptr(), hd.data_ptr(), dw2.data_ptr(), chunk,
                            ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "siq_flce_fwd_bwd")
    assert torch.equal(loss, loss2)
    assert torch.equal(hd.view(torch.int16), dh.view(torch.int16))
    assert torch.equal(dw2.view(torch.int16), dw.view(torch.int16))
