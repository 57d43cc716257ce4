"""GPU parity of the indexer key write into vLLM's paged SHUFFLE cache (bit-exact bytes vs the oracle) and of the
paged logits over it (vs the fp64 oracle within the logits tolerance, identical -inf pattern, next_n > 1 and 2-D
seq_lens; bit-identical to the 132-byte-row kernel on the same keys where no clamp applies)."""
import numpy as np
import pytest
import torch

from oracle import spmla_ref as ref
from tests.helpers import bf16_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs,ue8m0", [(64, False), (16, True), (128, False)])
def test_key_write_shuffle(dev, bs, ue8m0):
    from arcagi2_flashnext_dots3_amd import kernels
    nb, n = 7, 300
    g = torch.Generator().manual_seed(bs)
    k = torch.randn(n, 128, generator=g).to(torch.bfloat16) * torch.exp(torch.randn(n, 1, generator=g) * 2).to(torch.bfloat16)
    k[3] = 0
    slots = torch.randperm(nb * bs, generator=g)[:n].to(torch.int64)
    slots[::17] = -1
    slots[5] = nb * bs + 9
    cache = torch.full((nb, bs, 1, 132), 0xA5, dtype=torch.uint8, device=dev)
    print(f"[shuffle write] bs={bs} ue8m0={ue8m0}", flush=True)
    kernels.index_key_write_shuffle(k.to(dev), slots.to(dev), cache, ue8m0=ue8m0)
    torch.cuda.synchronize()
    exp = np.full((nb, bs * 132), 0xA5, dtype=np.uint8)
    ref.index_key_write_shuffle(bf16_bits(k), slots.numpy(), exp, bs, ue8m0=ue8m0)
    assert np.array_equal(cache.cpu().numpy().reshape(nb, -1), exp)


@pytest.mark.parametrize("B,nn,L,two_d", [(4, 1, 2048, False), (3, 3, 5000, False), (2, 2, 700, True)])
def test_paged_mqa_logits(dev, B, nn, L, two_d):
    from arcagi2_flashnext_dots3_amd import kernels
    bs = 64
    nbp = (L + bs - 1) // bs
    nb = B * nbp + 2
    g = torch.Generator().manual_seed(L)
    k = torch.randn(nb * bs, 128, generator=g).to(torch.bfloat16)
    rows = np.zeros((nb * bs, 132), dtype=np.uint8)
    ref.index_key_write(bf16_bits(k), np.arange(nb * bs), rows)
    cache = torch.from_numpy(ref.shuffle_layout(rows, bs)).to(dev).view(nb, bs, 1, 132)
    bt = torch.randperm(nb, generator=g)[: B * nbp].reshape(B, nbp).to(torch.int32)
    q = torch.randn(B, nn, 64, 128, generator=g).to(torch.bfloat16)
    w = torch.rand(B * nn, 64, generator=g)
    if two_d:
        sl = torch.randint(L // 2, L + 1, (B, nn), generator=g).to(torch.int32)
    else:
        sl = torch.randint(L // 2, L + 1, (B,), generator=g).to(torch.int32)
        sl[0] = L
    print(f"[paged logits] B={B} next_n={nn} L={L} 2d={two_d}", flush=True)
    out = kernels.paged_mqa_logits(q.to(dev), cache, w.to(dev), sl.to(dev), bt.to(dev), L)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    exp = ref.paged_mqa_logits(q.float().numpy(), ref.shuffle_layout(rows, bs), w.numpy(), sl.numpy(), bt.numpy(), bs, L)
    assert np.array_equal(np.isinf(got), np.isinf(exp))
    fin = np.isfinite(exp)
    err = np.abs(got[fin] - exp[fin]) / np.maximum(1.0, np.abs(exp[fin]))
    print(f"[paged logits] max rel err {err.max():.3e}", flush=True)
    assert err.max() <= 2e-5
    # the same keys as 132-byte rows through the shard kernel: identical bits (only the addressing differs)
    req, ctx = kernels.paged_ctx(sl.to(dev), nn)
    out2 = kernels.index_logits(q.reshape(B * nn, 64, 128).to(dev), w.to(dev),
                                torch.from_numpy(rows).to(dev).view(nb, bs, 132), bt.to(dev), bs, req, ctx, L)
    torch.cuda.synchronize()
    assert torch.equal(out, out2)


def test_paged_logits_fp8_query(dev):
    """An e4m3 query (the reference's dtype) gives the logits of its exact bf16 widening."""
    from arcagi2_flashnext_dots3_amd import kernels
    bs, nb, B, L = 16, 8, 2, 100
    g = torch.Generator().manual_seed(3)
    rows = np.zeros((nb * bs, 132), dtype=np.uint8)
    ref.index_key_write(bf16_bits(torch.randn(nb * bs, 128, generator=g)), np.arange(nb * bs), rows)
    cache = torch.from_numpy(ref.shuffle_layout(rows, bs)).to(dev)
    q8 = (torch.randn(B, 1, 64, 128, generator=g) * 4).to(torch.float8_e4m3fn).to(dev)
    w = torch.rand(B, 64, generator=g).to(dev)
    bt = torch.arange(nb, dtype=torch.int32).reshape(B, nb // B).to(dev)
    sl = torch.tensor([L, 37], dtype=torch.int32, device=dev)
    a = kernels.paged_mqa_logits(q8, cache, w, sl, bt, L)
    b = kernels.paged_mqa_logits(q8.to(torch.bfloat16), cache, w, sl, bt, L)
    torch.cuda.synchronize()
    assert torch.equal(a, b)


def test_mqa_logits_flat(dev):
    """Prefill logits over a flat key gather [N, 128] + scales [N] with per-row [ks, ke) ranges vs the oracle."""
    from arcagi2_flashnext_dots3_amd import kernels
    N, M = 3000, 9
    g = torch.Generator().manual_seed(6)
    k = torch.randn(N, 128, generator=g).to(torch.bfloat16)
    rows = np.zeros((N, 132), dtype=np.uint8)
    ref.index_key_write(bf16_bits(k), np.arange(N), rows)
    codes = torch.from_numpy(rows[:, :128].copy())
    scales = torch.from_numpy(rows[:, 128:].copy().view(np.float32)[:, 0].copy())
    q = torch.randn(M, 64, 128, generator=g).to(torch.bfloat16)
    w = torch.rand(M, 64, generator=g)
    ks = torch.tensor([0, 0, 100, 2999, 500, 1000, 0, 64, 2048], dtype=torch.int32)
    ke = torch.tensor([3000, 1, 2100, 3000, 500, 2999, 257, 96, 3000], dtype=torch.int32)
    print("[mqa logits] flat", flush=True)
    out = kernels.mqa_logits(q.to(dev), (codes.to(dev).view(torch.float8_e4m3fn), scales.to(dev).view(N, 1)),
                             w.to(dev), ks.to(dev), ke.to(dev))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    exp = ref.mqa_logits(q.float().numpy(), rows[:, :128], rows[:, 128:].copy().view(np.float32)[:, 0], w.numpy(),
                         ks.numpy(), ke.numpy())
    assert np.array_equal(np.isinf(got), np.isinf(exp))
    fin = np.isfinite(exp)
    err = np.abs(got[fin] - exp[fin]) / np.maximum(1.0, np.abs(exp[fin]))
    print(f"[mqa logits] max rel err {err.max():.3e}", flush=True)
    assert err.max() <= 2e-5


@pytest.mark.parametrize("M,N", [(8, 1), (9, 511), (33, 512), (130, 513), (300, 1537), (67, 9000)])
def test_mqa_logits_many_rows(dev, M, N):
    """The many-row kernel (512 keys a workgroup, up to 64 rows past them) against the row-at-a-time kernel, which
    serves launches of fewer than 8 rows: bit for bit, over ranges that are empty, single keys, end inside a tile, miss a
    workgroup's keys or reach past N, signed weights, strided queries and 132-byte key rows; and against the oracle."""
    from arcagi2_flashnext_dots3_amd import kernels
    g = torch.Generator().manual_seed(M + N)
    k = torch.randn(N, 128, generator=g).to(torch.bfloat16)
    rows = np.zeros((N, 132), dtype=np.uint8)
    ref.index_key_write(bf16_bits(k), np.arange(N), rows)
    kd = torch.from_numpy(rows).to(dev)
    scales = torch.from_numpy(rows[:, 128:].copy().view(np.float32)[:, 0].copy()).to(dev)
    q = torch.randn(M, 64, 136, generator=g).to(torch.bfloat16).to(dev)[:, :, :128]
    w = torch.randn(M, 64, generator=g).to(dev)
    ks = torch.randint(0, N, (M,), generator=g).to(torch.int32)
    ke = (ks + torch.randint(0, N, (M,), generator=g)).to(torch.int32)
    ks[0], ke[0] = 0, N + 5
    ks[1], ke[1] = N - 1, N
    ke[2] = ks[2]
    ks[3], ke[3] = 0, 1
    print(f"[mqa logits] M={M} N={N}", flush=True)
    got = kernels.mqa_logits(q, (kd[:, :128], scales), w, ks.to(dev), ke.to(dev))
    one = torch.cat([kernels.mqa_logits(q[m:m + 7], (kd[:, :128], scales), w[m:m + 7], ks[m:m + 7].to(dev),
                                        ke[m:m + 7].to(dev)) for m in range(0, M, 7)])
    torch.cuda.synchronize()
    assert torch.equal(got, one)
    t = list(range(0, M, 29))
    exp = ref.mqa_logits(q[t].float().cpu().numpy(), rows[:, :128], scales.cpu().numpy(), w[t].cpu().numpy(), ks[t].numpy(),
                         ke[t].numpy())
    fin = np.isfinite(exp)
    assert np.array_equal(fin, np.isfinite(got[t].cpu().numpy()))
    # 2e-5 of sum |w| times the standard deviation of q . k (sqrt(128)): the bar of the one-signed logits above, relative
    # to the terms, since signed weights cancel
    scale = np.broadcast_to(np.abs(w[t].cpu().numpy()).sum(1)[:, None] * 128 ** 0.5, exp.shape)
    assert np.all(np.abs(got[t].cpu().numpy()[fin] - exp[fin]) <= 2e-5 * scale[fin])


@pytest.mark.parametrize("M,N,nreq", [(64, 16384, 8), (256, 9000, 5), (100, 40000, 64), (40, 20000, 1)])
def test_mqa_logits_short_ranges(dev, M, N, nreq):
    """Rows of several requests, each over its own keys, a small part of all: the workgroups of keys that no row of a chunk
    sees share the others' rows. The same bits as the row-at-a-time kernel, -inf everywhere else."""
    from arcagi2_flashnext_dots3_amd import kernels
    g = torch.Generator().manual_seed(M + N)
    codes = torch.randint(0, 120, (N, 128), generator=g, dtype=torch.uint8).to(dev)
    scales = torch.rand(N, generator=g).to(dev)
    q = torch.randn(M, 64, 128, generator=g).to(torch.bfloat16).to(dev)
    w = torch.randn(M, 64, generator=g).to(dev)
    r = torch.arange(M) * nreq // M
    ks = (r * (N // max(nreq, 8))).to(torch.int32)
    ke = (ks + 1 + torch.randint(0, N // max(nreq, 8), (M,), generator=g)).to(torch.int32)
    ke[M // 2] = ks[M // 2]
    ks, ke = ks.to(dev), ke.to(dev)
    print(f"[mqa logits] short ranges M={M} N={N} nreq={nreq}", flush=True)
    got = kernels.mqa_logits(q, (codes, scales), w, ks, ke)
    exp = torch.cat([kernels.mqa_logits(q[i:i + 4], (codes, scales), w[i:i + 4], ks[i:i + 4], ke[i:i + 4]) for i in range(0, M, 4)])
    assert torch.equal(got, exp) and int((got > -float("inf")).sum()) == int((ke - ks).sum())



@pytest.mark.parametrize("B,nn,two_d,dtype", [(3, 2, False, torch.int64), (3, 4, True, torch.int32), (5, 1, False, torch.int32)])
def test_paged_logits_rows_formed_in_the_kernel(dev, B, nn, two_d, dtype):
    """spmla_paged_mqa_logits_seq (the wrapper) against spmla_paged_mqa_logits with explicit per-row requests and
    contexts: the same bits; a context shorter than next_n leaves its first rows without keys."""
    from arcagi2_flashnext_dots3_amd import _lib, kernels
    bs, L = 16, 130
    nbp = (L + bs - 1) // bs
    g = torch.Generator().manual_seed(B * nn)
    cache = torch.zeros(B * nbp, bs, 132, dtype=torch.uint8, device=dev)
    kernels.index_key_write_shuffle(torch.randn(B * nbp * bs, 128, generator=g).to(torch.bfloat16).to(dev),
                                    torch.arange(B * nbp * bs, device=dev), cache)
    bt = torch.randperm(B * nbp, generator=g).view(B, nbp).to(torch.int32).to(dev)
    q = torch.randn(B, nn, 64, 128, generator=g).to(torch.bfloat16).to(dev)
    w = torch.rand(B * nn, 64, generator=g).to(dev)
    sl = torch.randint(1, L + 1, (B, nn) if two_d else (B,), generator=g).to(dtype)
    sl.view(-1)[0] = 1
    sl = sl.to(dev)
    print(f"[paged logits] B={B} next_n={nn} 2d={two_d}", flush=True)
    a = kernels.paged_mqa_logits(q, cache, w, sl, bt, L)
    req, ctx = kernels.paged_ctx(sl, nn)
    b = torch.empty_like(a)
    _lib.call("spmla_paged_mqa_logits", q.data_ptr(), q.stride(1), q.stride(2), w.data_ptr(), w.stride(0),
              cache.data_ptr(), B * nbp, bs, cache.stride(0), bt.data_ptr(), bt.stride(0), req.data_ptr(), ctx.data_ptr(),
              B * nn, 64, 128, L, 0, b.data_ptr(), b.stride(0), kernels._stream(q))
    torch.cuda.synchronize()
    assert torch.equal(a, b)
