"""The training forwards write every score and every winner, on buffers that
hold a sentinel before the call: -1 where there is no winner (a document that is
empty or out of range), else a token of the document; entries of query tokens past
their query's end (or of a query out of range), which nothing reads, hold either. Packed documents with empty ones, pair lists with ids out of
range, queries of one and of several column chunks, 16-bit and fp32 rows, rows
wider than a column block."""

import ctypes

import pytest
import torch

from late_interaction_kernels import _lib

pytestmark = pytest.mark.gpu

STALE = 0x7FFFFFFF
DTYPES = [torch.bfloat16, torch.float16, torch.float32]


def _cu(lens):
    return torch.nn.functional.pad(torch.tensor(lens).cumsum(0), (1, 0)).to(torch.int32).cuda()


def _buffers(units, docs, lq):
    out = torch.full((units, docs) if docs else (units,), float("nan"), device="cuda")
    return out, torch.full((units * max(docs, 1), lq), STALE, device="cuda", dtype=torch.int32)


def _check(out, am, q_lens, d_lens):
    """``q_lens`` / ``d_lens``: the query and document length of each row of ``am`` (0: no winner)."""
    assert torch.isfinite(out).all()
    am = am.cpu()
    assert (am >= -1).all() and (am < d_lens[:, None]).all()  # no sentinel; -1 for length 0
    token = (torch.arange(am.shape[1])[None] < q_lens[:, None]) & (d_lens[:, None] > 0)
    assert (am[token] >= 0).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d", [64, 128, 1024])
@pytest.mark.parametrize("q_lens", [[32, 5, 0, 17], [7], [300, 1, 129], [700, 33], [1300, 20]])
def test_packed_cross_product(q_lens, d, dtype):
    d_lens = [40, 0, 1, 300, 32, 0, 33, 64, 0]
    g = torch.Generator().manual_seed(d + sum(q_lens))
    Q = torch.randn(sum(q_lens), d, generator=g).to(dtype).cuda()
    D = torch.randn(sum(d_lens), d, generator=g).to(dtype).cuda()
    cq, cd, lq = _cu(q_lens), _cu(d_lens), max(q_lens)
    out, am = _buffers(len(q_lens), len(d_lens), lq)
    qs = _lib.seqs(Q, n=len(q_lens), length=lq, stride_l=d, cu=cq)
    ds = _lib.seqs(D, n=len(d_lens), length=max(d_lens), stride_l=d, cu=cd)
    lib = _lib.load()
    nbytes = lib.lik_maxsim_workspace_size(ctypes.byref(qs), ctypes.byref(ds), 0)
    ws = _lib.workspace(nbytes, Q.device)
    rc = lib.lik_maxsim_argmax(ctypes.byref(qs), ctypes.byref(ds), 0, out.data_ptr(), out.stride(0), out.stride(1),
                               am.data_ptr(), _lib.ptr(ws), nbytes, _lib.stream_of(out))
    _lib.check(rc, "lik_maxsim_argmax")
    _check(out, am, torch.tensor(q_lens).repeat_interleave(len(d_lens)), torch.tensor(d_lens).repeat(len(q_lens)))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d", [64, 128, 1024])
@pytest.mark.parametrize("q_lens", [[32, 5, 0, 17], [7], [300, 1, 129], [700, 33], [1300, 20]])
def test_pairs(q_lens, d, dtype):
    d_lens = [40, 0, 1, 300, 32, 33, 64]
    nq, nd = len(q_lens), len(d_lens)
    g = torch.Generator().manual_seed(d + sum(q_lens))
    Q = torch.randn(sum(q_lens), d, generator=g).to(dtype).cuda()
    D = torch.randn(sum(d_lens), d, generator=g).to(dtype).cuda()
    pq = torch.randint(0, nq, (61,), generator=g).to(torch.int32)
    pd = torch.randint(0, nd, (61,), generator=g).to(torch.int32)
    pq[3], pq[4], pd[5], pd[6], pd[60] = -1, nq, -1, nd, nd + 100
    cq, cd, lq = _cu(q_lens), _cu(d_lens), max(q_lens)
    out, am = _buffers(61, 0, lq)
    qs = _lib.seqs(Q, n=nq, length=lq, stride_l=d, cu=cq)
    ds = _lib.seqs(D, n=nd, length=max(d_lens), stride_l=d, cu=cd)
    pqd, pdd = pq.cuda(), pd.cuda()
    rc = _lib.load().lik_maxsim_pairs_argmax(ctypes.byref(qs), ctypes.byref(ds), pqd.data_ptr(), pdd.data_ptr(), 61, 0,
                                             out.data_ptr(), am.data_ptr(), _lib.stream_of(out))
    _lib.check(rc, "lik_maxsim_pairs_argmax")
    def at(lens, i):  # 0 for an id out of range
        return torch.where((i >= 0) & (i < len(lens)), torch.tensor(lens)[i.long().clamp(0, len(lens) - 1)], 0)

    _check(out, am, at(q_lens, pq), at(d_lens, pd))
    assert (out.cpu()[(at(q_lens, pq) == 0) | (at(d_lens, pd) == 0)] == 0).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kd", [False, True])
@pytest.mark.parametrize("Lq,d", [(32, 128), (5, 64), (300, 128), (700, 128), (32, 1024)])
def test_padded_with_masks(Lq, d, kd, dtype):
    Nq, K, Ld = 3, 5, 75
    nd = Nq * K if kd else 4 * K
    g = torch.Generator().manual_seed(Lq + d)
    Q = torch.randn(Nq, Lq, d, generator=g).to(dtype).cuda()
    D = torch.randn(nd, Ld, d, generator=g).to(dtype).cuda()
    dm = torch.rand(nd, Ld, generator=g) > 0.4  # holes
    dm[::3] = torch.arange(Ld)[None] < torch.randint(1, Ld + 1, (dm[::3].shape[0], 1), generator=g)  # prefixes
    dm[1::4] = False  # empty
    per = K if kd else nd
    out, am = _buffers(Nq, per, Lq)
    m = dm.to(torch.int8).cuda()
    qs = _lib.seqs(Q, n=Nq, length=Lq, stride_n=Lq * d, stride_l=d)
    ds = _lib.seqs(D, n=nd, length=Ld, stride_n=Ld * d, stride_l=d, mask=m, mask_strides=(Ld, 1))
    flags = _lib.LIK_KD_LAYOUT if kd else 0
    lib = _lib.load()
    nbytes = lib.lik_maxsim_workspace_size(ctypes.byref(qs), ctypes.byref(ds), flags)
    ws = _lib.workspace(nbytes, Q.device)
    rc = lib.lik_maxsim_argmax(ctypes.byref(qs), ctypes.byref(ds), flags, out.data_ptr(), out.stride(0), out.stride(1),
                               am.data_ptr(), _lib.ptr(ws), nbytes, _lib.stream_of(out))
    _lib.check(rc, "lik_maxsim_argmax")
    docs = torch.arange(nd) if kd else torch.arange(nd).repeat(Nq)
    last = torch.where(dm, torch.arange(1, Ld + 1)[None], 0).amax(1)  # 0: empty
    _check(out, am, torch.full((Nq * per,), Lq), last[docs])
    a = am.cpu().long()
    assert dm[docs].gather(1, a.clamp_min(0))[a >= 0].all()  # no dropped token wins
