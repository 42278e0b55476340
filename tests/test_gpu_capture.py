"""Capture-side index upkeep from captured graph views (typed, strided), bit for
bit against ordered fp32 sums on the host: the query accumulator with the
query-span row filter (llama-memory-kvmem.cpp:3417-3433, 3470-3483), the
mean-K sums (write_layer_mean_k, raw_kv_store.cpp:685-705) and the decode
running sum with its flush (kvmem_meank_*, llama-kvmem-stagein.cu:1066-1097;
write_layer_mean_sum, raw_kv_store.cpp:707-731)."""
import numpy as np
import pytest
import torch

from gpu_util import host
from kvmem_amd import api

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _captured(rng, n_tok, heads, dims, dt, layout):
    """A [tokens][heads][dims] view of the given dtype: contiguous, or the
    [heads][tokens][dims] tensor ggml captures before a permute (strided), or
    every other dim of a wider tensor (nb0 of two elements)."""
    x = torch.from_numpy((rng.standard_normal((n_tok, heads, dims)) * 3).astype(np.float32)).to(DT[dt]).cuda()
    if layout == "contiguous":
        return x
    if layout == "heads_major":
        return x.permute(1, 0, 2).contiguous().permute(1, 0, 2)
    wide = torch.zeros((n_tok, heads, 2 * dims), dtype=DT[dt], device="cuda")
    wide[:, :, ::2] = x
    return wide[:, :, ::2]


def _f32_rows(v):
    return v.float().cpu().numpy().reshape(v.shape[0], -1)


def _ordered_sum(acc, rows):
    acc = acc.astype(np.float32).copy()
    for r in rows:
        acc = (acc + r).astype(np.float32)
    return acc


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("layout", ["contiguous", "heads_major", "strided_dim"])
def test_query_add_view(kvm_state, dt, layout):
    rng = np.random.default_rng(len(dt) * 7 + len(layout))
    n_head, D = 24, 256
    qa = api.QueryAcc(kvm_state, 2, n_head, D)
    qa.reset()
    q = _captured(rng, 9, n_head, D, dt, layout)
    keep = rng.random(9) < 0.6
    keep[0] = True
    qa.add_view(1, q, keep)
    qa.add_view(1, q[:3], None)
    rows = _f32_rows(q)
    want = _ordered_sum(np.zeros(n_head * D, np.float32), list(rows[keep]) + list(rows[:3]))
    got = host(qa.q_sum)
    assert np.array_equal(got[1].view(np.uint32), want.view(np.uint32))
    assert not got[0].any() and list(host(qa.q_count)) == [0, int(keep.sum()) + 3]


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("n", [32, 33, 128, 257, 600])
@pytest.mark.parametrize("offset", [0, 1])
def test_query_add_view_long_runs(kvm_state, dt, n, offset):
    """Row counts around the long-run form's threshold and LDS buffers, and the
    same rows from a base that is not 16-byte aligned (the general form), bit for
    bit: both keep the row order, and a row the mask leaves out is never added
    (it holds NaN here)."""
    rng = np.random.default_rng(n * 3 + offset)
    heads, D = 3, 128
    x = torch.from_numpy((rng.standard_normal((n, heads * D)) * 3).astype(np.float32)).to(DT[dt])
    keep = rng.random(n) < 0.7
    keep[: min(n, 70)] &= rng.random(min(n, 70)) < 0.1
    keep[n // 2] = True
    x[torch.from_numpy(~keep)] = float("nan")
    flat = torch.empty(n * heads * D + 1, dtype=DT[dt], device="cuda")
    q = flat[offset:offset + n * heads * D].view(n, heads, D)
    q.copy_(x.view(n, heads, D))
    qa = api.QueryAcc(kvm_state, 1, heads, D)
    qa.reset()
    qa.add_view(0, q, keep)
    rows = _f32_rows(q)
    want = _ordered_sum(np.zeros(heads * D, np.float32), list(rows[keep]))
    assert np.array_equal(host(qa.q_sum)[0].view(np.uint32), want.view(np.uint32))
    assert int(qa.q_count[0]) == int(keep.sum())


@pytest.mark.parametrize("n", [1, 3, 4, 5, 16, 17, 31])
def test_query_add_view_few_rows(kvm_state, n):
    """Row counts around the general form's loads in flight (4, 16), with and without
    a mask whose last row is kept."""
    rng = np.random.default_rng(n)
    qa = api.QueryAcc(kvm_state, 1, 3, 128)
    qa.reset()
    q = _captured(rng, n, 3, 128, "bf16", "heads_major")
    keep = rng.random(n) < 0.5
    keep[-1] = True
    qa.add_view(0, q, keep)
    qa.add_view(0, q)
    rows = _f32_rows(q)
    want = _ordered_sum(np.zeros(384, np.float32), list(rows[keep]) + list(rows))
    assert np.array_equal(host(qa.q_sum)[0].view(np.uint32), want.view(np.uint32))
    assert int(host(qa.q_count)[0]) == int(keep.sum()) + n


def test_query_add_view_more_rows_than_one_launch(kvm_state):
    rng = np.random.default_rng(5)
    qa = api.QueryAcc(kvm_state, 1, 2, 128)
    qa.reset()
    q = _captured(rng, 2100 + 37, 2, 128, "f16", "heads_major")
    keep = rng.random(q.shape[0]) < 0.5
    qa.add_view(0, q, keep)
    want = _ordered_sum(np.zeros(256, np.float32), _f32_rows(q)[keep])
    assert np.array_equal(host(qa.q_sum)[0].view(np.uint32), want.view(np.uint32))
    assert int(host(qa.q_count)[0]) == int(keep.sum())


@pytest.mark.parametrize("dt,layout", [("f16", "heads_major"), ("bf16", "strided_dim"), ("f32", "contiguous")])
def test_meank_add_view(kvm_state, dt, layout):
    """Prefill ubatches at positions 0.. and 300.. (the second continues the
    block the first left partly filled), as the capture hook hands them over."""
    rng = np.random.default_rng(11)
    H, D, bt = 4, 256, 128
    ix = api.MeanKIndex(kvm_state, 2, 8, H, D, bt)
    k1 = _captured(rng, 300, H, D, dt, layout)
    k2 = _captured(rng, 150, H, D, dt, layout)
    ix.add_view(1, 0, k1)
    ix.add_view(1, 300, k2)
    rows = np.concatenate([_f32_rows(k1), _f32_rows(k2)])
    got = host(ix.block_sums())[1]
    for b in range(4):
        n = min(bt, 450 - b * bt)
        want = _ordered_sum(np.zeros(H * D, np.float32), rows[b * bt:b * bt + n])
        assert np.array_equal(got[b].view(np.uint32), want.view(np.uint32)), b
    assert list(host(ix.mean_tokens)[1][:5]) == [128, 128, 128, 66, 0]
    assert list(host(ix.present)[:5]) == [1, 1, 1, 1, 0]


@pytest.mark.parametrize("H,D,bt", [(4, 256, 128), (3, 128, 64), (1, 128, 192)])
@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
def test_meank_add_forms_block_terms(kvm_state, H, D, bt, dt):
    """An add over ragged position ranges (a part of one block, whole blocks, the
    block continued) leaves the sums of an index without terms and the terms
    kvm_meank_refresh forms from those sums, bit for bit; blocks it did not
    touch keep theirs."""
    rng = np.random.default_rng(H * D + bt)
    nb = 6
    ix = api.MeanKIndex(kvm_state, 1, nb, H, D, bt, norms=True)
    plain = api.MeanKIndex(kvm_state, 1, nb, H, D, bt)
    ix.k_norm.fill_(-1.0)
    for pos0, n in ((0, 1), (bt + 5, 2 * bt), (3 * bt + 5, bt - 5 + 3)):
        k = _captured(rng, n, H, D, dt, "contiguous")
        ix.add_view(0, pos0, k)
        plain.add_view(0, pos0, k)
    assert torch.equal(ix.k_sum.view(torch.int32), plain.k_sum.view(torch.int32))
    assert torch.equal(ix.mean_tokens, plain.mean_tokens)
    got = ix.k_norm.clone()
    assert bool((got[0, :, 5] == -1.0).all())
    ix.refresh()
    assert torch.equal(got[0, :, :5].contiguous().view(torch.int32), ix.k_norm[0, :, :5].contiguous().view(torch.int32))


@pytest.mark.parametrize("norms", [False, True])
@pytest.mark.parametrize("n", [1, 2, 3, 8, 9, 47, 48, 49, 64, 65])
def test_meank_add_token_counts(kvm_state, n, norms):
    """Token counts around the kernel's loads in flight (2, 8, 64), across the end of
    a block: the sums in token order, the counts, and the terms of a refresh."""
    rng = np.random.default_rng(n)
    H, D, bt = 2, 256, 64
    ix = api.MeanKIndex(kvm_state, 1, 4, H, D, bt, norms=norms)
    first = _captured(rng, bt - n // 2, H, D, "f32", "contiguous")
    k = _captured(rng, n, H, D, "bf16", "strided_dim")
    ix.add_view(0, 0, first)
    ix.add_view(0, bt - n // 2, k)
    rows = np.concatenate([_f32_rows(first), _f32_rows(k)])
    got = host(ix.block_sums())[0]
    for b in range(2):
        want = _ordered_sum(np.zeros(H * D, np.float32), rows[b * bt:(b + 1) * bt])
        assert np.array_equal(got[b].view(np.uint32), want.view(np.uint32)), b
    assert list(host(ix.mean_tokens)[0][:2]) == [bt, len(rows) - bt]
    if norms:
        terms = ix.k_norm.clone()
        ix.refresh()
        assert torch.equal(terms.view(torch.int32), ix.k_norm.view(torch.int32))


def test_meank_decode_running_sum_and_flush(kvm_state):
    """Accepted decode tokens go to the running sum (two commits, the second
    keeping 2 of 3 MTP tokens), which is flushed into a block the prompt left
    partly filled (its sum += the running sum, not a continued ordered sum) and,
    after a zero, into a fresh block (its sum = the running sum)."""
    rng = np.random.default_rng(13)
    H, D, bt = 4, 256, 128
    ix = api.MeanKIndex(kvm_state, 1, 4, H, D, bt)
    prompt = _captured(rng, 200, H, D, "f32", "contiguous")
    ix.add_view(0, 0, prompt)                        # block 1 holds positions 128..199
    ix.acc_zero(0)
    d1 = _captured(rng, 2, H, D, "bf16", "heads_major")
    d2 = _captured(rng, 3, H, D, "bf16", "heads_major")
    ix.acc_add(0, d1, 0, 2)
    ix.acc_add(0, d2, 0, 2)
    ix.acc_flush(0, 200, 4)                          # positions 200..203 of block 1
    ix.acc_zero(0)
    d3 = _captured(rng, 5, H, D, "f16", "strided_dim")
    ix.acc_add(0, d3, 1, 4)
    ix.acc_flush(0, 256, 4)                          # positions 256..259: block 2 starts
    rows = _f32_rows(prompt)
    block1 = _ordered_sum(np.zeros(H * D, np.float32), rows[128:200])
    acc1 = _ordered_sum(np.zeros(H * D, np.float32), list(_f32_rows(d1)) + list(_f32_rows(d2)[:2]))
    acc2 = _ordered_sum(np.zeros(H * D, np.float32), _f32_rows(d3)[1:5])
    got = host(ix.block_sums())[0]
    assert np.array_equal(got[1].view(np.uint32), (block1 + acc1).astype(np.float32).view(np.uint32))
    assert np.array_equal(got[2].view(np.uint32), acc2.view(np.uint32))
    assert np.array_equal(host(ix.acc)[0].view(np.uint32), acc2.view(np.uint32))     # flush keeps it
    assert list(host(ix.mean_tokens)[0]) == [128, 76, 4, 0]


def test_view_shape_is_checked(kvm_state):
    qa = api.QueryAcc(kvm_state, 1, 8, 128)
    with pytest.raises(api.L.KvmError):
        qa.add_view(0, torch.zeros((2, 4, 128), dtype=torch.float16, device="cuda"))
    ix = api.MeanKIndex(kvm_state, 1, 4, 2, 128, 128)
    k = torch.zeros((2, 2, 128), dtype=torch.float32, device="cuda")
    v = api.view(k)
    v.type = api.L.T_Q8_0                            # a quantised view is not a captured output
    assert kvm_state.lib.kvm_meank_add_view(kvm_state.h, api.C.byref(ix.c), 0, 0, api.C.byref(v)) == api.L.KVM_EUNSUPPORTED


@pytest.mark.parametrize("H,G,D", [(4, 6, 256), (8, 4, 128), (1, 5, 128), (8, 3, 256)])
@pytest.mark.parametrize("n,dt", [(1, "f32"), (4, "bf16"), (8, "f16"), (9, "f32")])
def test_query_add_few_rows_with_terms(kvm_state, H, G, D, n, dt):
    """The one-launch form for a few rows and the general one past its limits (more
    rows, more than 1,024 kv values): sums in row order, the mask's rows only, and
    the terms that kvm_query_refresh forms from those sums, bit for bit."""
    rng = np.random.default_rng(H * G + n)
    qa = api.QueryAcc(kvm_state, 2, H * G, D, n_head_kv=H)
    qa.reset()
    total, want = 0, np.zeros(H * G * D, np.float32)
    for rnd in range(2):
        q = _captured(rng, n, H * G, D, dt, "heads_major" if rnd else "contiguous")
        keep = None if rnd else np.arange(n) % 3 != 1
        qa.add_view(1, q, keep)
        rows = _f32_rows(q)
        rows = rows if keep is None else rows[keep]
        want = _ordered_sum(want, list(rows))
        total += len(rows)
    assert np.array_equal(host(qa.q_sum)[1].view(np.uint32), want.view(np.uint32))
    assert not host(qa.q_sum)[0].any() and list(host(qa.q_count)) == [0, total]
    vec, norm = qa.q_vec.clone(), qa.q_norm.clone()
    qa.refresh()
    assert torch.equal(vec.view(torch.int32), qa.q_vec.view(torch.int32))
    assert torch.equal(norm.view(torch.int32), qa.q_norm.view(torch.int32))
