"""Shared helpers for the GPU parity tests: move workload arrays to the device, run the oracle on a
subset of sequences, and compare verify results with the documented exemptions."""
from __future__ import annotations

import os

import numpy as np
import torch

import oracle
from kyro_amd import workloads as wl

ATOL_BF16 = 2e-2   # attention outputs, bf16 inputs
ATOL_F32 = 1e-3    # attention outputs, f32 inputs
# The same for averages of N(0, 1) values over up to 6000 tokens: scores of at most 64 roundings in a chain
# (2^-24 of partial sums up to about 4 after the scale: 1.5e-5 of a weight if all had one sign, 2e-6 as they
# fall) and sums of weights and values about as deep; 3.5e-7 rms and below 3e-6 at most as measured. A
# token lost or doubled in 6000 moves an output by about 1 / 6000.
ATOL_F32_SUMS = 1e-5
PROB_ATOL = 1e-5   # p_i(x_i), q_i(x_i)
MARGIN = 1e-5      # decisions with |u - boundary| below this may differ under f32 rounding
ORACLE_THREADS = max(1, min(16, os.cpu_count() or 1))


def to_device(a: np.ndarray, device, bf16: bool = False) -> torch.Tensor:
    t = torch.from_numpy(np.ascontiguousarray(a))
    if bf16:
        t = t.view(torch.bfloat16)
    return t.to(device)


def attention_tensors(case: wl.AttentionCase, device):
    bf16 = case.dtype == "bf16"
    return dict(
        query=to_device(case.query, device, bf16),
        key_cache=to_device(case.key_cache, device, bf16),
        value_cache=to_device(case.value_cache, device, bf16),
        block_table=to_device(case.block_table, device),
        context_lens=to_device(case.context_lens, device),
        q_start_loc=to_device(case.q_start_loc, device),
    )


def oracle_attention(case: wl.AttentionCase, seqs=None, causal=True) -> dict:
    """Oracle rows for the chosen sequences, gathering only their blocks (so a full-size case is
    checked without running the oracle over the whole batch). Returns {seq: [q_len, H, D]}."""
    seqs = range(case.batch) if seqs is None else seqs
    res = {}
    for b in seqs:
        ctx = int(case.context_lens[b])
        nb = max(1, -(-ctx // case.block_size))
        blocks = case.block_table[b, :nb]
        q0, q1 = int(case.q_start_loc[b]), int(case.q_start_loc[b + 1])
        res[b] = oracle.paged_attention_mq(
            case.query[q0:q1], case.key_cache[blocks], case.value_cache[blocks],
            np.arange(nb, dtype=np.int64)[None], np.array([ctx], np.int64),
            num_heads=case.num_heads, num_kv_heads=case.num_kv_heads, head_dim=case.head_dim,
            block_size=case.block_size, q_start_loc=np.array([0, q1 - q0], np.int32), causal=causal,
            threads=ORACLE_THREADS)
    return res


def attention_float64(case: wl.AttentionCase) -> torch.Tensor:
    """Causal attention of every query row in 64 bits, [total_q, H, D], on the host."""
    H, Hkv, D = case.num_heads, case.num_kv_heads, case.head_dim
    cast = (lambda x: wl.bf16_bits_to_f32(x)) if case.dtype == "bf16" else np.asarray
    out = torch.zeros(case.query.shape, dtype=torch.float64)
    for b in range(case.batch):
        ctx = int(case.context_lens[b])
        q0, q1 = int(case.q_start_loc[b]), int(case.q_start_loc[b + 1])
        n = q1 - q0
        if n == 0 or ctx == 0:
            continue
        ids = case.block_table[b, :-(-ctx // case.block_size)]
        k, v = (torch.from_numpy(cast(x[ids])).double().transpose(0, 1).reshape(Hkv, -1, D)[:, :ctx]
                for x in (case.key_cache, case.value_cache))
        q = torch.from_numpy(cast(case.query[q0:q1])).double().view(n, Hkv, H // Hkv, D).permute(1, 2, 0, 3)
        s = torch.matmul(q.reshape(Hkv, -1, D), k.transpose(1, 2)).view(Hkv, H // Hkv, n, ctx) / D ** 0.5
        seen = torch.arange(ctx) <= ctx - n + torch.arange(n).view(-1, 1)
        p = torch.softmax(s.masked_fill(~seen, float("-inf")), -1).nan_to_num()  # a row that sees nothing: 0
        o = torch.matmul(p.view(Hkv, -1, ctx), v).view(Hkv, H // Hkv, n, D)
        out[q0:q1] = o.permute(2, 0, 1, 3).reshape(n, H, D)
    return out


def assert_attention_close(out: torch.Tensor, case: wl.AttentionCase, expected: dict, atol: float):
    got = out.float().cpu().numpy()
    worst = 0.0
    for b, ref in expected.items():
        q0, q1 = int(case.q_start_loc[b]), int(case.q_start_loc[b + 1])
        err = float(np.max(np.abs(got[q0:q1] - ref))) if q1 > q0 else 0.0
        worst = max(worst, err)
        assert np.isfinite(got[q0:q1]).all(), f"non-finite output in sequence {b}"
        assert err <= atol, f"sequence {b}: max abs error {err:.3g} > {atol}"
    return worst


def verify_tensors(case: wl.VerifyCase, device, with_draft=True):
    return dict(
        target_logits=to_device(case.target, device),
        draft_logits=to_device(case.draft, device) if with_draft else None,
        draft_tokens=to_device(case.draft_tokens.astype(np.int32), device),
        num_draft=to_device(case.num_draft.astype(np.int32), device),
        temperature=to_device(case.temperature.astype(np.float32), device),
        u_accept=to_device(case.u_accept, device),
        u_resample=to_device(case.u_resample, device),
    )


def oracle_verify(case: wl.VerifyCase) -> dict:
    return oracle.spec_verify(case.target, case.draft, case.draft_tokens, case.num_draft,
                              case.temperature, case.u_accept, case.u_resample)


def assert_verify_parity(res, case: wl.VerifyCase, orc: dict, max_exempt: int = 0):
    """Accepted lengths and emitted tokens bit-exact, except decisions the oracle places within
    MARGIN of a boundary. Probabilities within PROB_ATOL. Returns the number of exemptions."""
    acc = res.accepted.cpu().numpy()
    tok = res.tokens.cpu().numpy().view(np.uint32)
    exempt = 0
    for b in range(case.batch):
        a_g, a_o = int(acc[b]), int(orc["accepted"][b])
        if a_g != a_o:
            i = min(a_g, a_o)
            m = orc["accept_margin"][b, i]
            assert m < MARGIN, f"seq {b}: accepted {a_g} vs oracle {a_o}, margin {m:.3g} at position {i}"
            exempt += 1
            continue
        if not np.array_equal(tok[b], orc["tokens"][b]):
            assert np.array_equal(tok[b, :a_g], orc["tokens"][b, :a_g]), f"seq {b}: accepted drafts differ"
            m = orc["resample_margin"][b]
            assert m < MARGIN, (f"seq {b}: emitted {tok[b, a_g]} vs oracle {orc['tokens'][b, a_g]}, "
                                f"resample margin {m:.3g}")
            exempt += 1
    assert exempt <= max_exempt, f"{exempt} margin exemptions"
    if res.p_draft is not None:
        # The scan stops at the first rejection: probabilities exist for drafts 0 .. accepted of
        # sampled sequences and are NaN after it.
        pos = np.arange(case.draft_tokens.shape[1])[None, :]
        evaluated = ((pos < case.num_draft[:, None]) & (pos <= acc[:, None])
                     & (case.temperature[:, None] > 0))
        for name in ("p_draft", "q_draft"):
            g = getattr(res, name).cpu().numpy().astype(np.float64)
            assert np.array_equal(~np.isnan(g), evaluated), f"{name}: NaN pattern differs from the scan"
            o = orc[name]
            both = ~np.isnan(g) & ~np.isnan(o)
            if both.any():
                err = np.max(np.abs(g[both] - o[both]))
                assert err <= PROB_ATOL, f"{name} max abs error {err:.3g}"
    return exempt
