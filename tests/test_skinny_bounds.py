"""CPU: the address range of the short-prompt (T <= 64) streamed GEMMs, bounded on the host.

The index arithmetic of yalm_amd/csrc/prefill_skinny.h (stream_gemm_kernel) and prefill.hip
(plan_stream) is restated here for every GEMM the prefill launches at T = 1..64 (enqueue_prefill,
the `small` path) at the production shapes: the A-row and weight-row DMA sources (rows clamped to
T - 1, the workgroup's rows inside the matrix, columns inside the slice), the LDS destinations of
every stage inside the ring, the partial slots inside their buffer, and the K slices, which cover K
once each.
"""
import math

import pytest

from yalm_amd import models as M

SK_MAX_T, KSTG, CUS = 64, 128, 256


def sk_rows(T):
    return 16 if T <= 16 else 32 if T <= 32 else 64


def sk_cols(T):
    return 64 if T <= 32 else 128


def plan_stream(T, N, nst, cap):
    """prefill.hip plan_stream."""
    blocks, rows = -(-N // sk_cols(T)), sk_rows(T)
    slots = CUS * (2 if T <= 32 else 1)
    best, least = None, 0.0
    for ks in range(1, min(16, nst) + 1):
        nsc = -(-nst // ks)
        k = -(-nst // nsc)
        floats = k * rows * blocks * sk_cols(T)
        if k != ks or (ks > 1 and (nsc < 2 or floats > cap)):
            continue
        items = blocks * ks
        t = math.ceil(items / slots) * (nsc * max(0.7, 1.27 * min(1.0, items / slots)) + 2.0)
        if ks > 1:
            t += 4.0 + floats * 8.0 / 5e6
        if best is None or t < least:
            best, least = (ks, nsc), t
    return best


def stream_cfg(T, eb, dual):
    """StreamCfg: (waves, MT, stage bytes, ring depth, weight / A DMAs per wave)."""
    mt, nw = {16: (1, 4), 32: (2, 4), 64: (4, 8)}[sk_rows(T)]
    wb, ab = nw * 16 * KSTG * eb, 16 * mt * KSTG * 2
    sb = wb + ab * (2 if dual else 1)
    fit2, fit1 = 81920 // sb, 163840 // sb
    ns = min(fit2, 6) if fit2 >= 3 else min(fit1, 4)
    assert ns >= 2 and ns * sb <= 163840 and 4 * mt % nw == 0
    return nw, mt, wb, ab, sb, ns, KSTG * eb // 64, 4 * mt // nw


CFGS = {"mistral-7b": M.MISTRAL_7B, "llama-3.2-3b": M.LLAMA_32_3B,
        "gqa-d128": M.ModelConfig(dim=512, hidden_dim=1024, head_dim=128, n_layers=3, n_heads=4, n_kv_heads=2,
                                  vocab_size=1024, max_seq_len=320, rope_theta=1e6),
        "d768": M.ModelConfig(dim=768, hidden_dim=1536, head_dim=128, n_layers=2, n_heads=6, n_kv_heads=2,
                              vocab_size=1920, max_seq_len=40, rope_theta=1e6)}


@pytest.mark.parametrize("eb", [1, 2])
@pytest.mark.parametrize("name", list(CFGS))
def test_stream_gemm_stays_inside_its_buffers(name, eb):
    c = CFGS[name]
    cap16 = -(-c.max_seq_len // 16) * 16
    np_qkv = c.q_dim + 2 * c.kv_dim
    skp = min(32 << 20, 16 * max(cap16, SK_MAX_T) * (max(np_qkv, c.dim, 2 * c.hidden_dim) + 64))
    for T in range(1, min(SK_MAX_T, c.max_seq_len) + 1):
        # (lda, K, B row width, columns, halves of A, GLU)
        gemms = [("qkv", 2 * c.dim, c.dim, np_qkv, True, False), ("wo", c.q_dim, c.q_dim, c.dim, False, False),
                 ("glu", c.dim, c.dim, 2 * c.hidden_dim, False, True), ("w2", c.hidden_dim, c.hidden_dim, c.dim, False, False)]
        for g, lda, K, N, dual, glu in gemms:
            nw, mt, wb, ab, sb, ns, nwi, na = stream_cfg(T, eb, dual)
            assert K % KSTG == 0 and N % (16 * nw) == 0, (name, g)
            ks, nsc = plan_stream(T, N, K // KSTG, skp)
            slices = [(i * nsc, min(nsc, K // KSTG - i * nsc)) for i in range(ks)]
            assert all(n > 0 for _, n in slices) and sum(n for _, n in slices) == K // KSTG
            assert ks == 1 or ks * 16 * mt * N <= skp
            for lane in range(64):
                for wave in range(nw):
                    for i in range(na):  # A: 4 rows of 256 bytes per DMA
                        r = 4 * (wave * na + i) + (lane >> 4)
                        assert r < 16 * mt and 8 * ((lane & 15) ^ (r & 15)) + 8 <= KSTG
                        assert (wave * na + i + 1) * 1024 <= ab
                    for i in range(nwi):
                        rr = 4 * i + (lane >> 4) if eb == 2 else 8 * i + (lane >> 3)
                        ch = (lane & 15) ^ rr if eb == 2 else (lane & 7) ^ ((rr >> 1) & 7)
                        assert rr < 16 and (16 // eb) * ch + 16 // eb <= KSTG
                        assert (wave * nwi + i + 1) * 1024 <= wb
            st0, n = slices[-1]
            k_end = (st0 + n) * KSTG
            assert k_end <= K and (min(16 * mt - 1, T - 1) * lda + k_end + (K if dual else 0)) <= T * lda


@pytest.mark.parametrize("eb", [1, 2])
def test_stream_gemm_fragments_read_what_the_dma_wrote(eb):
    """The swizzle of the DMA's source and of the fragment reads: lane (n, q) of k-step j gets the 8 columns
    32 j + 8 q .. of row n, for A and weights, and no bank is read twice by 32 lanes of one weight read."""
    a_lds, w_lds = {}, {}
    for lane in range(64):
        for i in range(4):
            r = 4 * i + (lane >> 4)
            a_lds[i * 1024 + lane * 16] = (r, 8 * ((lane & 15) ^ (r & 15)))
        for i in range(KSTG * eb // 64):
            rr = 4 * i + (lane >> 4) if eb == 2 else 8 * i + (lane >> 3)
            ch = (lane & 15) ^ rr if eb == 2 else (lane & 7) ^ ((rr >> 1) & 7)
            w_lds[i * 1024 + lane * 16] = (rr, 16 // eb * ch)
    for j in range(4):
        banks = [set(), set()]
        for lane in range(64):
            n, q = lane & 15, lane >> 4
            assert a_lds[n * 256 + 16 * ((4 * j + q) ^ n)] == (n, 32 * j + 8 * q)
            if eb == 2:
                at, off = n * 256 + 16 * ((4 * j + q) ^ n), 0
            else:
                at, off = n * 128 + 16 * ((2 * j + (q >> 1)) ^ ((n >> 1) & 7)), 8 * (q & 1)
            row, col = w_lds[at]
            assert (row, col + off) == (n, 32 * j + 8 * q)
            if eb == 1:
                banks[lane >> 5].add((at + off) % 256)
        assert eb == 2 or all(len(b) == 32 for b in banks)
