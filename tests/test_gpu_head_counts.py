"""Other head counts than Bonsai's 8 KV heads (n_head = 4 n_kv_head, the only
grouping the reference accepts: src/model.rs:672), HIP path vs CPU oracle.

The kernels take the head count from the model: grids, the decode layouts (four
KV heads per workgroup only when n_kv_head is a multiple of 4) and the XCD
order of the prefill grid all follow it. Same bars as test_gpu_parity.py:
cache bytes and normalized q bit-exact, attention within max-abs 2e-3 and
rel-L2 1e-3 of the oracle.
"""
import sys

import numpy as np
import pytest

from bonsai_pot_amd import layout
from helpers import DeviceScenario, Scenario, assert_attn_close

pytestmark = pytest.mark.gpu

KV_HEADS = [1, 2, 4, 12]


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _cfg(kv):
    return layout.Config(n_layer=2, n_head=4 * kv, n_kv_head=kv)


def _prefill_cache(sc, il, n_rows, seed):
    if n_rows == 0:
        return
    pre = Scenario(sc.cfg, sc.max_seq, n_rows, seed=seed, with_q=False)
    pre.oracle_writeback(il, 0)
    sc.kv_k[:], sc.kv_v[:] = pre.kv_k, pre.kv_v


@pytest.mark.parametrize("kv", KV_HEADS)
def test_writeback_and_q_norm_rope(cuda, kv):
    _say(f"[heads] writeback n_kv_head={kv}")
    sc = Scenario(_cfg(kv), max_seq=64, m_tokens=5, seed=10 + kv, w_std=0.1)
    dev = DeviceScenario(sc)
    dev.writeback(il=1, pos_base=10)
    dev.q_norm_rope(10)
    sc.oracle_writeback(il=1, pos_base=10)
    sc.oracle_q_norm_rope(10)
    k, v = dev.kv_host()
    assert np.array_equal(k, sc.kv_k) and np.array_equal(v, sc.kv_v), "cache bytes differ"
    assert np.array_equal(dev.act_host(), sc.act), "q_norm_rope output differs"


@pytest.mark.parametrize("kv", KV_HEADS)
@pytest.mark.parametrize("pos", [300, 500, 9000])
def test_decode_step(cuda, kv, pos):
    """The fused step: the single layout at 300 rows, narrow splits at 500, and at
    9000 the wide layout when n_kv_head % 4 == 0."""
    _say(f"[heads] decode step n_kv_head={kv} pos={pos}")
    cfg = _cfg(kv)
    sc = Scenario(cfg, max_seq=pos + 4, m_tokens=1, seed=20 + kv + pos)
    _prefill_cache(sc, 1, pos, seed=30 + kv + pos)
    dev = DeviceScenario(sc, upload_kv=True)
    dev.decode_step(1, pos)
    sc.oracle_q_norm_rope(pos)
    sc.oracle_writeback(1, pos)
    k, v = dev.kv_host()
    assert np.array_equal(k, sc.kv_k) and np.array_equal(v, sc.kv_v), "cache bytes differ"
    _, want = sc.oracle_decode(1, pos)
    assert_attn_close(dev.out_f32(1)[0], want, f"decode step n_kv_head={kv} pos={pos}")


@pytest.mark.parametrize("kv", KV_HEADS)
@pytest.mark.parametrize("m,pos_base", [(70, 0), (33, 100)])
@pytest.mark.parametrize("hpw", ["1", "1w4", "2"])
def test_prefill(cuda, monkeypatch, kv, m, pos_base, hpw):
    monkeypatch.setenv("BP_PREFILL_HEADS_PER_WAVE", hpw[0])
    monkeypatch.setenv("BP_PREFILL_WG_WAVES", "4" if hpw.endswith("w4") else "8")
    _say(f"[heads] prefill n_kv_head={kv} m={m} pos_base={pos_base} heads_per_wave={hpw}")
    cfg = _cfg(kv)
    sc = Scenario(cfg, max_seq=pos_base + m + 3, m_tokens=m, seed=40 + kv + m + pos_base)
    _prefill_cache(sc, 0, pos_base, seed=50 + kv + pos_base)
    sc.oracle_q_norm_rope(pos_base)
    sc.oracle_writeback(0, pos_base)
    dev = DeviceScenario(sc, upload_kv=True)
    dev.attention(0, pos_base, is_prefill=True)
    want = sc.oracle_attention(0, pos_base, is_prefill=True)
    assert_attn_close(dev.out_f32(), want, f"prefill n_kv_head={kv} m={m} pos_base={pos_base}")


@pytest.mark.parametrize("kv", KV_HEADS)
@pytest.mark.parametrize("m,pos", [(70, 0), (33, 100)])
def test_prefill_step(cuda, kv, m, pos):
    """The fused prefill step (preparation pass over (KV head, chunk, part)
    grids of this head count): cache bytes and normalized q bit-exact,
    attention within tolerance."""
    _say(f"[heads] prefill step n_kv_head={kv} m={m} pos={pos}")
    cfg = _cfg(kv)
    sc = Scenario(cfg, max_seq=pos + m + 3, m_tokens=m, seed=60 + kv + m + pos, w_std=0.1)
    _prefill_cache(sc, 1, pos, seed=70 + kv + pos)
    dev = DeviceScenario(sc, upload_kv=True)
    dev.model.dispatch_attention_prefill_step(dev.act.data_ptr(), dev.w.data_ptr(), sc.q_off, sc.k_off,
                                              sc.v_off, sc.out_off, sc.w_q_off, sc.w_k_off, 1, pos, m)
    sc.oracle_q_norm_rope(pos)
    sc.oracle_writeback(1, pos)
    k, v = dev.kv_host()
    assert np.array_equal(k, sc.kv_k) and np.array_equal(v, sc.kv_v), "cache bytes differ"
    act = dev.act_host()
    q = slice(sc.q_off, sc.q_off + m * cfg.q_dim)
    assert np.array_equal(act[q], sc.act[q]), "normalized q differs"
    want = sc.oracle_attention(1, pos, is_prefill=True)
    assert_attn_close(dev.out_f32(), want, f"prefill step n_kv_head={kv} m={m} pos={pos}")


@pytest.mark.parametrize("kv", KV_HEADS)
def test_prefill_key_split(cuda, monkeypatch, kv):
    """The key-split 4-wave layout (grid y = splits x 4 head sets) at this head count."""
    monkeypatch.setenv("BP_PREFILL_HEADS_PER_WAVE", "1")
    monkeypatch.setenv("BP_PREFILL_WG_WAVES", "4")
    monkeypatch.setenv("BP_PREFILL_KSPLIT", "3")
    _say(f"[heads] prefill key split n_kv_head={kv}")
    cfg = _cfg(kv)
    m, pos = 40, 1500
    sc = Scenario(cfg, max_seq=pos + m + 3, m_tokens=m, seed=80 + kv)
    _prefill_cache(sc, 0, pos, seed=90 + kv)
    sc.oracle_q_norm_rope(pos)
    sc.oracle_writeback(0, pos)
    dev = DeviceScenario(sc, upload_kv=True)
    dev.attention(0, pos, is_prefill=True)
    want = sc.oracle_attention(0, pos, is_prefill=True)
    assert_attn_close(dev.out_f32(), want, f"prefill key split n_kv_head={kv}")


# Default choices that depend on the head count: the split kernel (a few tiles over 10
# to 20 chunks at 1 or 2 heads, from 24 or 8 chunks per tile at 16 or 32), the 16x16
# kernel with 4 waves and 8 (12 heads near an empty cache), prefill32_kernel with one
# tile per workgroup, with a key split, with light tiles beyond the CUs (4) and on
# pairs with an odd number of tiles and a ragged last one (12).
@pytest.mark.parametrize("kv,m,pos", [(1, 64, 800), (1, 64, 1300), (2, 100, 700), (2, 300, 900), (4, 48, 800), (4, 64, 1000), (4, 700, 900),
                                      (4, 2100, 100), (12, 24, 500), (12, 48, 800), (12, 64, 1000), (12, 128, 200), (12, 384, 30),
                                      (12, 260, 900), (12, 900, 300), (12, 740, 40), (16, 24, 300), (16, 64, 3040), (16, 64, 2900),
                                      (16, 500, 200), (32, 16, 700), (32, 33, 700), (32, 100, 2000), (32, 200, 600)])
def test_prefill_default_choices(cuda, kv, m, pos):
    _say(f"[heads] prefill choices n_kv_head={kv} m={m} pos={pos}")
    sc = Scenario(_cfg(kv), max_seq=pos + m, m_tokens=m, seed=100 + kv + m)
    _prefill_cache(sc, 0, pos, seed=110 + kv)
    sc.oracle_q_norm_rope(pos)
    sc.oracle_writeback(0, pos)
    dev = DeviceScenario(sc, upload_kv=True)
    dev.attention(0, pos, is_prefill=True)
    tokens = np.unique(np.concatenate([np.arange(0, m, 37), [t for t in (1, 15, 16, 31, 32, m - 2, m - 1) if 0 <= t < m]])).astype(int)
    want = sc.oracle_attention(0, pos, is_prefill=True, tokens=tokens)
    assert_attn_close(dev.out_f32()[tokens], want, f"prefill n_kv_head={kv} m={m} pos={pos}")
