"""Regions of act that share memory. The fused decode step gives what
q_norm_rope, kv_writeback and attention_decode give one after the other, so out
may lie over k_cur / v_cur (dead once the row is written) and over q. Where a
workgroup of the one-launch layout could store into what another still reads,
the step takes two launches; the launches are counted in a captured graph.
"""
import sys

import numpy as np
import pytest

from bonsai_pot_amd import layout
from helpers import DeviceScenario, Scenario, assert_attn_close, launches_of

pytestmark = pytest.mark.gpu

def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _scenario(pos, n_kv, seed):
    cfg = layout.Config(n_layer=2, n_head=4 * n_kv, n_kv_head=n_kv)
    sc = Scenario(cfg, max_seq=pos + 8, m_tokens=1, seed=seed, w_std=0.1)
    if pos:
        pre = Scenario(cfg, sc.max_seq, pos, seed=seed + 1, with_q=False)
        pre.oracle_writeback(1, 0)
        sc.kv_k[:], sc.kv_v[:] = pre.kv_k, pre.kv_v
    return sc


# act is q | k | v | out; out moved to the named place (element offsets), and the
# launches of the step at up to 320 rows
PLACES = {"apart": (lambda sc: sc.out_off, 1), "q": (lambda sc: sc.q_off, 1), "k": (lambda sc: sc.k_off, 2),
          "v": (lambda sc: sc.v_off, 2), "end of v": (lambda sc: sc.v_off + sc.cfg.kv_dim - 4, 2)}


@pytest.mark.parametrize("place", sorted(PLACES))
@pytest.mark.parametrize("pos,n_kv", [(0, 8), (100, 8), (300, 12), (320, 1), (321, 8)])
def test_decode_step_out_over_inputs(cuda, place, pos, n_kv):
    _say(f"[overlap] decode step out over {place} pos={pos} n_kv_head={n_kv}")
    at, launches = PLACES[place]
    sc = _scenario(pos, n_kv, seed=1500 + pos)
    sc.out_off = at(sc)
    dev = DeviceScenario(sc, upload_kv=True)
    assert launches_of(dev.model, lambda: dev.decode_step(1, pos)) == (launches if pos <= 320 else 2)
    dev.decode_step(1, pos)
    sc.oracle_q_norm_rope(pos)
    sc.oracle_writeback(1, pos)
    _, want = sc.oracle_decode(1, pos)
    k, v = dev.kv_host()
    assert np.array_equal(k, sc.kv_k) and np.array_equal(v, sc.kv_v), "cache bytes differ"
    assert_attn_close(dev.out_f32(1)[0], want, f"decode step, out over {place}, pos={pos}")
    rest = np.ones(sc.act.size, bool)
    rest[sc.out_off:sc.out_off + sc.cfg.q_dim] = False
    assert np.array_equal(dev.act_host()[rest], sc.act[rest]), "act beside out differs"


@pytest.mark.parametrize("shift,launches", [(0, 1), (512, 2), (4, 2), (4096, 1)])
@pytest.mark.parametrize("pos", [100, 127, 128, 300])
def test_decode_out_over_q(cuda, shift, launches, pos):
    """The plain decode with out on q itself, across other heads' q, behind q."""
    _say(f"[overlap] decode out over q + {shift} pos={pos}")
    sc = _scenario(pos + 1, 8, seed=1600 + pos)
    sc.out_off = sc.q_off + shift
    dev = DeviceScenario(sc, upload_kv=True)
    assert launches_of(dev.model, lambda: dev.decode(1, pos)) == launches
    dev.decode(1, pos)
    _, want = sc.oracle_decode(1, pos)
    assert_attn_close(dev.out_f32(1)[0], want, f"decode, out over q + {shift}, pos={pos}")


@pytest.mark.parametrize("shift,launches", [(0, 2), (512, 3), (8, 3)])
@pytest.mark.parametrize("m,pos", [(64, 448), (64, 576), (48, 500), (32, 288)])
def test_prefill_step_out_over_q(cuda, m, pos, shift, launches):
    """A short chunk over 4 to 11 key chunks per tile: out on q itself, and across
    other heads' q, where the merge pass has to store it."""
    _say(f"[overlap] prefill step out over q + {shift} m={m} pos={pos}")
    cfg = layout.Config(n_layer=2)
    sc = Scenario(cfg, max_seq=pos + m, m_tokens=m, seed=1700 + m + pos, w_std=0.1)
    pre = Scenario(cfg, sc.max_seq, pos, seed=1701, with_q=False)
    pre.oracle_writeback(1, 0)
    sc.kv_k[:], sc.kv_v[:] = pre.kv_k, pre.kv_v
    sc.out_off = sc.q_off + shift
    if shift:   # out of the last token reaches into k, which the preparation pass has read by then
        assert sc.out_off + m * cfg.q_dim <= sc.v_off
    dev = DeviceScenario(sc, upload_kv=True)

    def step():
        dev.model.dispatch_attention_prefill_step(dev.act.data_ptr(), dev.w.data_ptr(), sc.q_off, sc.k_off, sc.v_off,
                                                  sc.out_off, sc.w_q_off, sc.w_k_off, 1, pos, m)
    assert launches_of(dev.model, step) == launches
    step()
    sc.oracle_q_norm_rope(pos)
    sc.oracle_writeback(1, pos)
    k, v = dev.kv_host()
    assert np.array_equal(k, sc.kv_k) and np.array_equal(v, sc.kv_v), "cache bytes differ"
    assert_attn_close(dev.out_f32(), sc.oracle_attention(1, pos), f"prefill step, out over q + {shift}, m={m} pos={pos}")
