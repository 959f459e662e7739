"""GPU tests of the tiles that experts of long prompts take: whole rounds of 256 x 256 tiles with the columns behind them in a launch of their own, more experts than the
wave that counts their row tiles has lanes, experts without rows -- the logits of a one-layer model against the float64 oracle, the same bound as its other tests.
Rows whose second and third expert are nearly tied are left out: a router's score is a sum of products of numbers rounded to bf16 (2^-9 of each, size one in all), so scores
within 0.05 may change places, and with them the experts."""
import numpy as np
import pytest

from tests import febivik_oracle as fo
from tests.test_gpu_febivik import TOL, engine

pytestmark = pytest.mark.gpu


def _moe_ff(h, f, w, p, gaps):
    """fo.moe_ff, an expert's rows at a time"""
    z = np.sort(h @ w[p + 'router'].T, axis=1)
    gaps.append(z[:, -2] - z[:, -3])
    idx, sc = fo.route(h, w[p + 'router'], int(f['router']['top']))
    idx, sc = np.asarray(idx), np.asarray(sc)
    out = np.zeros((h.shape[0], w[p + 'e0.down'].shape[0]))
    for e in range(int(f['router']['experts'])):
        t, k = np.nonzero(idx == e)
        if len(t):
            out[t] += float(f['router'].get('scale', 1.0)) * sc[t, k][:, None] * fo.relu2_expert(h[t], w, p + f'e{e}.')
    return out + fo.relu2_expert(h, w, p + 'shared.') if f.get('shared') else out


# tokens a sequence, experts, width, their inner size: 16530 rows of nine experts (2560 of 2816 columns in three rounds of large tiles), 71 of which a few have rows,
# 130 of which none has many
@pytest.mark.parametrize('lens,experts,width,ff,same', [([551] * 10, 8, 512, 2816, False), ([200], 70, 64, 40, True), ([70, 130], 129, 64, 72, False)])
@pytest.mark.parametrize('dtype', ['bfloat16', 'float32'])
def test_tiles_of_experts(tmp_path, cuda, monkeypatch, lens, experts, width, ff, same, dtype):
    if ff > 1000 and dtype == 'float32':
        pytest.skip('two launches are for 16-bit products')
    cfg = fo.make_config(width, 97, [fo.lightning_layer(2, 8, 8, [0.9, 0.9], fo.moe(experts, 2, ff, 1.0, ff))])
    w = fo.random_weights(cfg, experts)
    folder = str(tmp_path / 'm')
    fo.write_checkpoint(folder, cfg, w)
    rng = np.random.default_rng(experts)
    reqs = [[5] * n if same else rng.integers(0, 97, n).tolist() for n in lens]
    eng = engine(folder, dtype, max_batch_size=len(lens), cache_blocks=sum(n // 64 + 2 for n in lens), session_len=1024, max_prefill_token_num=8192)
    sess = [eng.open_session() for _ in reqs]
    got = eng.step_tokens([(s, r, list(range(len(r)))) for s, r in zip(sess, reqs)]).reshape(sum(lens), -1)
    gaps = []
    monkeypatch.setattr(fo, 'moe_ff', lambda *a: _moe_ff(*a, gaps))
    ref = np.concatenate([fo.forward(cfg, w, r) for r in reqs])
    clear = np.concatenate(gaps) > 0.05
    assert clear.mean() > 0.5 and np.abs(got - ref)[clear].max() <= TOL[dtype] * np.abs(ref).max()
    eng.close()
