"""GPU tests of recorded steps (step_tokens) of one token a session, which run as graphs from the second step of as many rows on: the same bits as launch by launch, over prompts,
other numbers of rows, sessions that close and open, and steps that want other rows in between; contexts grow over the ends of cache blocks.  A step that is refused leaves no
trace."""
import numpy as np
import pytest

from lmdeploy_amd import _ffi
from tests.gpu_helpers import release_all
from tests import test_gpu_bedenex, test_gpu_febivik, test_gpu_layered, test_gpu_mededra, test_gpu_roravik
from tests.test_gpu_sanozen import engine as sanozen_engine
from tests.test_gpu_sanozen import full_model as sanozen_model
from tests.test_gpu_sanozen import model_folder as sanozen_folder

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


def _walk(eng, vocab):
    """every logits row that a fixed course of sessions gives"""
    rng, out = np.random.default_rng(3), []

    def step(entries):
        out.append(eng.step_tokens(entries).copy())

    def one(sessions, want=True):
        step([(s, rng.integers(0, vocab, 1), [0] if want else []) for s in sessions])
    a, b, c = (eng.open_session() for _ in range(3))
    step([(a, rng.integers(0, vocab, 60), [59]), (b, rng.integers(0, vocab, 61), [3, 60]), (c, rng.integers(0, vocab, 7), [])])
    for i in range(8):
        one((a, b, c))
        if i == 4:
            d = eng.open_session()
            step([(d, rng.integers(0, vocab, 30), [29]), (a, rng.integers(0, vocab, 1), [0])])      # a portion beside a decoded token
    for i in range(5):
        one((b, d) if i % 2 else (d, a, b, c), i != 2)
    step([(a, rng.integers(0, vocab, 1), [0]), (c, rng.integers(0, vocab, 1), [])])                     # one of two rows wanted
    eng.close_session(b)
    e = eng.open_session()
    step([(e, rng.integers(0, vocab, 5), [4])])
    for _ in range(4):
        one((e, c, a))
        one((a, ))
    for s in (a, c, d, e):
        eng.close_session(s)
    return out


def _fokonex(tmp_path, dtype):
    cfg, w = test_gpu_layered.small_model(2)
    return cfg['vocab'], lambda **kw: test_gpu_layered.engine_for(cfg, w, dtype, **kw)


def _of(module, cfg):
    def build(tmp_path, dtype):
        c = cfg(dtype)
        folder = module.model_folder(tmp_path, c, 2)[0]
        return c['vocab'], lambda **kw: module.engine(folder, dtype, **kw)
    return build


def _sanozen(tmp_path, dtype):
    folder, _ = sanozen_folder(tmp_path, sanozen_model(), 2)
    return sanozen_model()['vocab'], lambda **kw: sanozen_engine(folder, dtype, **kw)


FAMILIES = {'fokonex': _fokonex, 'bedenex': _of(test_gpu_bedenex, test_gpu_bedenex.looped_model), 'febivik': _of(test_gpu_febivik, test_gpu_febivik.full_model),
            'mededra': _of(test_gpu_mededra, lambda dtype: test_gpu_mededra.full_model()), 'sanozen': _sanozen,
            'roravik': _of(test_gpu_roravik, lambda dtype: test_gpu_roravik.full_model())}


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('family', FAMILIES)
def test_graphs_give_the_bits_of_launches(tmp_path, cuda, family, dtype):
    vocab, build = FAMILIES[family](tmp_path, dtype)
    rows = []
    for graphs in (0, 1):
        eng = build(use_graph=graphs)
        rows.append(_walk(eng, vocab))
        rows.append(_walk(eng, vocab))      # with the graphs of the first course
        eng.close()
    for other in rows[1:]:
        assert len(other) == len(rows[0]) and all(np.array_equal(x.view(np.uint32), y.view(np.uint32)) for x, y in zip(rows[0], other))
    assert all(np.isfinite(x).all() for x in rows[0]) and not np.array_equal(rows[0][1], rows[0][2])


def test_as_many_graphs_as_numbers_of_rows(tmp_path, cuda):
    """sessions that pause and go on: 20 numbers of rows, with and without logits, three times round, against launch by launch"""
    cfg = sanozen_model()
    folder, _ = sanozen_folder(tmp_path, cfg, 6)
    rows = []
    for graphs in (0, 1):
        eng = sanozen_engine(folder, 'float32', use_graph=graphs, max_batch_size=20, cache_blocks=60)
        rng = np.random.default_rng(8)
        sess, out = [eng.open_session() for _ in range(20)], []
        eng.step_tokens([(s, rng.integers(0, cfg['vocab'], 3 + i), []) for i, s in enumerate(sess)])
        for _ in range(3):
            for n in range(20, 0, -1):
                for want in ([0], []):
                    out.append(eng.step_tokens([(s, rng.integers(0, cfg['vocab'], 1), want) for s in sess[:n]]).copy())
        rows.append(np.concatenate(out))
        eng.close()
    assert np.array_equal(rows[0].view(np.uint32), rows[1].view(np.uint32)) and np.isfinite(rows[0]).all()


@pytest.mark.parametrize('graphs', [0, 1])
@pytest.mark.parametrize('n', [1, 2, 70])
def test_a_refused_step_leaves_its_sessions_as_they_were(tmp_path, cuda, n, graphs):
    """logits are wanted and there is no place for them: the next step has the logits of a session that never saw the refusal (keys, values and states included)"""
    cfg = sanozen_model()
    folder, _ = sanozen_folder(tmp_path, cfg, 4)
    eng = sanozen_engine(folder, 'float32', use_graph=graphs)
    rng = np.random.default_rng(n)
    first, other = rng.integers(0, cfg['vocab'], (2, 20)).astype(np.int32)
    refused, then = rng.integers(0, cfg['vocab'], (2, n)).astype(np.int32)
    want = np.array([n - 1], np.int32)
    out = []
    for refuse in (False, True, False, True):
        a, b = eng.open_session(), eng.open_session()
        eng.step_tokens([(a, first, []), (b, other, [])])
        if refuse:
            entries = (_ffi.StepEntry * 2)(_ffi.StepEntry(b, other.ctypes.data, 1, None, 0), _ffi.StepEntry(a, refused.ctypes.data, n, want.ctypes.data, 1))
            assert eng._lib.tm_engine_step_tokens(eng._h, entries, 2, None) == 1      # TM_INVALID
        out.append(np.concatenate([eng.step_tokens([(a, then, [n - 1]), (b, other[:1], [0])]) for _ in range(3)]))
        eng.close_session(a)
        eng.close_session(b)
    eng.close()
    assert all(np.array_equal(out[0].view(np.uint32), o.view(np.uint32)) for o in out[1:])
