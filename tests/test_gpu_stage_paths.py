"""begin_step's two table scans and their edges against the oracle (bit for bit, as
test_gpu_stage.py compares them): the widest batches that one workgroup scans itself (8190
table entries over 3 requests; 128 requests) and the first that get the mark launch (8193;
129), and wide ones; more flush candidates in one step than a workgroup
holds threads, with the flush list filling up in the middle and blocks shared by requests;
more tokens in a step than the allocating workgroup maps; the invalidation in the collect's launch (a pair of requests and layers
past a multiple of four) and before the mark's."""
import numpy as np
import pytest
import torch

from amass import _hip
from helpers import announce
from test_gpu_stage import _Scenario, _schedule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("MP", [2730, 2731, 5461, 5600])
def test_table_scans(MP):
    announce(f"write path, {3 * MP} table entries")
    sc = _Scenario(seed=MP, NV=24, maxf=2, shared=True, MP=MP, NB=3 * MP + 5)
    for ql in _schedule(12, True):
        sc.step(ql)
    sc.stg.assert_free_partition()


@pytest.mark.parametrize("R", [127, 128, 129])
def test_many_requests(R):
    announce(f"write path, {R} requests")
    MP, rng = 6, np.random.default_rng(R)
    NB = R * MP + 3
    sc = _Scenario(seed=R, NV=3 * R, maxf=R, shared=True, MP=MP, NB=NB, R=R, max_tokens=8 * R)
    rest = rng.permutation(np.setdiff1d(np.arange(NB), sc.bt))[:(R - 3) * MP]
    sc.bt = np.concatenate([sc.bt, rest.reshape(R - 3, MP)])
    sc.bt_d = torch.tensor(sc.bt, dtype=torch.int32, device="cuda")
    for _ in range(5):
        sc.step(rng.integers(0, 6, R) * (sc.sl < 4 * MP - 6))
    sc.stg.assert_free_partition()


@pytest.mark.parametrize("maxf", [1500, 4000])
@pytest.mark.parametrize("shared", [False, True])
def test_many_candidates(maxf, shared):
    announce(f"write path, 3600 candidates in a step, flush list of {maxf}, shared {shared}")
    sc = _Scenario(seed=maxf, NV=3800, maxf=maxf, shared=shared, MP=1300, NB=3950,
                   max_tokens=15000)
    sc.step([4800, 4790, 4777])
    for _ in range(4):
        sc.step([1, 1, 1])
    sc.step([0, 3, 1])
    sc.stg.assert_free_partition()


def test_many_tokens():
    announce("write path, 17000 tokens in a step")
    sc = _Scenario(seed=3, NV=4400, maxf=4400, shared=False, MP=1600, NB=4850, max_tokens=17000)
    sc.step([6000, 5999, 5001])
    sc.step([1, 1, 1])
    sc.stg.assert_free_partition()


@pytest.mark.parametrize("MP", [40, 5600])
@pytest.mark.parametrize("shared", [False, True])
def test_invalidation_in_the_same_call(MP, shared):
    announce(f"write path with its invalidation, {3 * MP} table entries, shared {shared}")
    sc = _Scenario(seed=MP + 1, NV=24, maxf=3, shared=shared, MP=MP, NB=3 * MP + 5)
    stream = _hip.current_stream(sc.bt_d.device)

    def step(bt, sl, qsl, n_tok, pool, pool_valid):
        _hip.begin_step(sc.res.invalidate_args(bt, sl, qsl),
                        sc.stg.step_args(bt, sl, qsl, n_tok, pool, pool_valid), stream)

    sc.res.invalidate_written = lambda *rows: None
    sc.stg.begin_step = step
    for ql in _schedule(12, True):
        sc.step(ql)
    sc.stg.assert_free_partition()
