"""First graph decodes of new batches, one after another and from eight threads
at once: each captures on a stream taken from the shared pool.  (A decoder is
made, and a result read back, while no other thread captures: the HIP runtime
refuses work on the legacy stream during a capture.)"""
import threading

import numpy as np
import pytest

from tests.conftest import gpu_available, ribbon
from tests.test_gpu_resid import stream

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


@pytest.mark.parametrize("threads", [1, 8])
def test_first_graph_decodes(coracle, threads):
    import torch
    from meshpress_amd.batch import BatchDecoder
    datas = [stream(*ribbon(n), 12, 3) for n in (9, 130, 400)]
    refs = [coracle.decode(d) for d in datas]
    step = threading.Barrier(threads)
    done, wrong = [], []

    def turns(seed):
        side = torch.cuda.Stream()
        rng = np.random.default_rng(seed)
        for _ in range(6):
            order = rng.integers(0, 3, int(rng.integers(1, 20)))
            with torch.cuda.stream(side):
                bd = BatchDecoder([datas[i] for i in order])
                bd.d_verts.fill_(-1)
                step.wait(60)
                bd.decode("graph")
                step.wait(60)
                side.synchronize()
                v, t = bd.d_verts.cpu().numpy(), bd.d_tris.cpu().numpy()
                for (Vg, Tg), i in zip(bd.split(v, t), order):
                    if not (np.array_equal(Tg.astype(np.int64), refs[i][1])
                            and np.array_equal(Vg.view(np.uint32), refs[i][0].view(np.uint32))):
                        wrong.append((seed, int(i)))
                step.wait(60)
        done.append(seed)

    pool = [threading.Thread(target=turns, args=(s,)) for s in range(threads)]
    for x in pool:
        x.start()
    for x in pool:
        x.join()
    assert not wrong and sorted(done) == list(range(threads))
