"""A signal's tables in the batched backward hold its cells' maps alone: 400 cells
leave a CU four blocks, as a small picture's do."""
import ctypes

import numpy as np

from libcpab_amd import _native as N


def test_long_tessellations_of_signals_share_the_first_class():
    dummy = (ctypes.c_int * 4)()
    insts = (N.CpabInstance * 3)()
    for I, (nc, osz) in zip(insts, [([400], [2000]), ([2, 2], [40, 40]), ([700], [500])]):
        I.tess.ndim, I.tess.nc = len(nc), N.int3(nc)
        I.tess.nC = int(np.prod(nc)) * (4 if len(nc) == 2 else 1)
        I.tess.d = 1
        I.tess.planes = I.tess.nbr = ctypes.addressof(dummy)
        I.outsize, I.nP = N.int3(osz), int(np.prod(osz))
    ptr = ctypes.cast(insts, ctypes.c_void_p)
    total = N.lib().cpab_batch_plan(ptr, 3, 2, None, 0)
    items = (ctypes.c_int * total)()
    assert N.lib().cpab_batch_plan(ptr, 3, 2, ctypes.cast(items, ctypes.c_void_p), total) == total
    assert [I.item0 for I in insts] == [0, insts[0].tiles, insts[0].tiles + insts[1].tiles]
    assert (np.frombuffer(items, dtype=np.int32)[:insts[0].tiles] == 0).all()
