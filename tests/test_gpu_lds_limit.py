"""Cells of different sizes through the kernels that use more LDS than every kernel may
have, at the same time from several host threads: the limit they raise is an attribute of
the function, shared by all threads."""
import ctypes as ct
import threading

import numpy as np
import pytest

from camellia2_amd import capi, dpg

from helpers import poisson2d

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


class FuncAttributes(ct.Structure):  # hipFuncAttributes
    _fields_ = [("binaryVersion", ct.c_int), ("constSizeBytes", ct.c_size_t), ("localSizeBytes", ct.c_size_t),
                ("maxDynamicSharedSizeBytes", ct.c_int), ("maxThreadsPerBlock", ct.c_int), ("numRegs", ct.c_int),
                ("preferredShmemCarveout", ct.c_int), ("ptxVersion", ct.c_int), ("sharedSizeBytes", ct.c_size_t)]


def lds_limit(kernel):
    hip, own = ct.CDLL("libamdhip64.so"), ct.CDLL(capi.lib()._name)
    attr = FuncAttributes()
    at = ct.addressof(ct.c_char.in_dll(own, kernel))
    hip.hipFuncGetAttributes.argtypes = [ct.POINTER(FuncAttributes), ct.c_void_p]
    assert hip.hipFuncGetAttributes(ct.byref(attr), at) == 0
    return attr.maxDynamicSharedSizeBytes


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def cells(k, kt, n):
    f, b, nodes, par, _, load = poisson2d(n, n, k=k, kt=kt)
    return dpg.LocalAssembler(f, [b]), dev(nodes), dev(par), load


def test_a_small_launch_does_not_lower_the_limit():
    large, small = cells(3, 6, 2), cells(3, 4, 2)  # 190 and 122 rows: 161 and 75 KB
    for A, nodes, par, load in (large, small):
        assert A.local_stiffness_and_rhs(0, nodes, par, None, load, want_schur=True)[1] == 0
    got = lds_limit("_ZN3dpg18cell_factor_kernelENS_14CellFactorArgsE")
    print("limit", got)
    assert got >= 161280


def test_threads_with_cells_of_different_sizes():
    kinds = [cells(3, 6, 3), cells(3, 4, 3), cells(4, 6, 3), cells(6, 8, 3)]  # 161 and 75 KB; panels of 128, fields of 58 KB
    def call(A, nodes, par, load, stream):
        out, bad = A.local_stiffness_and_rhs(0, nodes, par, None, load, want_schur=True, stream=stream)
        u = torch.ones((nodes.shape[0], out["K"].shape[1]), dtype=torch.float64, device="cuda:0")
        stream.synchronize()
        bad += A.recover_fields(0, out["K"], out["rhs"], u, stream=stream)
        stream.synchronize()
        return bad, out["K"], out["schur"], u
    streams = [torch.cuda.Stream() for _ in kinds]
    torch.cuda.synchronize()
    ref = [call(*k, s) for k, s in zip(kinds, streams)]
    errors = []

    def work(i):
        try:
            with torch.cuda.stream(streams[i]):
                for _ in range(40):
                    got = call(*kinds[i], streams[i])
                    assert got[0] == 0 and all(torch.equal(a, b) for a, b in zip(got[1:], ref[i][1:]))
        except BaseException as e:
            errors.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(kinds))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
