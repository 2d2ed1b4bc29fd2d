"""Host arithmetic of the batched GEMM's workspace, on the CPU: the planes sized for passes of up to n tokens hold
those of every shorter pass (a launch checks its own against what it is given)."""
import ctypes
import random

from adaforge_amd import _native as N


def sizes():
    lib = ctypes.CDLL(N.lib()._name)
    out = []
    for name in ("_ZN2af20batch_gemm_part_needEjjjb", "_ZN2af21batch_gemm_part_bytesEjjjb"):
        f = getattr(lib, name)
        f.restype = ctypes.c_size_t
        f.argtypes = [ctypes.c_uint32] * 3 + [ctypes.c_bool]
        out.append(f)
    return out


def test_planes_of_every_pass_fit():
    need, most = sizes()
    rng = random.Random(1)
    shapes = [(9281, 222), (8192, 120), (3840, 128), (3840, 480), (15360, 120), (5120, 128), (1024, 512), (16, 1)]
    shapes += [(rng.randint(16, 17000), rng.randint(1, 512)) for _ in range(150)]
    split = 0
    for rows, blocks in shapes:
        for pair in (False, True):
            of = [need(rows, blocks, t, pair) for t in range(1, 513)]
            split += sum(n > 0 for n in of)
            for tokens in [1, 8, 9, 16, 17, 32, 33, 64, 65, 128, 129, 512] + [rng.randint(1, 512) for _ in range(4)]:
                assert max(of[:tokens]) <= most(rows, blocks, tokens, pair), (rows, blocks, tokens, pair)
    assert split > 10000  # (most of the passes do split K)
