"""CPU check of the table of register-direct transforms: the lengths 16..768 with
prime factors up to 13 have all four kernels, except those with kernels of their
own; every other length has none."""
import ctypes

import dnsproj as D

CT = (32, 64, 96, 128, 192, 256, 384, 512, 768)


def smooth(n):
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            n //= p
    return n == 1


def test_register_direct_lengths():
    ops = getattr(D.lib(), "_ZN4dnsp6rg_opsEi")
    ops.argtypes, ops.restype = [ctypes.c_int], ctypes.POINTER(ctypes.c_void_p * 4)
    for n in range(1, 1025):
        p = ops(n)
        if 16 <= n <= 768 and smooth(n) and n not in CT:
            assert p and all(p.contents[:]), n
        else:
            assert not p, n
