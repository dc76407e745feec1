"""Device memory that a plain domain holds, and its give-back."""
import pytest

pytestmark = pytest.mark.gpu


def test_plain_domain_bytes_per_cell(amca):
    """256^3: per slot (1.048 per cell with the ghost layer's bricks) 98.4 bytes, per cell
    41 and per ghosted cell (1.024) 8, 152.3 bytes a cell in all; two lists of their own
    would be 12 more.  Closing gives all of it back."""
    import ctypes as C

    from amca3d_amd._lib import load
    info = load().hipMemGetInfo  # of the runtime that the library is linked to
    info.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]

    def free():
        f, t = C.c_size_t(0), C.c_size_t(0)
        assert info(C.byref(f), C.byref(t)) == 0
        return f.value

    def make():
        return amca.OwnedDomain(nx=256, ny=256, nz=256, h=2e-6, orient_capacity=100)

    make().close()  # the library's own set-up
    free0 = free()
    d = make()
    used = free0 - free()
    d.close()
    n = 256 ** 3
    # the allocator gives whole 32 MB (315 of 128^3 came as 320), here 2 bytes a cell
    assert 150 * n < used < 152.5 * n + (32 << 20)
    assert free() >= free0 - (32 << 20)
