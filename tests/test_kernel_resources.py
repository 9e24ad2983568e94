"""What the compiler gave the kernels of the built library: registers kept in scratch memory are a trip to memory for every use of them, in
launches that are one chain of dependent products.  Read from the metadata the compiler leaves beside its own output; no GPU involved."""
import os

import pytest

msgpack = pytest.importorskip("msgpack")
LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "deep-prove_amd", "lib", "libdpsumcheck.so")


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    data = open(LIB, "rb").read()
    found, at = {}, data.find(b"\xaeamdhsa.kernels")
    while at >= 0:
        unpacker = msgpack.Unpacker(raw=False, max_buffer_size=0)
        unpacker.feed(data[at - 1 : at + (16 << 20)])  # (a map of up to 15 entries, this key its first)
        for k in unpacker.unpack()["amdhsa.kernels"]:
            found[k[".name"]] = k
        at = data.find(b"\xaeamdhsa.kernels", at + 1)
    return found


def test_resident_sums_over_several_eq_factors_keep_their_registers(kernels):
    ours = {n: k for n, k in kernels.items() if "slice_kernel" in n and "SliceArgsEqs" in n}
    assert len(ours) == 3  # degrees 2, 3, 4
    for n, k in ours.items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, n


def test_launches_over_several_eq_factors_keep_their_registers(kernels):
    ours = {n: k for n, k in kernels.items() if "wsum" in n}
    assert ours
    for n, k in ours.items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, n
