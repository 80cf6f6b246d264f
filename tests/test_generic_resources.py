"""The generic kernel of compositions without fweno_t is built without its
unrolled arrays (CPU test, on the library's own code objects): their spilled
registers made every other composition slower."""
from test_kernel_resources import _code_objects, _kernels


def test_fweno_costs_the_others_no_scratch(tmp_path):
    found = {}
    for obj in _code_objects(tmp_path):
        for k in _kernels(obj):
            if "k_flux_div_generic" in k["name"]:
                found["Lb1" in k["name"]] = int(k["private_segment_fixed_size"])
    print(found)
    assert set(found) == {False, True}
    assert found[False] <= 256 < found[True]
