"""Source splits of the one-sided T3 Ewald kernel, which holds a table window
in LDS: between N = 4096 and 4608 there is about one workgroup a CU.  Launches are counted on a host-memory runtime."""
import pytest

import fake_hip


@pytest.mark.parametrize("N", [4097, 4200, 4500, 4607])
@pytest.mark.parametrize("precision", [0, 1])
def test_t3_ewald_workgroups(tmp_path, N, precision):
    out = fake_hip.run(tmp_path, f"""
T = np.zeros((20, 20, 20, 3))
T[3, 4, 5, 2] = 1e-3                                # not odd: the one-sided kernel
d, keep = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=100.0, t3_table=T.reshape(-1), precision={precision})
steps.force_eval(d, *cloud({N}, 100.0))
print(launches("pair_kernel"), launches("pair_kernel", 1), launches("sym_"))
""")
    launches, blocks, sym = [int(v) for v in out[0].split()]
    assert launches == 1 and sym == 0
    assert blocks <= 18 * 15                            # row blocks x splits of 320 sources; 256 CUs
