"""rein_matvec_multi_xq8 with the activation rows staged in LDS (rein_mvl_multi_*, rein_mvql_multi_t4_m): every output against the oracle
and, bit for bit, the launch of that matrix alone -- odd heights, heights that leave workgroups or wavefronts without rows, more rows than
one round of the wavefronts, contractions in slices, formats and geometries that differ."""
import pytest

import reinstinct_amd as rein
from reinstinct_amd import hip
from reinstinct_amd._lib import init
from test_gpu_matvec_multi import check

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    init()
    hip.set_device(0)
    yield
    hip.synchronize()


# tests/test_few_row_launches.py asserts what every case launches
DOT4 = [
    ([rein.Q4_K, rein.Q4_K, rein.Q6_K], 2304, [517, 130, 65]),
    ([rein.Q8_0, rein.Q4_0], 1056, [33, 4099]),
    ([rein.Q5_K, rein.IQ4_XS, rein.IQ3_S, rein.Q8_0], 256, [1, 3, 2500, 2]),
    ([rein.Q6_K, rein.Q5_K], 512, [4097, 5003]),                    # two rows to a wavefront, or two workgroups to a CU
    ([rein.IQ3_S, rein.IQ4_XS], 256, [16001, 9003]),                # more than one round
]
MATRIX = [
    ([rein.Q5_K, rein.Q5_K], 1024, [32770, 32773], 4, None),        # several rounds of the workgroups' wavefronts
    ([rein.IQ3_S, rein.Q4_0], 1024, [40001, 26003], 3, None),
    ([rein.Q6_K, rein.Q6_K], 8192, [4099, 4097], 3, None),          # contractions in slices
    ([rein.Q8_0, rein.Q8_0], 8448, [8197, 8201], 4, None),          # three parts to a trip, the largest LDS
    ([rein.Q8_0, rein.Q6_K], 5376, [8209, 8195], 4, None),
    ([rein.Q4_K, rein.Q6_K], 5120, [13109, 9], 3, "1"),             # one in slices, the other not
]


@pytest.mark.parametrize("n_rows", [2, 3, 4])
@pytest.mark.parametrize("fmts,in_dim,out_dims", DOT4)
def test_dot4_form(fmts, in_dim, out_dims, n_rows, options):
    options.set("REIN_MV_LDS", "1")
    check(fmts, in_dim, out_dims, seed=n_rows, n_rows=n_rows, options=options)


@pytest.mark.parametrize("n_rows", [2, 4])
def test_dot4_form_where_it_is_chosen(n_rows, options):
    check([rein.Q5_K, rein.Q5_K, rein.Q6_K], 4096, [4096, 1024, 1024], seed=3, n_rows=n_rows, options=options)


@pytest.mark.parametrize("fmts,in_dim,out_dims,n_rows,pin", MATRIX)
def test_matrix_form(fmts, in_dim, out_dims, n_rows, pin, options):
    if pin:
        options.set("REIN_QUAD_LDS", pin)
    check(fmts, in_dim, out_dims, seed=5, n_rows=n_rows, one_by_one=True)
