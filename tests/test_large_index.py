"""Index expressions of the geometry kernels at the largest sizes they accept,
evaluated on the host (such a layout takes about 50 GB of tables)."""
from tests._host_cpp import run_host_cpp

LARGEST = 2 ** 31 - 1  # rows of a radius-0 layout


def test_coordinate_rows_beyond_a_third_of_the_32_bit_range(tmp_path):
    """The rows are 32-bit in the kernel; their entries of the coordinate table are not."""
    rows = [0, 1, 715827882, 715827883, 1024 ** 3 - 1, LARGEST - 1]
    body = "".join(f'{{ const int32_t row = {r}; printf("%lld\\n", (long long)p3d::coord_start(row)); }}\n' for r in rows)
    assert [int(v) for v in run_host_cpp(tmp_path, ["index.hpp"], body)] == [3 * r for r in rows]
