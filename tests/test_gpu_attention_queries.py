"""Eight queries a key head (two rows of four): eight waves, a launch that has to ask for its LDS, the longest partitions."""
import pytest

from test_gpu_attention import hip, run_case  # noqa: F401  (a fixture among them)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_heads,cap,position,window", [
    (1, 512, 4096, 512),      # one round of 16-token partitions
    (1, 8192, 8190, 0),       # partitions of 32 tokens, the private rows in a last one of their own
    (8, 8192, 8190, 0),       # 256 tokens and a last partition that takes the private rows as well
    (8, 64, 0, 0),            # nothing but the private rows
])
def test_eight_queries_match_the_oracle(hip, gfo, kv_heads, cap, position, window):  # noqa: F811
    run_case(hip, gfo, 2, 4 * kv_heads, kv_heads, cap, position, window, seed=position + kv_heads)
