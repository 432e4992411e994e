"""Products of 33 to 64 tokens around the last block of 16 tokens, which is formed and stored only where there are tokens in it: the bits of results that
leave one by one, and nothing written beyond them."""

import pytest

from tests import test_stream_rows_gpu as rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [34, 47, 48, 49, 63])
@pytest.mark.parametrize("m, k, form", [(200, 136, "float32"), (1032, 520, "bfloat16"), (200, 136, "gated"), (516, 2056, "shares"), (20004, 72, "float32")])
def test_the_last_block_of_tokens(m, k, form, n):
    rows.test_rows_leave_whole(n=n, m=m, k=k, form=form)
