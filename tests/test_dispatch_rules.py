"""Which form of a kernel a call takes: rules of sizes alone, on the host."""

from __future__ import annotations

import pytest

from quickstart_streaming_agents_amd.ops import ext, have_ext

pytestmark = pytest.mark.skipif(not have_ext(), reason="extension not built")


@pytest.mark.parametrize("pages", [0, 1, 16, 17, 40])
def test_decode_attention_of_no_rows(pages):
    """A batch without rows has no blocks to share its pages."""
    assert ext().paged_attn_split(0, 32, 8, pages, 128)[1] == 1
