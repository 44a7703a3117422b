"""What kivi.cache_prefill refuses before any launch (host checks only: the
kernel writes all its outputs by the extents of k_rows and chunk_min)."""
import pytest
import torch

from zoomkv_revision_amd import kivi
from zoomkv_revision_amd._lib import ZkvError

BS, KV, ROWS, CHUNKS, CHUNK = 2, 3, 96, 4, 16


def _args(**changed):
    mk = lambda *s: torch.zeros(BS, KV, *s, dtype=torch.bfloat16)
    a = dict(keys=mk(80, 128), values=mk(80, 128), sink=8, local=8, k_rows=mk(ROWS, 128), v_rows=mk(ROWS, 128),
             sink_row=64, ret_row=0, local_row=72, chunk_size=CHUNK, chunk_min=mk(CHUNKS, 128),
             chunk_max=mk(CHUNKS, 128), chunk_centroid=mk(CHUNKS, 128),
             chunk_valid=torch.zeros(BS, KV, CHUNKS, dtype=torch.bool),
             packed_K=torch.zeros(BS, KV, CHUNKS, 16, CHUNK, dtype=torch.int32))
    a.update(changed)
    return a


@pytest.mark.parametrize("name,bad", [
    ("v_rows", lambda t: t[:, :, :ROWS - 1]),                   # fewer rows at k_rows' strides
    ("v_rows", lambda t: t[:, :, :ROWS // 2].contiguous()),
    ("k_rows", lambda t: t[:1]),
    ("chunk_min", lambda t: t[:, :2].contiguous()),
    ("chunk_max", lambda t: t[:, :, :CHUNKS - 1].contiguous()),
    ("chunk_max", lambda t: t[..., :64].contiguous()),
    ("chunk_centroid", lambda t: t[:1].contiguous()),
    ("chunk_centroid", lambda t: t.transpose(0, 1).contiguous().transpose(0, 1)),
    ("chunk_valid", lambda t: t[:, :, :CHUNKS - 1].contiguous()),
    ("chunk_valid", lambda t: t.repeat(1, 1, 2)[:, :, ::2]),   # every other byte
    ("packed_K", lambda t: t[:, :, :CHUNKS - 1].contiguous()),
])
def test_buffers_the_kernel_would_leave_are_refused(name, bad):
    with pytest.raises(ValueError, match=name):
        kivi.cache_prefill(**_args(**{name: bad(_args()[name])}))


@pytest.mark.parametrize("name", ["k_rows", "v_rows", "chunk_min", "chunk_max", "chunk_centroid", "chunk_valid",
                                  "packed_K"])
def test_other_dtypes_are_refused(name):
    with pytest.raises(TypeError, match=name):
        kivi.cache_prefill(**_args(**{name: _args()[name].to(torch.float64)}))


def test_matching_buffers_pass_the_host_checks():
    """... up to the one that they are on the GPU."""
    with pytest.raises(ZkvError, match="device tensors"):
        kivi.cache_prefill(**_args())


class _Rows:
    """A [2, 3, 80, 128] tensor's layout on some device."""
    dtype, is_cuda, shape = torch.bfloat16, True, (2, 3, 80, 128)

    def __init__(self, index, ptr=4096):
        self.device, self._ptr = torch.device("cuda", index), ptr

    def stride(self, dim=None):
        s = (80 * 3 * 128, 128, 3 * 128, 1)
        return s if dim is None else s[dim]

    def data_ptr(self):
        return self._ptr


def test_rows_of_two_devices_are_not_taken_in_place():
    """polar_cache copies such a prompt piece by piece: a kernel of one device
    cannot read the other's memory."""
    assert kivi.cache_prefill_takes(_Rows(0), _Rows(0))
    assert not kivi.cache_prefill_takes(_Rows(0), _Rows(0, ptr=4098))
    assert not kivi.cache_prefill_takes(_Rows(0), _Rows(1))
