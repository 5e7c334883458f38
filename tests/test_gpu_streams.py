"""stream_handle gives the stream that torch calls current, whichever way it was made current."""
import threading

import pytest

pytestmark = pytest.mark.gpu


def test_stream_handle_is_the_current_stream(gpu):
    import torch

    from fusor_kernels._lib import stream_handle

    def handles():
        return stream_handle().value or 0, torch.cuda.current_stream().cuda_stream

    seen = [handles()]
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        seen.append(handles())
        assert (stream_handle(torch.cuda.default_stream()).value or 0) == torch.cuda.default_stream().cuda_stream
    seen.append(handles())
    torch.cuda.set_stream(side)
    worker = threading.Thread(target=lambda: seen.append(handles()))  # a thread has a current stream of its own
    worker.start()
    worker.join()
    seen.append(handles())
    torch.cuda.set_stream(torch.cuda.default_stream())
    assert all(got == want for got, want in seen) and seen[1][0] == side.cuda_stream == seen[4][0] != seen[3][0]
