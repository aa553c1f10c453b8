"""Where the device memory of a context comes from, as the sources have it."""
import os

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sun_amd", "csrc")


def test_scratch_is_taken_on_its_contexts_device():
    with open(os.path.join(CSRC, "sun_api.hip")) as f:
        body = f.read().split("hipError_t sun::CallScratch::take(size_t bytes) {")[1].split("\n}")[0]
    assert body.index("hipSetDevice(ctx_->device)") < body.index("spare.take")
