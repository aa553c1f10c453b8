"""Where the device memory of a context comes from, as the sources have it: every allocation goes through
Workspaces::allocate, which gives the idle blocks back and tries again when the card is full (the one other
place is a call under stream capture), on the context's device."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sun_amd", "csrc")


def test_device_allocations_give_idle_blocks_back():
    found = {}
    for name in sorted(os.listdir(CSRC)):
        with open(os.path.join(CSRC, name)) as f:
            code = re.sub(r"//[^\n]*|\"[^\"\n]*\"", "", f.read())
        for m in re.finditer(r"\bhipMalloc\(", code):
            owner = re.findall(r"sun::(\w+::\w+)\([^;{}]*\{", code[: m.start()])[-1:]
            found.setdefault((name, *owner), 0)
            found[(name, *owner)] += 1
    assert found == {("sun_api.hip", "Workspaces::allocate"): 2, ("sun_api.hip", "CallScratch::take"): 1}


def test_scratch_is_taken_on_its_contexts_device():
    with open(os.path.join(CSRC, "sun_api.hip")) as f:
        body = f.read().split("hipError_t sun::CallScratch::take(size_t bytes) {")[1].split("\n}")[0]
    assert body.index("hipSetDevice(ctx_->device)") < body.index("spare.take")
