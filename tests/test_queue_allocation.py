"""A block for a queue comes from the queue's device: where the selection of it or the allocation fails, the reason is raised (a stand-in library)."""
import ctypes

import pytest

from swiftrt_amd import native
from swiftrt_amd.platform import HipQueue


class Library:
    """The three calls behind HipQueue.allocate."""

    def __init__(self, device, memory):
        self.device, self.memory, self.calls = device, memory, []

    def srtSetDevice(self, gpu_id):
        self.calls.append(("select", gpu_id))
        return native.SUCCESS if self.device else native.ERROR_NO_DEVICE

    def srtDeviceAllocate(self, pointer, size, stream):
        self.calls.append(("allocate", size))
        ctypes.cast(pointer, ctypes.POINTER(ctypes.c_void_p))[0] = 4096 if self.memory else None
        return native.SUCCESS if self.memory else native.ERROR_OUT_OF_MEMORY

    def srtQueueAllocate(self, gpu_id, size, stream):
        return None   # as after either failure, or a shortage that has passed meanwhile

    def srtDeviceFree(self, pointer):
        return native.SUCCESS


def queue_of(library):
    queue = HipQueue.__new__(HipQueue)
    queue.device_index, queue.gpu_id, queue.lib, queue.stream = 4, 3, library, None
    return queue


def test_a_failed_selection_allocates_nothing():
    library = Library(device=False, memory=True)
    with pytest.raises(native.SrtError):
        queue_of(library).allocate(100)
    assert library.calls == [("select", 3)]


def test_a_failed_allocation_is_raised():
    library = Library(device=True, memory=False)
    with pytest.raises(native.SrtError):
        queue_of(library).allocate(100)
    assert library.calls == [("select", 3), ("allocate", 128)]


def test_the_second_try_is_on_the_queues_device():
    library = Library(device=True, memory=True)
    block = queue_of(library).allocate(100)
    assert block.pointer == 4096 and library.calls == [("select", 3), ("allocate", 128)]
