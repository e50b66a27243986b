"""What one stream makes and every other may take."""
import torch


def settled(device: torch.device) -> bool:
    """Asked before something is kept for later calls that the current stream was just given to make (a copy of weights in
    another order, stacked weights): True once it is made, so that a call on any stream may read it.  False under capture:
    nothing is made there before a replay, and the memory is the graph's own; the caller then keeps nothing."""
    if device.type != "cuda":
        return True
    with torch.cuda.device(device):
        if torch.cuda.is_current_stream_capturing():
            return False
        torch.cuda.current_stream().synchronize()
    return True
