"""Device-memory plumbing: numpy <-> torch device tensors, workspaces, streams.

torch only provides memory and streams here; every computation is a libhalma call.
"""
import numpy as np
import torch

from . import _lib


def device():
    if not torch.cuda.is_available():
        raise RuntimeError("pyhalma_amd needs a ROCm GPU (torch.cuda.is_available() is False)")
    return torch.device("cuda", torch.cuda.current_device())


def stream_ptr(stream=None):
    s = stream if stream is not None else torch.cuda.current_stream()
    return int(s.cuda_stream)


def ptr(t):
    """Device pointer of a tensor (None -> NULL)."""
    if t is None:
        return None
    return int(t.data_ptr())


def to_dev(a, dtype=None):
    """numpy array (or tensor) -> contiguous device tensor of the given numpy dtype."""
    if isinstance(a, torch.Tensor):
        t = a
        if dtype is not None:
            t = t.to(dtype=_torch_dtype(dtype))
        return t.to(device()).contiguous()
    arr = np.asarray(a)
    if dtype is not None:
        arr = arr.astype(dtype, copy=False)
    arr = np.ascontiguousarray(arr)
    return torch.from_numpy(arr).to(device(), non_blocking=False)


# Host arrays of one call go up together up to this many bytes: a small copy costs its call and
# its wait, a large one its bytes, which packing reads and writes once more (seven arrays of
# 4 kB 125 us each for itself, 64 us packed; 1 MB in all 121 and 101; 2.8 MB 181 and 186).
PACK_BYTES = 1 << 20


def to_dev_all(arrays, dtype=None):
    """to_dev of several arrays: the host ones, up to PACK_BYTES in all, go up in one transfer
    (the tensors returned for them share one allocation)."""
    out = [None] * len(arrays)
    host, total = [], 0
    for k, a in enumerate(arrays):
        if not isinstance(a, torch.Tensor):
            arr = np.asarray(a)
            if dtype is not None:
                arr = arr.astype(dtype, copy=False)
            a = torch.from_numpy(np.ascontiguousarray(arr))
            if 0 < a.numel() and total + a.numel() * a.element_size() <= PACK_BYTES:
                host.append((k, a, total))
                total += -(-a.numel() * a.element_size() // 256) * 256
                continue
        out[k] = to_dev(a, dtype)
    if len(host) == 1:
        out[host[0][0]] = host[0][1].to(device(), non_blocking=False)
    elif host:
        buf = np.empty(total, np.uint8)
        for _, a, at in host:
            raw = a.numpy().reshape(-1).view(np.uint8)
            buf[at:at + raw.size] = raw
        buf = torch.from_numpy(buf).to(device(), non_blocking=False)
        for k, a, at in host:
            nb = a.numel() * a.element_size()
            out[k] = buf[at:at + nb].view(a.dtype).view(a.shape)
    return out


def _torch_dtype(npdtype):
    return {np.dtype(np.float32): torch.float32, np.dtype(np.float64): torch.float64,
            np.dtype(np.int32): torch.int32, np.dtype(np.int64): torch.int64,
            np.dtype(np.uint8): torch.uint8}[np.dtype(npdtype)]


def empty(n, npdtype):
    return torch.empty(int(n), dtype=_torch_dtype(npdtype), device=device())


def workspace(nbytes):
    """Caller-owned workspace for a libhalma call (at least 256 bytes)."""
    return torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=device())


def dtype_flag(t):
    if t.dtype == torch.float32:
        return _lib.F32
    if t.dtype == torch.float64:
        return _lib.F64
    raise TypeError(f"unsupported dtype {t.dtype} (float32 or float64)")


def float_tensor(a):
    """Device tensor keeping float32/float64 as given; other dtypes become float64
    (numpy's promotion of integer coordinates)."""
    if isinstance(a, torch.Tensor):
        t = a.to(device())
    else:
        arr = np.asarray(a)
        if arr.dtype not in (np.float32, np.float64):
            arr = arr.astype(np.float64)
        t = torch.from_numpy(np.ascontiguousarray(arr)).to(device())
    if t.dtype not in (torch.float32, torch.float64):
        t = t.to(torch.float64)
    return t.contiguous()
