"""Small shared helpers for the tests (no test logic)."""
import numpy as np


def rel_l2(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    den = np.linalg.norm(b)
    return float(np.linalg.norm(a - b) / (den if den > 0 else 1.0))


def circle_panels(npan, diam=1.0, cx=0.0, cy=0.0, external=True):
    """Node layout of SolidCircle::init_elements (src/BoundaryFeature.cpp:489-530): clockwise
    from theta = 0, nodes rounded to float as the reference stores them."""
    i = np.arange(npan, dtype=np.float32)
    th = 2.0 * np.pi * i.astype(np.float64) / np.float64(np.float32(npan))
    nx = (cx + 0.5 * diam * np.cos(th)).astype(np.float32)
    ny = (cy - 0.5 * diam * np.sin(th)).astype(np.float32)
    idx = np.stack([np.arange(npan), (np.arange(npan) + 1) % npan], 1).astype(np.uint32)
    if not external:
        idx = idx[:, ::-1].copy()
    return nx, ny, idx.ravel()


def particles(rng, n, lo=-1.0, hi=1.0, rad=(0.01, 0.05), smean=0.0, sstd=1.0):
    x = rng.uniform(lo, hi, n)
    y = rng.uniform(lo, hi, n)
    s = rng.normal(smean, sstd, n)
    r = rng.uniform(rad[0], rad[1], n)
    return x, y, s, r


def pair_sum(src, tgt, tr=None, core="gauss", most=262144):
    """The fp64 velocity of device tensors src = (x, y, s, r) at tgt = (x, y), pair by pair: the
    no-allocation entry never takes clusters, and adds `most` sources and targets at a time."""
    import ctypes

    import torch

    from omega2d_amd import _cabi
    from omega2d_amd.device import env_for
    u, v = (torch.zeros(tgt[0].numel(), dtype=torch.float64, device="cuda") for _ in range(2))
    env = env_for(u.device, core, "fp64", "vel")
    p = lambda a: None if a is None else ctypes.c_void_p(a.data_ptr())  # noqa: E731
    for i in range(0, u.numel(), most):
        cut = slice(i, i + most)
        t = [a[cut].contiguous() for a in (*tgt, *([] if tr is None else [tr]))]
        for j in range(0, src[0].numel(), most):
            s = [a[j:j + most].contiguous() for a in src]
            _cabi.call("o2d_hip_points_on_points_noalloc_dev_d", ctypes.byref(env), s[0].numel(),
                       *[p(a) for a in s], t[0].numel(), p(t[0]), p(t[1]),
                       p(t[2]) if tr is not None else None, p(u[cut]), p(v[cut]), None, None)
        torch.cuda.synchronize()
    return u, v
