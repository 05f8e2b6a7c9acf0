"""LOR preprocessing for the TOR model, on the device.

Restates src/python/srf/preprocess/function/on_tor_lors.py (reference) with
torch float64 tensor ops in the same order as the reference's numpy
expressions, so results are identical on any device.  Output groups are
structure-of-arrays float32 tensors in the group frame, ready for the ops:

  recon_process(lors[N, 7], tof_res)  -> {'x','y','z'}: [10, N_a]
      rows p1 (3), p2 (3), TOF centre (3), sigma2 factor, in the group frame
  map_process(lors[N, 6])             -> {'x','y','z'}: [7, N_a]
      rows p1 (3), p2 (3), sigma2 factor

Row order inside a group is the reference's: ascending event index
(np.intersect1d) for rows with d_axis >= 0, then those with d_axis < 0
(SwapPointsOrder).  ``order`` maps output rows to input rows.

float32 and float64 rows on a GPU go through the HIP kernels
(srfx_split_lors_*, srfx_locality_sort), which give the same bits; other rows
(host tensors, other types, rows that carry a gradient or a tangent, calls under
a tracer, a dispatch mode or stream capture) through the torch operations below.
"""
import ctypes

import torch
from torch.autograd import forward_ad
from torch.utils._python_dispatch import is_in_torch_dispatch_mode

from . import _lib

AXES = ("x", "y", "z")
GAUSSIAN_FACTOR = 2.35482005  # on_tor_lors.py:220
# Column permutations into the group frame, on_tor_lors.py:246-247, 259-260.
PERM_RECON = {"x": [1, 2, 0, 4, 5, 3, 7, 8, 6], "y": [0, 2, 1, 3, 5, 4, 6, 8, 7]}
PERM_MAP = {"x": [1, 2, 0, 4, 5, 3], "y": [0, 2, 1, 3, 5, 4]}


def sigma2_factor(lors):
    """on_tor_lors.py:137-166."""
    dx = lors[:, 3] - lors[:, 0]
    dy = lors[:, 4] - lors[:, 1]
    dz = lors[:, 5] - lors[:, 2]
    p_dis2 = (dx * dx + dy * dy) + dz * dz
    dsq = dx * dx + dy * dy
    rsq = lors[:, 0] * lors[:, 0] + lors[:, 3] * lors[:, 3] + lors[:, 1] * lors[:, 1] + \
        lors[:, 4] * lors[:, 4]
    return dsq * dsq / rsq / p_dis2 / 2


def dominant_masks(lors):
    """Partition rule, on_tor_lors.py:70-77."""
    d = (lors[:, 3:6] - lors[:, 0:3]).abs()
    ax, ay, az = d[:, 0], d[:, 1], d[:, 2]
    return {"x": (ax >= ay) & (ax >= az), "y": (ay > ax) & (ay >= az),
            "z": (az > ax) & (az > ay)}


def _partition_swap(lors, axis, mask):
    """Partition then SwapPointsOrder (on_tor_lors.py:175-193)."""
    a = AXES.index(axis)
    idx = torch.nonzero(mask, as_tuple=False).reshape(-1)
    part = lors[idx]
    d = part[:, 3 + a] - part[:, a]
    pos = d >= 0
    neg = d < 0
    positive = part[pos]
    negative = part[neg]
    if lors.shape[1] > 7:
        swapped = torch.cat([negative[:, 3:6], negative[:, 0:3], 0 - negative[:, 6:7],
                             negative[:, 7:]], 1)
    else:
        swapped = torch.cat([negative[:, 3:6], negative[:, 0:3], negative[:, 6:7]], 1)
    order = torch.cat([idx[pos], idx[neg]])
    return torch.cat([positive, swapped], 0), order


def cut_lors(lors, tof_res):
    """CutLoRs, on_tor_lors.py:196-229: output (p0, p1, centre, extra)."""
    p0 = lors[:, 0:3]
    p_diff = lors[:, 3:6] - p0
    p_dis = torch.sqrt((p_diff[:, 0] * p_diff[:, 0] + p_diff[:, 1] * p_diff[:, 1]) +
                       p_diff[:, 2] * p_diff[:, 2])
    dcos = p_diff / p_dis[:, None]
    ratio = 0.5 - (lors[:, 6] / p_dis)
    center = ratio[:, None] * p_diff + p0
    c0 = center - p0
    dcs = torch.sqrt((c0[:, 0] * c0[:, 0] + c0[:, 1] * c0[:, 1]) + c0[:, 2] * c0[:, 2])
    q0 = p0.clone()
    q1 = lors[:, 3:6].clone()
    if tof_res < 10000:
        limit = tof_res * 0.15 / GAUSSIAN_FACTOR * 3
        index = dcs > limit
        q0 = torch.where(index[:, None], center - limit * dcos, q0)
        q1 = torch.where(index[:, None], center + limit * dcos, q1)
    return torch.cat([q0, q1, center, lors[:, 7:]], 1)


def _as64(lors, ncols):
    if not isinstance(lors, torch.Tensor):
        lors = torch.as_tensor(lors)
    if lors.dim() != 2 or lors.shape[1] != ncols:
        raise ValueError(f"expected [N, {ncols}] rows, got {tuple(lors.shape)}")
    return lors.to(torch.float64)


def _native(t):
    return (type(t) is torch.Tensor and t.device.type == "cuda" and not t.requires_grad
            and not torch.jit.is_tracing() and not is_in_torch_dispatch_mode()
            and t.dim() == 2 and t.numel() > 0 and not t.is_neg()
            and forward_ad.unpack_dual(t).tangent is None
            and not torch.cuda.is_current_stream_capturing())


SPLIT_ROWS = 1024  # rows per workgroup of srfx_split_lors_count


def _split(rows, ncols, cut, limit, return_order):
    """recon_process (ncols 7) or map_process (6) of float32 / float64 device
    rows through srfx_split_lors_*: one count, the group sizes read back, one
    fill."""
    n, dev = rows.shape[0], rows.device
    with torch.cuda.device(dev):
        st = torch.cuda.current_stream().cuda_stream
        src = (rows.data_ptr(), n, rows.stride(0), rows.stride(1),
               1 if rows.dtype == torch.float64 else 0)
        work = torch.empty(6 * -(-n // SPLIT_ROWS), dtype=torch.int32, device=dev)
        totals = torch.empty(6, dtype=torch.int64, device=dev)
        _lib.call("srfx_split_lors_count", *src, work.data_ptr(), totals.data_ptr(), st)
        t = totals.tolist()
        sizes = [t[0] + t[1], t[2] + t[3], t[4] + t[5]]
        k = 10 if ncols == 7 else 7
        out = [torch.empty((k, m), dtype=torch.float32, device=dev) for m in sizes]
        order = [torch.empty(m, dtype=torch.int64, device=dev) if return_order else None
                 for m in sizes]
        ptrs = (ctypes.c_void_p * 3)(*[o.data_ptr() for o in out])
        lds = (ctypes.c_int64 * 3)(*sizes)
        ords = (ctypes.c_void_p * 3)(*[None if o is None else o.data_ptr() for o in order])
        _lib.call("srfx_split_lors_fill", *src, ncols, 1 if cut else 0, float(limit),
                  work.data_ptr(), totals.data_ptr(), ptrs, lds, ords, st)
    out = dict(zip(AXES, out))
    return (out, dict(zip(AXES, order))) if return_order else out


def _splittable(lors, ncols):
    return (_native(lors) and lors.shape[1] == ncols and lors.shape[0] < 2 ** 31
            and lors.dtype in (torch.float32, torch.float64))


def recon_process(lors, tof_res, return_order=False):
    """on_tor_lors.py:251-262.  lors: [N, 7] rows (x1, y1, z1, x2, y2, z2, tof)."""
    if _splittable(lors, 7):
        return _split(lors, 7, tof_res < 10000, tof_res * 0.15 / GAUSSIAN_FACTOR * 3,
                      return_order)
    lors = _as64(lors, 7)
    lors = torch.cat([lors, sigma2_factor(lors)[:, None]], 1)
    masks = dominant_masks(lors)
    out, orders = {}, {}
    for a in AXES:
        g, order = _partition_swap(lors, a, masks[a])
        g = cut_lors(g, tof_res)
        if a in PERM_RECON:
            g = torch.cat([g[:, PERM_RECON[a]], g[:, 9:]], 1)
        out[a] = g.to(torch.float32).t().contiguous()
        orders[a] = order
    return (out, orders) if return_order else out


def map_process(lors, return_order=False):
    """on_tor_lors.py:243-248.  lors: [N, 6] rows (x1, y1, z1, x2, y2, z2)."""
    if _splittable(lors, 6):
        return _split(lors, 6, False, 0.0, return_order)
    lors = _as64(lors, 6)
    lors = torch.cat([lors, sigma2_factor(lors)[:, None]], 1)
    masks = dominant_masks(lors)
    out, orders = {}, {}
    for a in AXES:
        g, order = _partition_swap(lors, a, masks[a])
        if a in PERM_MAP:
            g = torch.cat([g[:, PERM_MAP[a]], g[:, 6:]], 1)
        out[a] = g.to(torch.float32).t().contiguous()
        orders[a] = order
    return (out, orders) if return_order else out


def _spread8(v):
    """Spread the low 8 bits of v so that bit i moves to bit 4 i (for a
    4-way Morton interleave)."""
    v = v & 0xFF
    out = torch.zeros_like(v)
    for i in range(8):
        out |= ((v >> i) & 1) << (4 * i)
    return out


def locality_key(soa, center_z, zc_bin=40.0, slope_bin=0.04, pos_bin=6.0):
    """int64 key per event of a [10, N] group (op frame) that places events
    with nearby, nearly parallel tubes and nearby TOF centres next to each
    other: coarse TOF-centre position along the slice axis first, then a
    Morton interleave of the two slopes and the crossing point with the
    plane z = center_z."""
    x1, y1, z1 = soa[0].double(), soa[1].double(), soa[2].double()
    dx = soa[3].double() - x1
    dy = soa[4].double() - y1
    dz = soa[5].double() - z1
    dz = torch.where(dz == 0, torch.full_like(dz, 1e-12), dz)
    sx, sy = dx / dz, dy / dz
    X0 = x1 + sx * (center_z - z1)
    Y0 = y1 + sy * (center_z - z1)

    def q(v, step):
        return torch.clamp(torch.floor(v / step) + 128, 0, 255).long()

    zc = torch.clamp(torch.floor(soa[8].double() / zc_bin) + 64, 0, 127).long()
    m = _spread8(q(sx, slope_bin)) | (_spread8(q(sy, slope_bin)) << 1) | \
        (_spread8(q(X0, pos_bin)) << 2) | (_spread8(q(Y0, pos_bin)) << 3)
    return (zc << 32) | m


# locality_key's bins: TOF centre (mm), slopes, crossing point (mm)
ZC_BIN, SLOPE_BIN, POS_BIN = 40.0, 0.04, 6.0


def _sortable(soa, nb_subsets):
    return (_native(soa) and soa.dtype == torch.float32 and soa.shape[0] >= 9
            and soa.shape[1] < 2 ** 31 - 1 and hasattr(nb_subsets, "__index__")
            and 1 <= nb_subsets <= 1 << 24
            and soa.stride(1) == 1 and soa.stride(0) >= soa.shape[1])


def _locality_sort(soa, nb_subsets, center_z, gather):
    """(reordered group or None, order) through srfx_locality_sort."""
    with torch.cuda.device(soa.device):
        n = soa.shape[1]
        out = torch.empty((soa.shape[0], n), dtype=soa.dtype,
                          device=soa.device) if gather else None
        order = torch.empty(n, dtype=torch.int64, device=soa.device)
        _lib.call("srfx_locality_sort", soa.data_ptr(), n, soa.stride(0), soa.shape[0],
                  int(nb_subsets), float(center_z), ZC_BIN, SLOPE_BIN, POS_BIN,
                  out.data_ptr() if gather else None, order.data_ptr(),
                  torch.cuda.current_stream().cuda_stream)
    return out, order


def locality_order(soa, nb_subsets, center_z=0.0):
    """Permutation of a group's events that sorts each OSEM subset's rows
    [k N / K, (k+1) N / K) by locality_key and leaves subset membership
    unchanged."""
    if _sortable(soa, nb_subsets):
        return _locality_sort(soa, nb_subsets, center_z, False)[1]
    n = soa.shape[1]
    if n == 0 and soa.shape[0] >= 9 and hasattr(nb_subsets, "__index__"):
        return torch.empty(0, dtype=torch.int64, device=soa.device)
    key = locality_key(soa, center_z)
    order = torch.empty(n, dtype=torch.int64, device=soa.device)
    for k in range(nb_subsets):
        lo, hi = (k * n) // nb_subsets, ((k + 1) * n) // nb_subsets
        if hi > lo:
            order[lo:hi] = lo + torch.argsort(key[lo:hi], stable=True)
    return order


def reorder_groups(groups, nb_subsets, centers=None):
    """Apply locality_order to every group; returns (groups, orders) with
    orders[a][i] = original row of output row i."""
    out, orders = {}, {}
    for a, soa in groups.items():
        cz = 0.0 if centers is None else centers[a]
        if _sortable(soa, nb_subsets):
            out[a], orders[a] = _locality_sort(soa, nb_subsets, cz, True)
            continue
        o = locality_order(soa, nb_subsets, cz)
        out[a] = soa[:, o].contiguous()
        orders[a] = o
    return out, orders
