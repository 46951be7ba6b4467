"""Sample plans: tile binning of one trajectory against one oversampled grid.

A plan is built once per (trajectory, grid geometry, kernel width) and reused by
every interp / gridding / gradient call on that trajectory, so the CG loop pays
for binning once. Building it runs a stable LSD radix sort of the samples by
(tile, corner position in the tile) -- two or three counting-sort passes of a
per-chunk histogram, a scan and a stable scatter -- and two small passes for the
work items; the only host synchronisation is the work-item count.

Coordinate handling is bit-exact with the reference:
  * ``triton_nufft._scale_trj`` (fourier.py:420-430): t = fl32(fl32(k * fl32(G/N)) + G//2)
  * ``prep_ungrid_shapes`` / ``prep_grid_shapes`` (ungrid.py:864-865, grid.py:516-517):
    t = torch.remainder(t, G)
  * ``get_neighborhood`` (kernels.py:531-536): lower = ceil(t - w/2)
"""

from __future__ import annotations

import ctypes as C
import math
from dataclasses import dataclass

import torch

from . import _lib
from ._lib import check, lib, ptr, stream_ptr

MAX_DIGIT = 8192  # largest radix of one sort pass (mra_bin_build)


def binning_chunk(npts: int, ntiles: int, tile: int, ndim: int) -> int:
    """Samples per radix-sort chunk. One wave walks a chunk in order, so the chunks are the
    parallelism of each scatter pass (4096-sample chunks left a 131 k-sample trajectory 32
    waves); each pass's histogram holds digits x chunks counts, written and scanned whole.
    Aim for about 1024 chunks of 128..4096 samples, with at most 2^24 counts per histogram
    (measured: a 5.12 M-sample 3D plan takes 0.84 ms at 4096, 1.4 ms at 1024, 7 ms at 128)."""
    digits = max(tile ** ndim, min(ntiles + 1, MAX_DIGIT))
    c = -(-npts // 1024)
    c = min(max(-(-c // 64) * 64, 128), 4096)
    while c < 4096 and digits * -(-npts // c) > 1 << 24:
        c *= 2
    return min(c, 4096)


def item_lengths(npts: int, ndim: int = 2) -> tuple:
    """Work-item sizes to choose from, the preferred one first: about a thousand items per
    trajectory, 256..8192 samples each; in 3D at most 2560, so that the tiles of the k-space centre
    do not end a launch alone (gridding to images of a 128^3 kooshball of 5.12 M samples, 2560 /
    5120 samples an item: 32 coils 4.37 / 4.53 ms, 16 coils 2.34 / 2.54, 4 coils 0.87 / 1.08), with
    the uncapped size second."""
    s = -(-npts // 1024)
    s = min(max(-(-s // 256) * 256, 256), 8192)
    return (2560, s) if ndim == 3 and s > 2560 else (s,)


def default_samples_per_item(npts: int, ndim: int = 2) -> int:
    """Preferred work-item size (``item_lengths``)."""
    return item_lengths(npts, ndim)[0]


def choose_item_length(nitems, subgrid: int, limit: int) -> int:
    """Index of the work-item size a plan takes, of those that cut it into ``nitems`` items
    (preferred size first) with subgrids of ``subgrid`` points: the first one, unless the
    no-allocation gridding scratch (``limit`` bytes) holds more batch entries with a later one.
    Shorter items mean more partial subgrids, and a call that fits must not stop fitting (14 M
    samples on an 80^3 grid, one entry: 81 MB with items of 2560 samples, 30 MB with 8192)."""
    entries = [limit // (n * subgrid * 8) for n in nitems]
    return entries.index(max(entries))


def batch_samples_per_item(sizes) -> int:
    """Work-item size of problems that share their launches, ``sizes`` their (samples, coils):
    other problems' items fill the device, so an item may be longer, which saves partial subgrids,
    as long as about 4096 waves (of four coils) are left. Normal operator of a batch, us at 256 /
    512 / 1024 samples an item:
      24 problems x 25.6 k x 8 coils   191 /  202 /  229     24 x 25.6 k x 32       660 / 609 / 607
      24 x 51 k x 4                    347 /  360 /  388     16 x 131 k x 16       1068 / 928 / 947
      12 x 102 k x 8                   391 /  369 /  396     24 x 410 k x 8        1545 / 1244 / 1156
    and 24 of 20..130 k x 8..32 with 8 solver steps 14.5 / 12.8 / 12.5 ms; 2048 samples were slower
    than 1024 up to 8 M samples a problem (8 x 2 M x 8: 1355 / 1395 us)."""
    sizes = list(sizes)
    waves = sum(n * -(-c // 4) for n, c in sizes)
    fill = (waves // 4096 + 128) // 256 * 256
    return min(default_samples_per_item(sum(n for n, _ in sizes) // 2), 1024, max(fill, 256))


def dcf_samples_per_item(npts: int, ndim: int) -> int:
    """Work-item size of density compensation, whose one batch entry leaves one wave to an item:
    half the usual length, so that the launch does not end on its longest items, but not below 512
    samples, where the partial subgrids cost more than that (one iteration, us, at the usual length
    / half / a quarter: 96^3, 1.5 M samples: 178 / 151 / 169; 128^3, 5.1 M: 542 at 5120, 378 at 1280;
    256^2, 2 M: 140 / 128 / 152; at 512 / 256: 64^3, 0.38 M: 78 / 85; 256^2, 0.41 M: 53 / 62)."""
    s = default_samples_per_item(npts, ndim)
    return max(s // 2, min(s, 512))


def kernel_points(width: float) -> int:
    """Grid points per dimension a KB patch of width ``width`` can touch."""
    return int(math.floor(float(width))) + 1


@dataclass(frozen=True)
class GeomKey:
    nbatch: int
    ksp_stride: int
    out_scale: float
    grid_stride: int
    dcf_plan_order: bool = False
    ksp_plan_order: bool = False


class SamplePlan:
    """Tile-sorted samples of one trajectory on one grid.

    Parameters
    ----------
    coords : (..., D) float32 device tensor, reference units (see ``scale``)
    grid_size : tuple of D ints, the (oversampled) grid the samples live on
    width : kernel width in grid points (same in every dim)
    beta : Kaiser-Bessel shape parameter (or one per dimension)
    scale, shift : per-dim fp32 scale and shift applied before wrapping (the
        NUFFT's ``_scale_trj``); ``None`` means coordinates are already in grid
        units (the plain ``ungrid``/``grid`` surface)
    wrap : per-dim integer added to a grid index before it wraps mod G. The
        NUFFT uses ``-(G//2)`` so kernels address the unshifted FFT output.
    tile : tile edge in grid points (default: the edge selected for this thread, see
        ``_lib.tile_scope``; kernels are compiled for 2D edges 8, 16, 32, 1D 256, 3D 8)
    samples_per_item : max samples per work item (default: about 1k items)
    """

    def __init__(self, coords: torch.Tensor, grid_size, width: float, beta: float, *, scale=None, shift=None,
                 wrap=None, tile: int | None = None, samples_per_item: int | None = None):
        _lib.require_device(coords)
        L = lib()
        D = len(grid_size)
        if coords.shape[-1] != D:
            raise ValueError(f"coords last dim {coords.shape[-1]} != grid ndim {D}")
        if D < 1 or D > 3:
            raise ValueError("the HIP NUFFT supports 1D, 2D and 3D grids")
        if coords.dtype != torch.float32:
            raise TypeError(f"coordinates must be float32, got {coords.dtype}")
        self.device = coords.device
        self.ndim = D
        self.grid_size = tuple(int(g) for g in grid_size)
        self.width = float(width)
        self.P = kernel_points(width)
        if not 2 <= self.P <= 9:
            raise ValueError(f"kernel width {width} unsupported: floor(width)+1 must be in 2..9")
        if isinstance(beta, (tuple, list)):  # one KB shape per dimension (sigpy's `param` tuple)
            if len(beta) != D:
                raise ValueError(f"{len(beta)} betas for a {D}-dimensional grid")
            self.betas = tuple(float(b) for b in beta)
        else:
            self.betas = (float(beta),) * D
        self.beta = self.betas[0]
        self.coords_shape = tuple(coords.shape[:-1])
        self.npts = int(math.prod(self.coords_shape))
        if self.npts <= 0:
            raise ValueError("trajectory has no samples")
        self.tile = int(tile or L.mra_tile(D))
        with _lib.tile_scope(D, self.tile):  # raises for an edge without kernels
            pass
        self.ntile = [(g + self.tile - 1) // self.tile for g in self.grid_size]
        self.ntiles = int(math.prod(self.ntile))
        lengths = (int(samples_per_item),) if samples_per_item else item_lengths(self.npts, D)
        if lengths[0] < 1:
            raise ValueError("samples_per_item must be positive")
        self.wrap = tuple(int(w) for w in (wrap if wrap is not None else (0,) * D))

        flat = coords.reshape(-1, D).contiguous()
        dev = self.device
        chunk = binning_chunk(self.npts, self.ntiles, self.tile, D)
        wwords = int(L.mra_bin_workspace(D, self.npts, self.ntiles, self.tile, chunk))
        if wwords < 0:
            check(1)
        work = torch.empty(wwords, dtype=torch.int32, device=dev)
        self.tsort = torch.empty(self.npts * D, dtype=torch.float32, device=dev)
        self.perm = torch.empty(self.npts, dtype=torch.int32, device=dev)
        nkeys = self.ntiles + 1
        self.tile_start = torch.empty(nkeys + 1, dtype=torch.int32, device=dev)
        apply = scale is not None
        sc = _lib.floats(scale if apply else [1.0] * D)
        sh = _lib.floats(shift if shift is not None else [0.0] * D)
        st = stream_ptr(dev)
        check(L.mra_bin_build(D, ptr(flat), self.npts, _lib.ints(self.grid_size), sc, sh, int(apply),
                              self.width, self.tile, _lib.ints(self.wrap), chunk, ptr(work), ptr(self.tsort),
                              ptr(self.perm), ptr(self.tile_start), st))
        nitems_ws = torch.empty(nkeys + 1, dtype=torch.int32, device=dev)
        scan_ws2 = torch.empty(L.mra_scan_workspace(nkeys + 1), dtype=torch.int32, device=dev)
        cuts = []  # per work-item size: the items, and the first of each tile (tile ntiles: non-finite samples)
        for S in lengths:
            max_items = nkeys + (self.npts + S - 1) // S
            items = torch.empty((max_items, 4), dtype=torch.int32, device=dev)
            item_off = torch.empty(nkeys + 1, dtype=torch.int32, device=dev)
            check(L.mra_bin_items(ptr(self.tile_start), self.ntiles, S, 0, ptr(nitems_ws), ptr(item_off),
                                  ptr(scan_ws2), ptr(items), max_items, st))
            cuts.append((S, items, item_off))
        # KB weights (D x P per sorted sample) and subgrid offsets, once per trajectory
        self.wsort = torch.empty(self.npts * D * self.P, dtype=torch.float32, device=dev)
        self.lbase = torch.empty(self.npts, dtype=torch.int32, device=dev)
        with _lib.tile_scope(D, self.tile):
            check(L.mra_plan_weights_dims64(D, self.P, ptr(self.tsort), self.npts, _lib.ints(self.grid_size),
                                            _lib.ints(self.wrap), self.width, _lib.doubles(self.betas),
                                            ptr(self.wsort), ptr(self.lbase), st))
            self.subgrid = int(L.mra_subgrid_points(D, self.P))
            self.max_coil_chunk = int(L.mra_max_coil_chunk(D, self.P))
        # The only host synchronisation of a plan: the number of work items, which
        # sizes the launches and the gridding scratch.
        if len(cuts) == 1:
            nitems = [int(cuts[0][2][nkeys].item())]
        else:
            nitems = torch.stack([off[nkeys] for _, _, off in cuts]).tolist()
        i = choose_item_length(nitems, self.subgrid, int(L.mra_grid_noalloc_max_bytes()))
        self.nitems = nitems[i]
        self.S, self.items, self.tile_items = cuts[i]
        self.max_items = self.items.shape[0]
        # The workspaces go back to the caching allocator here; PyTorch only
        # hands them out again to work ordered after these kernels on this stream.
        del work, nitems_ws, scan_ws2, flat, cuts, items, item_off
        self._geoms: dict[GeomKey, torch.Tensor] = {}

    def coil_chunk(self, nbatch: int) -> int:
        """Coils per block: as many subgrids as the per-block LDS budget holds."""
        return max(1, min(nbatch, self.max_coil_chunk))

    def geom(self, nbatch: int, ksp_stride: int | None = None, out_scale: float = 1.0,
             grid_stride: int | None = None, dcf_plan_order: bool = False,
             ksp_plan_order: bool = False) -> torch.Tensor:
        """Device Geom table (one entry) for a call on ``nbatch`` grids; ``dcf_plan_order``:
        the gridding dcf comes in sorted (plan) order (``dcf[perm]``); ``ksp_plan_order``:
        k-space (interp output, gridding input) and dcf are all in sorted order."""
        gstride = int(grid_stride if grid_stride is not None else math.prod(self.grid_size))
        kstride = int(ksp_stride if ksp_stride is not None else self.npts)
        key = GeomKey(int(nbatch), kstride, float(out_scale), gstride, bool(dcf_plan_order), bool(ksp_plan_order))
        g = self._geoms.get(key)
        if g is None:
            g = make_geoms([dict(grid_off=0, grid_stride=gstride, ksp_off=0, ksp_stride=kstride, samp_off=0,
                                 nbatch=int(nbatch), npts=self.npts, grid_size=self.grid_size, tile=self.tile,
                                 wrap=self.wrap, beta=self.beta, width=self.width, out_scale=out_scale,
                                 item_base=0, scratch_off=0, tile_items_off=0,
                                 dcf_plan_order=bool(dcf_plan_order), ksp_plan_order=bool(ksp_plan_order))],
                           self.device)
            self._geoms[key] = g
        return g


    def geom_host(self, nbatch: int, out_scale: float = 1.0):
        """Host Geom record of a one-problem call on ``nbatch`` grids (what ``geom`` puts in
        device memory), for the no-allocation gridding entry point."""
        return pack_geoms([dict(grid_off=0, grid_stride=math.prod(self.grid_size), ksp_off=0, ksp_stride=self.npts,
                                samp_off=0, nbatch=int(nbatch), npts=self.npts, grid_size=self.grid_size,
                                tile=self.tile, wrap=self.wrap, beta=self.beta, width=self.width,
                                out_scale=out_scale)])


def pack_geoms(entries: list[dict]):
    """Pack Geom records (see common.h) into a host ctypes byte buffer."""
    L = lib()
    gsz = L.mra_geom_size()
    buf = (C.c_ubyte * (gsz * len(entries)))()
    for i, e in enumerate(entries):
        D = len(e["grid_size"])
        with _lib.tile_scope(D, e["tile"]):
            check(L.mra_geom_fill(C.addressof(buf) + i * gsz, e["grid_off"], e["grid_stride"], e["ksp_off"],
                                  e["ksp_stride"], e["samp_off"], e["nbatch"], e["npts"], D,
                                  _lib.ints(e["grid_size"]), e["tile"], _lib.ints(e["wrap"]), e["beta"], e["width"],
                                  e["out_scale"], e.get("item_base", 0), e.get("scratch_off", 0),
                                  e.get("tile_items_off", 0)))
        if e.get("dcf_plan_order"):
            check(L.mra_geom_set_dcf_plan_order(C.addressof(buf) + i * gsz, 1))
        if e.get("ksp_plan_order"):
            check(L.mra_geom_set_ksp_plan_order(C.addressof(buf) + i * gsz, 1))
    return buf


def make_geoms(entries: list[dict], device) -> torch.Tensor:
    """Pack Geom records (see common.h) into a device byte tensor."""
    host = torch.frombuffer(bytearray(bytes(pack_geoms(entries))), dtype=torch.uint8)
    return host.to(device)
