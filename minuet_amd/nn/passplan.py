"""Building the coordinate levels and kernel maps of a whole pass at once.

A network asks its :class:`~minuet_amd.nn.KernelMapCache` for the same levels
and maps for every cloud.  The cache keeps the list of what the last pass
asked for; at the first request of the next pass a :class:`PassPlan` hands the
whole list to the library (``mnt_pass_levels`` / ``mnt_pass_build``), which
builds it in about ten launches and one wait, where the requests one by one
take up to a hundred launches and a wait per level.  The results are those of
the single calls; what the pass then does not ask for leaves the list.  The
reference builds every map at the first layer that needs it
(minuet/nn/convolutions.py:58-173)."""
import ctypes
from typing import Optional

import numpy as np
import torch

from minuet_amd.nn.functional import _C
from minuet_amd.nn.kernel_map import KernelMap

__all__ = ["PassPlan", "BuiltPass"]

_INVERSE, _GROUPS, _TABLES = 1, 2, 4
_MAP_SHAPE = (_C.PassMap.num_offsets.offset // 8, _C.PassMap.num_sources.offset // 8, _C.PassMap.num_targets.offset // 8)
_MAP_AT = _C.PassMap.at.offset // 8


def requests_of(fast, reorder: bool):
    """What a layer that ran through the extension module with the map of the request
    ``fast`` (see ``PassPlan``) has asked for: that map, and the level it leads to."""
    _, _, _, kind, key, transposed = fast
    if key[0] != key[1]:
        yield "coords", key[0], key[1]
    yield "dense", key
    if kind == "IMPLICIT":
        if transposed:
            yield "invert", key
    elif kind == "GROUPS":
        yield "groups", key
    else:
        yield "tables", key, reorder
    yield fast


class PassPlan:
    """The list of a pass, laid out for the library.

    ``requests``: ``("coords", source_stride, target_stride)``, ``("dense", key)``,
    ``("invert", key)``, ``("groups", key)``, ``("tables", key, reorder)`` with
    ``key`` the cache's ``(source_stride, target_stride, kernel_size, dilation)``,
    ``("tiles", key, transposed)`` where the layers would have saved more by the
    tiles of the map (or its inverse) than making them takes, and
    ``("fast", shape_id, in_stride, kind, key, transposed)`` for the layers
    that ran through the extension module.  Raises ``ValueError`` when they
    cannot be built from a cloud of stride ``stride``."""

    def __init__(self, requests, offsets_of, stride, index_dtype: torch.dtype):
        self.requests = tuple(requests)
        self.stride = stride
        self.index_dtype = index_dtype
        self.level_of = {stride: 0}
        for entry in self.requests:
            if entry[0] == "coords":
                _, source, target = entry
                if target in self.level_of or any(t % s for t, s in zip(target, stride)):
                    raise ValueError(f"level {target} cannot be built from {stride}")
                self.level_of[target] = len(self.level_of)
        self.map_of = {}
        wants, reorders = {}, {}
        for entry in self.requests:
            kind = entry[0]
            if kind in ("dense", "invert", "groups", "tables"):
                key = entry[1]
                if key[0] not in self.level_of or key[1] not in self.level_of:
                    raise ValueError(f"map {key} cannot be built from {stride}")
                self.map_of.setdefault(key, len(self.map_of))
                if kind == "tables" and index_dtype != torch.int32:
                    continue                     # tables of another index type are cast: made when asked for
                wants[key] = wants.get(key, 0) | {"invert": _INVERSE, "groups": _GROUPS, "tables": _TABLES}.get(kind, 0)
                if kind == "tables":
                    reorders[key] = bool(entry[2])
        if not self.map_of:
            raise ValueError("nothing to build")
        self.wants, self.reorders = wants, reorders
        self.levels = (_C.PassLevel * max(1, len(self.level_of) - 1))()
        self.num_levels = len(self.level_of) - 1
        for target, level in self.level_of.items():
            if level:
                for k, value in enumerate(target):
                    self.levels[level - 1].stride[k] = int(value)
        self.maps = (_C.PassMap * len(self.map_of))()
        self._keep = []
        self._group_tables = {}
        self.host_words = 0
        self.host_at = {}
        for key, i in self.map_of.items():
            source, target, kernel_size, dilation = key
            offsets = offsets_of(source, kernel_size, dilation)
            self._keep.append(offsets)
            item = self.maps[i]
            item.source_level, item.target_level = self.level_of[source], self.level_of[target]
            item.want = wants.get(key, 0)
            item.reorder = 1 if reorders.get(key, False) else 0
            item.offsets_host = offsets.ctypes.data
            item.num_offsets = offsets.shape[0]
            if item.want & _GROUPS:
                table = _C.offset_group_table(offsets)
                if table is None:
                    raise ValueError(f"map {key} has no offset groups")
                self._group_tables[key] = (table, table.ctypes.data)
                item.group_offsets_host = table.ctypes.data
            if item.want & _TABLES:
                self.host_at[key] = self.host_words
                self.host_words += 2 * offsets.shape[0]
        # (the maps' tiles follow them in launches of their own, one set for all)
        self.tiles = [(entry[1], entry[2]) for entry in self.requests if entry[0] == "tiles" and entry[1] in self.map_of
                      and (not entry[2] or wants.get(entry[1], 0) & _INVERSE)]
        self.fast = [entry for entry in self.requests if entry[0] == "fast" and self._serves(entry)]
        # the library's results, one row of int64 words a map (the struct has no gaps)
        self._map_words = np.frombuffer(self.maps, dtype=np.int64).reshape(len(self.map_of), -1)

        # what there is beside tiles, and whether the layers of the extension module ask for all of it
        self._tiles_asked = {entry for entry in self.requests if entry[0] == "tiles"}
        self._asked = set(self.requests) - self._tiles_asked
        self._fast_alone = self._asked == {asked for entry in self.fast
                                           for asked in requests_of(entry, reorders.get(entry[4], False))}

    def is_repeated(self, built, requests, tiles) -> bool:
        """Whether a pass that ran on ``built``, whose layers asked Python for no more
        than ``requests`` and would ask for ``tiles``, asked for just this plan's list:
        ``is_for``, without putting that list together."""
        return (self._fast_alone and tiles == self._tiles_asked and len(built.entries) == len(self.fast)
                and all(entry.used for entry, _ in built.entries) and self._asked.issuperset(requests))

    def _serves(self, entry) -> bool:
        _, _, _, kind, key, transposed = entry
        if key not in self.map_of:
            return False
        want = self.wants.get(key, 0)
        if kind == "IMPLICIT":
            return not transposed or bool(want & _INVERSE)
        return bool(want & (_GROUPS if kind == "GROUPS" else _TABLES))

    def build(self, coordinates: torch.Tensor, batch_dims: Optional[torch.Tensor], bounds) -> Optional["BuiltPass"]:
        """Everything on the list for the sorted cloud ``coordinates``, or None
        where the library does not take it."""
        total = _C.pass_levels(coordinates, batch_dims, bounds, self.levels, self.num_levels, self.maps,
                               self._check_memory)
        if total is None:
            return None
        size, bounds = total
        hosts = np.empty(max(1, self.host_words), dtype=np.int64)
        base = hosts.ctypes.data
        for key, at in self.host_at.items():
            item = self.maps[self.map_of[key]]
            item.sizes_host = base + 8 * at
            item.order_host = base + 8 * (at + item.num_offsets)
        store = torch.empty(max(size, 256), dtype=torch.uint8, device=coordinates.device)
        _C.pass_build(coordinates, batch_dims, self.levels, self.maps, store)
        return BuiltPass(self, coordinates, batch_dims, bounds, store, hosts)

    def is_for(self, requests) -> bool:
        """Whether this is the plan of just these requests."""
        return len(self.requests) == len(requests) and all(entry in requests for entry in self.requests)

    # pair lists get room for their worst case (every (offset, target) pair a hit)
    def _check_memory(self, rows: int) -> bool:
        pairs = [self.maps[i].num_offsets for key, i in self.map_of.items() if self.wants.get(key, 0) & _TABLES]
        return not pairs or max(pairs) * rows * 8 <= _C.PAIR_LIST_SLACK_BYTES


class BuiltPass:
    """What a :class:`PassPlan` built for one cloud: views of one allocation,
    made when asked for."""

    def __init__(self, plan: PassPlan, coordinates, batch_dims, bounds, store, hosts):
        self.plan, self.bounds = plan, bounds
        self.store, self.hosts = store, hosts
        self.base = store.data_ptr()
        self.ints = store.view(torch.int32)
        device = coordinates.device
        ndim = coordinates.shape[1]
        self.device = device
        typed = self.ints if coordinates.dtype == torch.int32 else store.view(coordinates.dtype)
        size = coordinates.dtype.itemsize
        self.coordinates = {plan.stride: (coordinates, plan.stride, batch_dims)}
        boundaries = batch_dims.shape[0] if batch_dims is not None else 0
        typed_dims = None if batch_dims is None else typed if batch_dims.dtype == coordinates.dtype else store.view(batch_dims.dtype)
        self.batched = boundaries > 2    # (what says that there is one cloud is dropped)
        for target, level in plan.level_of.items():
            if level:
                item = plan.levels[level - 1]
                rows = typed.as_strided((item.count, ndim), (ndim, 1), item.coords_at // size)
                dims = batch_dims
                if item.batch_dims_at >= 0:
                    dims = typed_dims.as_strided((boundaries,), (1,), item.batch_dims_at // batch_dims.dtype.itemsize)
                elif batch_dims is not None:             # one cloud carrying its boundaries
                    dims = torch.tensor([0, item.count][:batch_dims.numel()], dtype=batch_dims.dtype, device=device)
                self.coordinates[target] = (rows, target, dims)
        words = plan._map_words.tolist()
        self.at = {key: words[i][_MAP_AT:] for key, i in plan.map_of.items()}
        o, s, t = _MAP_SHAPE
        self.shape = {key: (words[i][o], words[i][s], words[i][t]) for key, i in plan.map_of.items()}
        self.entries = []                # (extension's entry, the request it stands for)
        self.tiles, self.stream = {}, None
        if plan.tiles:                   # (key, transposed) -> tiles, and the stream that makes them
            self.tiles, self.stream = self._make_tiles(), torch.cuda.current_stream(device).cuda_stream

    def _make_tiles(self) -> dict:
        maps = {}
        for key, transposed in self.plan.tiles:
            offsets, sources, targets = self.shape[key]
            at, rows = self.at[key][1 if transposed else 0], sources if transposed else targets
            if at >= 0 and 0 < rows and offsets * rows <= _C.MOST_TILE_ENTRIES:
                maps[key, transposed] = (self.base + at, rows, offsets)
        try:
            return dict(zip(maps, _C.kernel_maps_tiles(list(maps.values()), self.device))) if maps else {}
        except torch.OutOfMemoryError:   # the layers run without
            return {}

    def tiles_of(self, key, transposed: bool, dense: torch.Tensor) -> Optional[torch.Tensor]:
        """The tiles made of the map ``dense``, if it is this pass's."""
        tiles = self.tiles.get((key, transposed))
        if tiles is None or dense.data_ptr() != self.base + self.at[key][1 if transposed else 0]:
            return None
        return tiles

    def _from(self, key, coordinates) -> bool:
        """Whether the map ``key`` was built from this very tensor of source coordinates."""
        if key not in self.shape:
            return False
        mine = self.coordinates[key[0]][0]
        return mine is coordinates or (mine.data_ptr() == coordinates.data_ptr() and mine.shape == coordinates.shape)

    def _view(self, at: int, rows: int, columns: int) -> torch.Tensor:
        return self.ints.as_strided((rows, columns), (columns, 1), at // 4)

    def dense(self, key, coordinates):
        if not self._from(key, coordinates):
            return None
        offsets, _, targets = self.shape[key]
        return self._view(self.at[key][0], offsets, targets)

    def inverse(self, key):
        if key not in self.shape or self.at[key][1] < 0:
            return None
        offsets, sources, _ = self.shape[key]
        return self._view(self.at[key][1], offsets, sources)

    def groups(self, key, coordinates):
        if not self._from(key, coordinates) or self.at[key][2] < 0:
            return None
        _, _, targets = self.shape[key]
        _, _, rank, src, head = self.at[key][:5]
        return _C.OffsetGroups(self._view(rank, 9, targets), self._view(src, 9 * targets, 4),
                               self.ints.as_strided((16,), (1,), head // 4), self.plan._group_tables[key][0], targets)

    def _host(self, key):
        at, offsets = self.plan.host_at[key], self.shape[key][0]
        return self.hosts[at:at + offsets], self.hosts[at + offsets:at + 2 * offsets]

    def tables(self, key, coordinates, reorder: bool) -> Optional[KernelMap]:
        if (not self._from(key, coordinates) or self.at[key][5] < 0 or self.plan.reorders[key] != reorder):
            return None
        offsets, sources, targets = self.shape[key]
        dense, _, _, _, _, smask, tmask, in_idx, out_idx, sizes, order = self.at[key]
        sizes_host, order_host = self._host(key)
        nnz = int(sizes_host.sum())
        line = lambda at, n: self.ints.as_strided((n,), (1,), at // 4)
        return KernelMap(self._view(smask, offsets, sources), self._view(tmask, offsets, targets),
                         line(order, offsets) if reorder else None, line(sizes, offsets), sizes_host=sizes_host,
                         order_host=order_host if reorder else None, in_idx=line(in_idx, nnz),
                         out_idx=line(out_idx, nnz), dense=self._view(dense, offsets, targets),
                         num_sources=sources, num_targets=targets)

    def fill_fast(self, fast_maps: dict):
        """Entries for the extension module: the layers that ran through it in
        the last pass find their maps without a detour through Python."""
        host = _C.load_host()
        if host is None:
            return
        index = self.device.index
        for request in self.plan.fast:
            _, shape_id, in_stride, kind, key, transposed = request
            offsets, sources, targets = self.shape[key]
            if kind == "IMPLICIT":
                a = self.at[key][1 if transposed else 0]
                pointers = (None if a < 0 else self.base + a,)
                owners = self.store
            elif kind == "GROUPS":
                table, address = self.plan._group_tables[key]
                at = [None if a < 0 else self.base + a for a in self.at[key]]
                pointers = (at[2], at[3], at[4], address)
                owners = (self.store, table)
            else:
                if not self.plan.reorders[key]:
                    continue
                sizes_host, order_host = self._host(key)
                at = [None if a < 0 else self.base + a for a in self.at[key]]
                smask, tmask, in_idx = (at[6], at[5], at[8]) if transposed else (at[5], at[6], at[7])
                pointers = (smask, tmask, at[10], at[9], sizes_host.ctypes.data, order_host.ctypes.data, in_idx)
                owners = (self.store, self.hosts)
            source, target = (key[1], key[0]) if transposed else (key[0], key[1])
            coordinates, stride, batch_dims = self.coordinates[target]
            if not self.batched:
                batch_dims = None
            entry = host.MapEntry(getattr(host, kind), coordinates, stride, batch_dims, owners, index, 0,
                                  targets if transposed else sources, sources if transposed else targets, pointers,
                                  self.coordinates[source][0].data_ptr(),
                                  self.tiles.get((key, transposed)) if kind == "IMPLICIT" else None)
            fast_maps.setdefault(shape_id, {})[in_stride] = entry
            self.entries.append((entry, request))
