"""The public ``NeighborList`` descriptor, executed on one AMD Instinct GPU.

Mirrors the reference's public class (generated by ``adapter_class`` from
``NeighborListKernel``, ``src/mdescriptor/descriptors/standalone/local/
__init__.py:17`` and ``src/mdescriptor/descriptors/_kernels/local.py:73-110``)
and its registry entry (``src/mdescriptor/registry/builtins.py:861-886``):

* keyword-only constructor ``NeighborList(*, cutoff=6.0,
  full_neighbor_list=True, self_pairs=False, output=None, execution=None)``;
* direct values of the wrong type are rejected as the reference's public
  parameter check rejects them (``src/mdescriptor/registry/info.py:493-570``,
  code ``invalid_parameter``), a non-positive cutoff as the kernel's
  ``ValueError`` wrapped into ``invalid_configuration``;
* the result is pair-level: values ``(dx, dy, dz, distance)``, one row per
  kept pair, per-structure row offsets and the pair samples
  ``[structure, local_i, local_j, shift_a, shift_b, shift_c]``.

The pairs are those of the reference's ``compute_neighbor_list``
(``cpp/src/standalone/neighbor_list.cpp:15-78``): boundary inclusive, the
exact self pair only with ``self_pairs``, one orientation per pair without
``full_neighbor_list`` (``cpp/include/mdescriptor/detail/neighbor_filter.hpp:
18-38``).  Graph, filter and record layout all run on the device
(``mdx_hip_neighbor_list``).
"""

from __future__ import annotations

import threading
from typing import Any

import numpy as np

from ..core.backends import HipBackend
from ..core.descriptor import Descriptor
from ..core.errors import DescriptorConfigError, DescriptorInputError
from ..core.options import CONFIGURATION_SCHEMA_VERSION, ExecutionOptions, OutputOptions, coerce_options
from ..core.result import DescriptorResult, format_values, metadata_envelope, owned_samples, owned_values

SUPPORTED_DEVICES = ("hip",)
LABELS = ("dx", "dy", "dz", "distance")
DEFAULTS = {"cutoff": 6.0, "full_neighbor_list": True, "self_pairs": False}
_SCHEMA_TYPES = {"cutoff": "number", "full_neighbor_list": "boolean", "self_pairs": "boolean"}


def _check_type(name: str, value: Any) -> None:
    """The direct-constructor type guard of the reference's registry schema
    (info.py:530-545): numbers are int or float but not bool, booleans are bool."""

    kind = _SCHEMA_TYPES[name]
    if kind == "number":
        valid = isinstance(value, (int, float, np.integer, np.floating)) and not isinstance(value, (bool, np.bool_))
    else:
        valid = isinstance(value, (bool, np.bool_))
    if not valid:
        raise DescriptorConfigError(f"descriptor parameter value does not match type {kind!r}",
                                    code="invalid_parameter", path=["parameters", name])


class NeighborList(Descriptor):
    """Neighbour pair displacements and distances, computed on an AMD GPU."""

    name = "NeighborList"
    supported_devices = SUPPORTED_DEVICES

    def __init__(self, *, cutoff: float | None = None, full_neighbor_list: bool | None = None,
                 self_pairs: bool | None = None, output: Any = None, execution: Any = None) -> None:
        super().__init__()
        given = {"cutoff": cutoff, "full_neighbor_list": full_neighbor_list, "self_pairs": self_pairs}
        for key, value in given.items():
            if value is not None:
                _check_type(key, value)
        self._output_options = coerce_options(output, OutputOptions, "output")
        self._execution_options = coerce_options(execution, ExecutionOptions, "execution")
        device = self._execution_options.device
        if device not in self.supported_devices:
            raise DescriptorConfigError(
                f"{self.name} does not support execution.device={device!r}; supported devices: "
                + ", ".join(self.supported_devices),
                code="unsupported_device",
                path=["execution", "device"],
                details={"supported": list(self.supported_devices)},
            )
        resolved = {key: DEFAULTS[key] if value is None else value for key, value in given.items()}
        self.cutoff = float(resolved["cutoff"])
        self.full_neighbor_list = bool(resolved["full_neighbor_list"])
        self.self_pairs = bool(resolved["self_pairs"])
        if self.cutoff <= 0.0:  # local.py:85-86; non-finite values reach the device check
            raise DescriptorConfigError(f"invalid {self.name} configuration: cutoff must be positive",
                                        code="invalid_configuration", path=["parameters", "cutoff"])
        parameters: dict[str, Any] = {
            "cutoff": resolved["cutoff"],
            "full_neighbor_list": self.full_neighbor_list,
            "self_pairs": self.self_pairs,
            "output": self._output_options.to_dict(),
            "execution": self._execution_options.to_dict(),
        }
        self._set_configuration(CONFIGURATION_SCHEMA_VERSION, parameters)
        backend_options = {
            "cutoff": self.cutoff,
            "full_neighbor_list": self.full_neighbor_list,
            "self_pairs": self.self_pairs,
            "output": self._output_options.to_dict(),
            "execution": self._execution_options.to_dict(),
        }
        self._backend = HipBackend(self.name, backend_options, len(LABELS), level="pair")
        self._lock = threading.Lock()
        self._metadata_snapshot = self._envelope()

    @property
    def feature_count(self) -> int:
        return len(LABELS)

    def _envelope(self) -> dict[str, Any]:
        raw = {"backend": "mdescriptor-hip", "descriptor": self.name, "output": self._output_options.to_dict(),
               "execution": self._execution_options.to_dict()}
        return metadata_envelope(raw, "pair", self.feature_count)

    def _compute_batch(self, batch: Any, *, control: Any = None) -> DescriptorResult:
        try:
            raw = self._backend.compute(batch, control)
        except DescriptorInputError:
            raise
        except ValueError as exc:
            raise DescriptorInputError(str(exc), path=["input"]) from exc
        values = raw["values"]
        options = self._output_options
        if options.sparse:
            values = format_values(values, dtype=options.dtype, sparse=True)
        elif values.dtype != np.dtype(options.dtype):
            values = owned_values(np.ascontiguousarray(values, dtype=options.dtype))
        else:
            values = owned_values(values)
        metadata = self._envelope()
        result = DescriptorResult(values, "pair", batch.ids, raw["row_offsets"], LABELS, metadata,
                                  samples=owned_samples(raw["samples"]), feature_count=self.feature_count,
                                  _atom_row_offsets=np.asarray(batch.offsets, dtype=np.int64))
        self._metadata_snapshot = metadata
        return result

    def close(self) -> None:
        if not self.closed:
            self._backend.close()
        super().close()


__all__ = ["NeighborList"]
