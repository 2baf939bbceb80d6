"""Callable wrapper around a native operator (reference: kernel_matmul/native_function.py:11-86).

``NativeFunction(name, config)(*args)`` asks the configuration for a cache key; when the key
changes (different batch rank, rhs width, ...) it asks for candidate define sets, times them if
there is more than one, and binds the winner through ``load_native``.  With the gfx950 table
the configurations return one candidate, so the timing branch only runs for caller-supplied
configurations with several.
"""
from __future__ import annotations

import multiprocessing.pool
from typing import Any

from kernel_matmul_amd import configurations
from kernel_matmul_amd.compile import Defines, find_best, load_native, module_environment
from kernel_matmul_amd.configurations import Configuration
from kernel_matmul_amd.util import format_dict

_SHARED_CONFIGURATIONS = frozenset({
    configurations.MatmulAutotuneConfiguration, configurations.MatmulBwdConfiguration,
    configurations.BilinearDerivativeConfiguration, configurations.IndexConfiguration,
    configurations.IndexBwdConfiguration, configurations.DenseConfiguration, configurations.DenseBwdConfiguration,
})
_SHARED_MODULES: dict = {}
_SHARED_LIMIT = 256

class NativeFunction:
    def __init__(
        self,
        name: str,
        config: Configuration,
        num_measurements: int = 1,
        verbose: bool = False,
        compile_pool: multiprocessing.pool.Pool | None = None,
    ):
        self.name = name
        self.config = config
        self.num_measurements = num_measurements
        self.verbose = verbose
        self.compile_pool = compile_pool
        self._defines: Defines | None = None
        self._cache_key: str | None = None
        self._module = None

    def _select(self, args: tuple) -> Defines:
        candidates = self.config.make_candidates(args)
        if len(candidates) == 1:
            return candidates[0]
        if self.verbose:
            print(f"Autotuning {self.name}...")
        best, timings = find_best(
            self.name,
            args,
            candidates,
            return_timings=True,
            num_measurements=self.num_measurements,
            compile_pool=self.compile_pool,
        )
        if self.verbose:
            for position, (timing, candidate) in enumerate(zip(timings, candidates)):
                print(f"  - Candidate {position}: {timing:.3f} ms ({format_dict(candidate)})")
            print(f"Best: {format_dict(best)}")
        return best

    def __call__(self, *args: Any) -> Any:
        key = self.config.cache_key(args)
        if self._module is None or key != self._cache_key:
            self._defines, self._module = self._bind(key, args)
            self._cache_key = key
        return self._module.call(*args)

    def _bind(self, key: str, args: tuple):
        """Define set and module for arguments of this cache key.  Operators are made anew for every set of
        hyper-parameters, so what the configurations of this package (whose one candidate follows from kernel
        type and cache key) lead to is shared by all functions."""
        if type(self.config) not in _SHARED_CONFIGURATIONS:
            defines = self._select(args)
            return defines, load_native(self.name, defines=defines)
        shared_key = (self.name, type(self.config), self.config.kernel_type, key, module_environment())
        shared = _SHARED_MODULES.get(shared_key)
        if shared is None:
            defines = self._select(args)
            shared = (defines, load_native(self.name, defines=defines))
            if len(_SHARED_MODULES) >= _SHARED_LIMIT:
                _SHARED_MODULES.clear()
            _SHARED_MODULES[shared_key] = shared
        defines, module = shared
        return dict(defines), module

    @property
    def defines(self) -> Defines | None:
        """Define set bound by the last (re)selection; ``None`` before the first call."""
        return self._defines
