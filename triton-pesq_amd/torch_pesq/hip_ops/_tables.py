"""Layout mark of the packed constant tables.

The modules carry their filter, STFT and model constants packed for the
kernels of the loaded library.  A module that is pickled whole takes these
bytes with it, and another build of the library may read them otherwise, at
the same size or another.  Each module therefore keeps the mark its tables
were packed under, and packs them again when it is loaded where the mark
differs.
"""

import functools
import hashlib

import numpy as np
import torch

from .. import _lib

__all__ = ["model_table_constants", "table_layout"]


@functools.lru_cache(maxsize=None)
def table_layout() -> str:
    """Digest of tables of every kind that the loaded library packs from fixed
    constants: what the tables hold, and where, decides it, so no number has to
    be raised by hand when either changes.  The same under any default device and
    dtype of the caller's.
    """

    with torch.device("cpu"):
        return _digest()


def _digest() -> str:

    from .chain import _pack_chain
    from .iir import _pack_cascade, _pack_table, sections_struct
    from .pipeline import pack_model_table
    from .spectral import _general_table

    bands = torch.arange(1, _lib.NBARKS + 1, dtype=torch.float64)
    window = torch.linspace(0.25, 0.75, _lib.NFFT, dtype=torch.float32)
    fbank = torch.zeros(_lib.NBARKS, _lib.NFFT // 2, dtype=torch.float32)
    fbank[torch.arange(_lib.NBARKS), torch.arange(_lib.NBARKS) + 1] = 1.0
    bins = np.arange(1, _lib.NBARKS + 1)
    sos = np.array([[0.5, 0.25, 0.125, 1.0, -0.5, 0.25], [0.75, -0.5, 0.25, 1.0, 0.25, 0.5]])
    tables = [
        _pack_table(sections_struct(0.5, [(s[0], s[1], s[2], s[4], s[5]) for s in sos])),
        _pack_cascade(sos),
        _pack_chain(bands, bands / 64, bands / 8, 6.0, 0.25),
        pack_model_table(None, None, None, None, window, fbank, bands, bands, bands / 64,
                         bands / 8, 6.0, 0.25),
        _general_table(window, bins, bins + 1, bands, _lib.NFFT, 160),
    ]
    digest = hashlib.sha256()
    for table in tables:
        digest.update(table.numpy().tobytes())
    return digest.hexdigest()


def model_table_constants(table: torch.Tensor) -> dict:
    """The float64 constants at the end of a model table of any build so far
    (``ModelTable`` in ``csrc/tables.hpp``; only what stands before them has
    changed): the correction of the 49 bands, and the thresholds, exponents and
    widths of up to 128.
    """

    end = 16 + 8 + 8  # n_fft, hop, counts; the calibration and the total width
    column = 8 * 128
    starts = {"width": end + column, "exp": end + 3 * column, "threshs": end + 4 * column}
    starts["corr"] = starts["threshs"] + 8 * _lib.NBARKS
    raw = table.detach().cpu().numpy()
    values = {}
    for name, start in starts.items():
        count = _lib.NBARKS if name == "corr" else 128
        at = raw.size - start
        values[name] = torch.from_numpy(raw[at : at + 8 * count].view(np.float64).copy())
    return values
