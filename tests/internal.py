"""Internal functions of libien_hip.so that the tests call by their C++ names
(no part of the C ABI: what they do is otherwise only reached through whole
networks)."""

import ctypes

import ien

_vp, _long, _int = ctypes.c_void_p, ctypes.c_long, ctypes.c_int


def _function(name, *argtypes, restype=_int):
    f = getattr(ien.load(), name)
    f.argtypes, f.restype = argtypes, restype
    return f


def _ptr(t):
    return None if t is None else t.data_ptr()


class LongSpectral:
    """lama.h spectral_new, _rows, _columns and _back: the fused spectral
    branch of maps with sides up to 128, a launch group at a time."""

    def __init__(self, ctx, height, width):
        h = _vp()
        new = _function("_ZN3ien12spectral_newEP7ien_ctxmmPP12ien_spectral", _vp, ctypes.c_size_t,
                        ctypes.c_size_t, ctypes.POINTER(_vp))
        ien.check(new(ctx.h, height, width, ctypes.byref(h)))
        self.h = h

    def rows(self, x, stride, m_in, spectral, r):
        f = _function("_ZN3ien13spectral_rowsEPK12ien_spectralPKtlPK10ien_matrixPtPf", _vp, _vp, _long, _vp, _vp, _vp)
        ien.check(f(self.h, _ptr(x), stride, m_in.h, _ptr(spectral), _ptr(r)))

    def columns(self, m_f, r, z, u):
        f = _function("_ZN3ien16spectral_columnsEPK12ien_spectralPK10ien_matrixPKfPtPf", _vp, _vp, _vp, _vp, _vp)
        ien.check(f(self.h, m_f.h, _ptr(r), _ptr(z), _ptr(u)))

    def back(self, m_out, spectral, u, out, stride, dst=None, add=None):
        f = _function("_ZN3ien13spectral_backEPK12ien_spectralPK10ien_matrixPKtPKfPtlSA_S7_", _vp, _vp, _vp, _vp, _vp,
                      _long, _vp, _vp)
        ien.check(f(self.h, m_out.h, _ptr(spectral), _ptr(u), _ptr(out), stride, _ptr(dst), _ptr(add)))

    def free(self):
        ien.load().ien_spectral_free(self.h)
        self.h = None


def conv_up_fits(h, w, c, n, ys):
    f = _function("_ZN3ien12conv_up_fitsElllll", *[_long] * 5, restype=ctypes.c_bool)
    return f(h, w, c, n, ys)


def conv_up(ctx, x, h, w, c, phases, y, ys, act):
    """ien_internal.h conv_up: a doubling's four phases in one launch."""
    f = _function("_ZN3ien7conv_upEP7ien_ctxPKtiiiPKP10ien_matrixPti7ien_act", _vp, _vp, _int, _int, _int,
                  ctypes.POINTER(_vp), _vp, _int, _int)
    handles = (_vp * 4)(*[m.h for m in phases])
    ien.check(f(ctx.h, _ptr(x), h, w, c, handles, _ptr(y), ys, act))


def conv3_choice(cus, workspace, ow, c, n, p_begin, p_end):
    """conv_common.h conv3_choice: (tile, split) of conv_wide, or None."""
    f = _function("_ZN3ien12conv3_choiceEiliiill", _int, _long, _int, _int, _int, _long, _long)
    r = f(cus, workspace, ow, c, n, p_begin, p_end)
    return None if r < 0 else (r // 16, r % 16)


def stride2_choice(cus, ow, n, p_begin, p_end):
    """conv_common.h stride2_choice: the general kernel's channels a chunk."""
    f = _function("_ZN3ien14stride2_choiceEiiill", _int, _int, _int, _long, _long)
    return f(cus, ow, n, p_begin, p_end)


def rows_choice(cus, workspace, m, k, n):
    """conv_common.h rows_choice: (waves a tile, splits)."""
    r = _function("_ZN3ien11rows_choiceEiliii", _int, _long, _int, _int, _int)(cus, workspace, m, k, n)
    return 8 if r < 0 else 4, abs(r)


def chain_choice(cus, h, w):
    """ien_internal.h chain_choice: the rows and columns of a chain's tiles, or None."""
    i = _function("_ZN3ien12chain_choiceEiii", _int, _int, _int)(cus, h, w)
    return None if i < 0 else [(8, 16), (12, 16), (16, 24)][i]
