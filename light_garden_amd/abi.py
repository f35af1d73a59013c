"""ctypes mirror of include/lg.h and the loader for the gfx950 library.

The library is light_garden_amd/build/liblg.so, built by light_garden_amd/build.py. There is
no fallback: if the library is missing or cannot open a gfx950 device, calls raise.
"""
import ctypes as C
import os

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "build", "liblg.so")

# ---- constants (lg.h) --------------------------------------------------------------------
LG_OK = 0
LG_E_INVALID = 1
LG_E_OOM = 2
LG_E_CAPACITY = 3
LG_E_HIP = 4
LG_E_UNSUPPORTED = 5
LG_E_NODEVICE = 6
LG_E_TIMEOUT = 7
LG_E_NOTFOUND = 8
STATUS_NAMES = {0: "LG_OK", 1: "LG_E_INVALID", 2: "LG_E_OOM", 3: "LG_E_CAPACITY", 4: "LG_E_HIP",
                5: "LG_E_UNSUPPORTED", 6: "LG_E_NODEVICE", 7: "LG_E_TIMEOUT", 8: "LG_E_NOTFOUND"}

SHAPE_LINE_SEGMENT = 0
SHAPE_CUBIC_BEZIER = 1
SHAPE_CIRCLE = 2
SHAPE_RECT = 3
SHAPE_LOGIC = 4
SHAPE_CONVEX_POLYGON = 5
SHAPE_ELLIPSE = 6

LOGIC_AND = 0
LOGIC_OR = 1
LOGIC_AND_NOT = 2

LIGHT_POINT = 0
LIGHT_DIRECTIONAL = 1
LIGHT_SPOT = 2

TRACE_FP64 = 1
SEG_VERTEX_COLORS = 1

MAX_SHAPES = 7
MAX_POLY_VERTICES = 16


class LgShape(C.Structure):
    _fields_ = [
        ("kind", C.c_int32), ("op", C.c_int32), ("child_a", C.c_int32), ("child_b", C.c_int32),
        ("n_vertices", C.c_int32), ("vertex_offset", C.c_int32),
        ("origin", C.c_double * 2), ("rotation", C.c_double * 4), ("p", C.c_double * 8),
    ]


class LgObject(C.Structure):
    _fields_ = [
        ("has_material", C.c_int32), ("n_shapes", C.c_int32), ("refractive_index", C.c_double),
        ("shapes", LgShape * MAX_SHAPES), ("vertices", C.c_double * (2 * MAX_POLY_VERTICES)),
    ]


class LgLight(C.Structure):
    _fields_ = [
        ("kind", C.c_int32), ("_pad0", C.c_int32), ("num_rays", C.c_uint64),
        ("color", C.c_float * 4), ("position", C.c_double * 2), ("direction", C.c_double * 2),
        ("spot_angle", C.c_double),
    ]


class LgParams(C.Structure):
    _fields_ = [
        ("max_bounce", C.c_uint32), ("flags", C.c_uint32), ("cutoff_color", C.c_float * 4),
        ("canvas", C.c_double * 4),
    ]


class LgView(C.Structure):
    _fields_ = [
        ("left", C.c_double), ("right", C.c_double), ("bottom", C.c_double), ("top", C.c_double),
        ("width", C.c_uint32), ("height", C.c_uint32),
    ]


class LgStageTime(C.Structure):
    _fields_ = [("name", C.c_char * 24), ("ms", C.c_float), ("launches", C.c_uint32),
                ("work", C.c_uint64), ("work2", C.c_uint64)]


class LgTuning(C.Structure):
    _fields_ = [("rays_per_item", C.c_uint32), ("min_piece", C.c_uint32), ("max_piece", C.c_uint32),
                ("trace_waves", C.c_uint32), ("bvh_min_objects", C.c_uint32), ("tile", C.c_uint32),
                ("trace_chunk", C.c_uint32), ("tile_block", C.c_uint32)]


class LgServerConfig(C.Structure):
    _fields_ = [("hbm_budget", C.c_uint64), ("max_batch", C.c_uint32), ("slots", C.c_uint32)]


class LgRequest(C.Structure):
    _fields_ = [("scene", C.c_void_p), ("image", C.c_void_p), ("params", LgParams), ("edit_index", C.c_int32),
                ("_pad0", C.c_int32), ("edit", LgObject), ("segments", C.c_void_p)]


class LgResult(C.Structure):
    _fields_ = [("status", C.c_int32), ("batch_size", C.c_uint32), ("segments", C.c_uint64),
                ("submit_us", C.c_double), ("start_us", C.c_double), ("end_us", C.c_double)]


class LgServerStats(C.Structure):
    _fields_ = [("submitted", C.c_uint64), ("completed", C.c_uint64), ("frames", C.c_uint64),
                ("evictions", C.c_uint64), ("resident_bytes", C.c_uint64), ("peak_resident_bytes", C.c_uint64),
                ("busy_us", C.c_double)]


SM_ADD, SM_MUL, SM_POW, SM_BASE = 0, 1, 2, 3
CURVE_CIRCLE, CURVE_COMPLEX_EXP, CURVE_HYPOTROCHOID, CURVE_LISSAJOUS = 0, 1, 2, 3
MAX_MOD_COLORS = 256
MAX_CROSSING_LINES = 1 << 18


class LgModRemColor(C.Structure):
    _fields_ = [("modulo", C.c_uint64), ("rem", C.c_uint64), ("color", C.c_float * 4)]


class LgStringMod(C.Structure):
    pass


LgStringMod._fields_ = [
    ("modulo", C.c_uint64), ("num", C.c_uint64), ("turns", C.c_uint64), ("mode", C.c_uint32),
    ("curve", C.c_uint32), ("curve_u", C.c_uint64 * 3), ("curve_f", C.c_double * 2), ("scale", C.c_double),
    ("color", C.c_float * 4), ("modulo_colors", C.POINTER(LgModRemColor)), ("n_modulo_colors", C.c_uint32),
    ("_pad0", C.c_uint32), ("nested", C.POINTER(LgStringMod)),
]


BF_ZERO, BF_ONE, BF_SRC, BF_ONE_MINUS_SRC, BF_SRC_ALPHA, BF_ONE_MINUS_SRC_ALPHA = 0, 1, 2, 3, 4, 5
BF_DST, BF_ONE_MINUS_DST, BF_DST_ALPHA, BF_ONE_MINUS_DST_ALPHA, BF_SRC_ALPHA_SATURATED = 6, 7, 8, 9, 10
BF_CONSTANT, BF_ONE_MINUS_CONSTANT = 11, 12
BO_MIN, BO_MAX, BO_ADD, BO_SUBTRACT, BO_REVERSE_SUBTRACT = 0, 1, 2, 3, 4
ENCODE_BGRA, ENCODE_RGBA = 0, 1


class LgBlendComponent(C.Structure):
    _fields_ = [("src_factor", C.c_uint32), ("dst_factor", C.c_uint32), ("operation", C.c_uint32)]


class LgBlend(C.Structure):
    _fields_ = [("color", LgBlendComponent), ("alpha", LgBlendComponent), ("constant", C.c_float * 4)]


assert C.sizeof(LgShape) == 136
assert C.sizeof(LgObject) == 16 + 7 * 136 + 256
assert C.sizeof(LgLight) == 72
assert C.sizeof(LgParams) == 56
assert C.sizeof(LgView) == 40

# Every function lg.h declares: name -> (restype, argtypes)
_P = C.c_void_p
_PP = C.POINTER(C.c_void_p)
FUNCTIONS = {
    "lg_last_error": (C.c_char_p, []),
    "lg_version": (C.c_int, []),
    "lg_ctx_create": (C.c_int, [C.c_int, _PP]),
    "lg_ctx_destroy": (C.c_int, [_P]),
    "lg_ctx_synchronize": (C.c_int, [_P]),
    "lg_ctx_set_profiling": (C.c_int, [_P, C.c_int]),
    "lg_ctx_stage_times": (C.c_int, [_P, C.POINTER(LgStageTime), C.c_int, C.POINTER(C.c_int)]),
    "lg_calibrate_lds_atomics": (C.c_int, [_P, C.POINTER(C.c_double)]),
    "lg_scene_create": (C.c_int, [_P, _PP]),
    "lg_scene_destroy": (C.c_int, [_P]),
    "lg_scene_clear": (C.c_int, [_P]),
    "lg_scene_clear_objects": (C.c_int, [_P]),
    "lg_scene_push_object": (C.c_int, [_P, C.POINTER(LgObject)]),
    "lg_scene_push_light": (C.c_int, [_P, C.POINTER(LgLight)]),
    "lg_scene_set_objects": (C.c_int, [_P, C.POINTER(LgObject), C.c_uint32]),
    "lg_scene_set_lights": (C.c_int, [_P, C.POINTER(LgLight), C.c_uint32]),
    "lg_scene_replace_object": (C.c_int, [_P, C.c_uint32, C.POINTER(LgObject)]),
    "lg_scene_remove_object": (C.c_int, [_P, C.c_uint32]),
    "lg_scene_remove_light": (C.c_int, [_P, C.c_uint32]),
    "lg_scene_counts": (C.c_int, [_P, C.POINTER(C.c_uint32), C.POINTER(C.c_uint32),
                                  C.POINTER(C.c_uint64)]),
    "lg_segments_create": (C.c_int, [_P, C.c_uint64, C.c_uint32, _PP]),
    "lg_segments_destroy": (C.c_int, [_P]),
    "lg_segments_count": (C.c_int, [_P, C.POINTER(C.c_uint64)]),
    "lg_segments_upload": (C.c_int, [_P, _P, _P, _P, C.c_uint64]),
    "lg_segments_download": (C.c_int, [_P, _P, _P, _P, _P, C.c_uint64, C.POINTER(C.c_uint64)]),
    "lg_segments_download_pos64": (C.c_int, [_P, _P, C.c_uint64, C.POINTER(C.c_uint64)]),
    "lg_segments_download_vertices": (C.c_int, [_P, _P, _P, C.c_uint64, C.POINTER(C.c_uint64)]),
    "lg_trace": (C.c_int, [_P, C.POINTER(LgParams), _P]),
    "lg_trace_all": (C.c_int, [_P, C.POINTER(LgParams), _P, _P, C.c_uint64,
                               C.POINTER(C.c_uint64)]),
    "lg_image_create": (C.c_int, [_P, C.POINTER(LgView), _PP]),
    "lg_image_destroy": (C.c_int, [_P]),
    "lg_image_clear": (C.c_int, [_P]),
    "lg_image_device_ptrs": (C.c_int, [_P, _PP, _PP]),
    "lg_image_download_rgba16f": (C.c_int, [_P, _P, C.c_uint64]),
    "lg_image_download_accum": (C.c_int, [_P, _P, C.c_uint64]),
    "lg_accumulate": (C.c_int, [_P, _P, _P]),
    "lg_accumulate_noalloc": (C.c_int, [_P, _P, _P]),
    "lg_resolve": (C.c_int, [_P, _P]),
    "lg_render": (C.c_int, [_P, C.POINTER(LgParams), _P, _P]),
    "lg_batch_render": (C.c_int, [_P, C.c_uint32, C.POINTER(C.c_void_p), C.POINTER(LgParams),
                                  C.POINTER(C.c_void_p), C.POINTER(C.c_void_p)]),
    "lg_ctx_set_graphs": (C.c_int, [_P, C.c_int]),
    "lg_ctx_set_packed_accumulation": (C.c_int, [_P, C.c_int]),
    "lg_ctx_get_tuning": (C.c_int, [_P, C.POINTER(LgTuning)]),
    "lg_ctx_set_tuning": (C.c_int, [_P, C.POINTER(LgTuning)]),
    "lg_server_create": (C.c_int, [_P, C.POINTER(LgServerConfig), _PP]),
    "lg_server_destroy": (C.c_int, [_P]),
    "lg_server_submit": (C.c_int, [_P, C.POINTER(LgRequest), C.POINTER(C.c_uint64)]),
    "lg_server_wait": (C.c_int, [_P, C.c_uint64, C.c_double, C.POINTER(LgResult)]),
    "lg_server_get_stats": (C.c_int, [_P, C.POINTER(LgServerStats)]),
    "lg_string_mod_draw": (C.c_int, [_P, C.c_uint32, C.POINTER(LgStringMod), _P]),
    "lg_string_mod_crossings": (C.c_int, [_P, C.POINTER(LgStringMod), _P, C.c_uint64,
                                          C.POINTER(C.c_uint64)]),
    "lg_image_set_blend": (C.c_int, [_P, C.POINTER(LgBlend)]),
    "lg_image_get_blend": (C.c_int, [_P, C.POINTER(LgBlend)]),
    "lg_image_encode_8bit": (C.c_int, [_P, C.c_uint32, _P, C.c_uint64]),
    "lg_encode_table": (C.c_int, [_P, _P]),
    "lg_scene_load_ron": (C.c_int, [_P, C.c_char_p, C.c_uint64]),
    "lg_scene_save_ron": (C.c_int, [_P, C.c_char_p, C.c_uint64, C.POINTER(C.c_uint64)]),
    "lg_ron_parse_scene": (C.c_int, [C.c_char_p, C.c_uint64, C.POINTER(LgObject), C.c_uint32,
                                     C.POINTER(C.c_uint32), C.POINTER(LgLight), C.c_uint32,
                                     C.POINTER(C.c_uint32)]),
    "lg_ron_write_scene": (C.c_int, [C.POINTER(LgObject), C.c_uint32, C.POINTER(LgLight),
                                     C.c_uint32, C.c_char_p, C.c_uint64, C.POINTER(C.c_uint64)]),
}

_lib = None


class LgError(RuntimeError):
    def __init__(self, code, where, msg):
        super().__init__("%s failed with %s: %s" % (where, STATUS_NAMES.get(code, code), msg))
        self.code = code


def load():
    """Opens liblg.so (built in-tree). Raises when it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError("light_garden_amd: %s is missing; run light_garden_amd/build.py "
                           "(or __graft_entry__.build())" % LIB_PATH)
    lib = C.CDLL(LIB_PATH)
    for name, (res, args) in FUNCTIONS.items():
        f = getattr(lib, name)
        f.restype = res
        f.argtypes = args
    _lib = lib
    return lib


def check(code, where):
    if code != LG_OK:
        msg = load().lg_last_error()
        raise LgError(code, where, msg.decode() if msg else "")
    return code


def call(name, *args):
    return check(getattr(load(), name)(*args), name)
