// Stands in for libftkernels.so: its calls launch nothing and return how many of them were made with Python's lock held.
#include <Python.h>

#include "../include/ftk.h"

static int held = 0;
static int call() { return held += PyGILState_Check(); }

extern "C" {
int ftk_b2b_gemm_f16(const void*, const void*, const void*, void*, int, int, int, int, int, ftk_stream_t) { return call(); }
int ftk_flash_attn_f16(const void*, const void*, const void*, void*, int, int, int, int, int, float, ftk_stream_t) { return call(); }
int ftk_flash_attn_ws_f16(const void*, const void*, const void*, void*, int, int, int, int, int, float, void*, size_t, ftk_stream_t) { return call(); }
int ftk_flash_attn_f32(const float*, const float*, const float*, float*, int, int, int, int, int, float, void*, size_t, ftk_stream_t) { return call(); }
size_t ftk_flash_attn_f16_workspace_bytes(int, int, int, int, int) { return 256; }
size_t ftk_flash_attn_f32_workspace_bytes(int, int, int, int, int) { return 256; }
size_t ftk_stacked_lstm_workspace_bytes(int, int, int, int) { return 256; }
size_t ftk_stacked_lstm_f16_workspace_bytes(int, int, int, int) { return 256; }
int ftk_stacked_lstm_f16(const void*, const void*, const float*, const int*, const int*, void*, void*, int, int, int, int, void*, size_t, ftk_stream_t) { return call(); }
int ftk_stacked_lstm_opts_f32(const float*, const float*, const float*, const int*, const int*, float*, float*, int, int, int, int,
                              const ftk_lstm_options*, void*, size_t, ftk_stream_t) { return call(); }
int ftk_stacked_lstm_result(const void*, int* small, ftk_stream_t) {
  *small = 0;
  return call();
}
}
